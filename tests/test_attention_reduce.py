"""The split-K reduce on both sides of its line between 16 and 4 waves a head
(512 heads, where the workspace has 64 rows or more), against the fp32
reference at the parity bar: one long sequence -- many pieces of the balanced
schedule -- among short and empty ones, and the partition grid's 64 rows a head."""

import pytest
import torch

import decodekernels_amd as dk
from decodekernels_amd.testing import make_paged_kv
from parity import assert_max_abs, attention_f32

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("head_dim", [64, 128, 256])
@pytest.mark.parametrize("seqs, bound", [(31, 32768), (32, 32256), (32, 32768), (40, 131072)])
def test_one_long_sequence(seqs, bound, head_dim, dtype, monkeypatch):
    monkeypatch.setenv("DK_ATTN_SCHEDULE", "balanced")
    lens = [20000, 0, 513] + [1 + 37 * i for i in range(seqs - 3)]
    print(f"{seqs} sequences, length bound {bound}, head_dim {head_dim}, {dtype}", flush=True)
    kv = make_paged_kv(lens, 1, head_dim, 16, dtype, "cuda", seed=seqs)
    g = torch.Generator(device="cuda").manual_seed(seqs)
    q = torch.randn(seqs, 16, head_dim, generator=g, device="cuda", dtype=dtype) * head_dim**-0.5
    out = dk.paged_attention_decode(q, kv.k_cache, kv.v_cache, kv.block_tables, kv.seq_lens, max_seq_len=bound)
    assert_max_abs(out, attention_f32(q, kv.k_cache, kv.v_cache, kv.block_tables, kv.seq_lens), dtype,
                   f"{seqs} sequences, bound {bound}, head_dim {head_dim}")
    assert (out[1] == 0).all()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("seqs", [31, 32])
def test_partition_rows(seqs, dtype, monkeypatch):
    """496 and 512 heads of 64, up to 64 rows of 512 tokens each."""
    monkeypatch.setenv("DK_ATTN_SCHEDULE", "partitions")
    lens = [32768, 0, 1] + [32768 - 997 * i for i in range(seqs - 3)]
    print(f"{seqs} sequences, {dtype}", flush=True)
    kv = make_paged_kv(lens, 1, 64, 16, dtype, "cuda", seed=seqs)
    g = torch.Generator(device="cuda").manual_seed(seqs)
    q = torch.randn(seqs, 16, 64, generator=g, device="cuda", dtype=dtype) * 64**-0.5
    out = dk.paged_attention_decode(q, kv.k_cache, kv.v_cache, kv.block_tables, kv.seq_lens, max_seq_len=32768)
    assert_max_abs(out, attention_f32(q, kv.k_cache, kv.v_cache, kv.block_tables, kv.seq_lens), dtype,
                   f"{seqs} sequences, partition rows")
    assert (out[1] == 0).all()
