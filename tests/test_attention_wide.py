"""Short decode calls around the lines between attention workgroups of NW and
of 2 NW waves (NW = 2 at head_dim > 128, else 4), against the fp32 reference
at the parity bar: one tile a wave and one token more, unit edges, ragged and
empty sequences, workgroup counts on both sides of each class's limit on 256
CUs (a round at head_dim > 128, half the CUs at <= 64, an eighth between)."""

import pytest
import torch

import decodekernels_amd as dk
from decodekernels_amd.testing import make_paged_kv
from parity import assert_max_abs, attention_f32

pytestmark = pytest.mark.gpu

FP8 = torch.float8_e4m3fn

# head_dim, KV heads, group, block size, lengths
CASES = [
    (256, 2, 8, 16, [32]),
    (256, 2, 8, 16, [33, 1]),
    (256, 1, 16, 8, [512, 0, 17, 511]),
    (192, 4, 1, 16, [513, 15, 1024]),
    (256, 2, 3, 16, [512] * 128),  # 256 workgroups
    (256, 2, 3, 16, [100] * 129),  # 258
    (64, 2, 7, 16, [64]),
    (64, 2, 7, 48, [65, 3]),
    (64, 8, 4, 16, [130, 0, 512] + [40] * 13),  # 128
    (64, 1, 4, 16, [65] * 129),  # 129
    (64, 2, 2, 8, [8192, 1, 700]),
    (128, 8, 4, 16, [64]),
    (128, 8, 4, 16, [65, 1, 0, 512]),  # 32
    (128, 8, 4, 16, [129] * 5),  # 40
    (128, 4, 7, 24, [1000, 513]),
    (96, 4, 8, 16, [512, 16, 17]),
]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("case", range(len(CASES)))
def test_short_calls(case, fp8, dtype):
    d, hkv, group, bs, lens = CASES[case]
    if fp8 and d % 64:
        pytest.skip("fp8 rows are read in 64-column pieces")
    print(f"case {case}: {CASES[case][:4]}, {len(lens)} sequences, fp8 {fp8}, {dtype}", flush=True)
    kv = make_paged_kv(lens, hkv, d, bs, FP8 if fp8 else dtype, "cuda", layout=["nhd", "vllm"][case % 2], seed=case)
    g = torch.Generator(device="cuda").manual_seed(case)
    q = torch.randn(len(lens), hkv * group, d, generator=g, device="cuda", dtype=dtype) * d**-0.5
    scales = dict(k_scale=0.5, v_scale=0.75) if fp8 else {}
    out = dk.paged_attention_decode(q, kv.k_cache, kv.v_cache, kv.block_tables, kv.seq_lens, max_seq_len=max(lens),
                                    **scales)
    k = kv.k_cache.float() * 0.5 if fp8 else kv.k_cache
    v = kv.v_cache.float() * 0.75 if fp8 else kv.v_cache
    assert_max_abs(out, attention_f32(q, k, v, kv.block_tables, kv.seq_lens), dtype, f"case {case}, fp8 {fp8}")
    assert (out[torch.tensor(lens, device="cuda") == 0] == 0).all()
