"""Seeded random shapes through the tiled gemm_tn (M > 64, and M <= 64 where
the plan is one of the same kernel's 64-row tiles): every tile shape and
split plan the launcher picks, ragged M / N / K, odd and 4-aligned N, with
and without a bias, fp16 and bf16, against an fp32 GEMM at the parity bar.
The torch op (workspace from the caching allocator, so split plans run) and
the workspace-free C entry point must also agree bit for bit whenever both run
the same unsplit plan."""

import ctypes
import random

import pytest
import torch

import decodekernels_amd as dk
from decodekernels_amd import capi
from parity import assert_max_abs, gemm_f32_gpu
from test_gemm_plan import replica_plan, runs_tile

pytestmark = pytest.mark.gpu


def _shapes(count=48, seed=2024):
    rng = random.Random(seed)
    out = []
    while len(out) < count:
        M = rng.choice([rng.randint(65, 700), rng.randint(700, 3000)])
        N = rng.choice([rng.randint(1, 6000), 4 * rng.randint(1, 2200), 64 * rng.randint(1, 140)])
        K = 8 * rng.randint(1, 400)
        out.append((M, N, K, rng.random() < 0.5, rng.random() < 0.5))
    # Decode sizes whose plan is one of the tiled kernel's 64-row tiles.
    while len(out) < count + 24:
        M = rng.randint(32, 64)
        N = rng.choice([rng.randint(1000, 20000), 4 * rng.randint(250, 5000), rng.randint(32769, 40000)])
        K = 8 * rng.randint(64, 1200)
        if runs_tile(replica_plan(M, N, K)):  # host arithmetic, checked against the library on the CPU
            out.append((M, N, K, rng.random() < 0.5, rng.random() < 0.5))
    return out


@pytest.mark.parametrize("M,N,K,with_bias,bf16", _shapes())
def test_tiled_gemm_random_shapes(M, N, K, with_bias, bf16):
    dtype = torch.bfloat16 if bf16 else torch.float16
    g = torch.Generator(device="cuda").manual_seed(M * 7919 + N * 31 + K)
    a = torch.randn(M, K, generator=g, device="cuda", dtype=dtype)
    b = torch.randn(N, K, generator=g, device="cuda", dtype=dtype) / K**0.5
    bias = torch.randn(N, generator=g, device="cuda", dtype=dtype) if with_bias else None
    plan = capi.gemm_plan(M, N, K)
    print(f"gemm {M}x{N}x{K} bias={with_bias} {dtype} plan {plan}", flush=True)
    out = dk.gemm(a, b, bias)
    assert_max_abs(out, gemm_f32_gpu(a, b, bias), dtype, f"gemm {M}x{N}x{K} plan {plan}")
    if plan[2] == 1:  # unsplit: the C entry point without a workspace runs the same kernel
        c = torch.empty(M, N, device="cuda", dtype=dtype)
        rc = capi.lib().dk_gemm_tn(capi.dtype_code(dtype), a.data_ptr(), b.data_ptr(),
                                   None if bias is None else bias.data_ptr(), c.data_ptr(), M, N, K, K, K, N,
                                   ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
        assert rc == 0, capi.last_error()
        torch.cuda.synchronize()
        assert torch.equal(c, out)


# (tile rows, tile columns, K splits) -> (M, N, K), larger than those of
# tests/test_gemm_tile.py: full tiles, ragged M, ragged N, both, K in one slice or
# two and K split, with the B loads of 128 x 160 uneven over the waves.
TILE_SHAPES = [
    ((128, 128, 1), (271, 6563, 5824)), ((128, 160, 1), (1003, 4608, 3584)), ((192, 192, 1), (612, 11259, 64)),
    ((192, 192, 1), (1536, 6144, 4096)), ((192, 192, 1), (1844, 4416, 72)), ((192, 192, 1), (3072, 6144, 4096)),
    ((192, 192, 4), (384, 6144, 4808)), ((192, 192, 4), (1152, 1800, 3528)), ((192, 192, 6), (132, 6168, 5440)),
    ((192, 192, 8), (131, 5464, 4512)), ((192, 256, 1), (263, 24976, 64)), ((192, 256, 1), (768, 28672, 4096)),
    ((192, 256, 1), (1049, 8736, 144)), ((192, 256, 1), (1728, 5472, 136)), ((256, 128, 1), (961, 6113, 5704)),
    ((256, 256, 1), (512, 28672, 4096)), ((256, 256, 1), (768, 18728, 120)), ((256, 256, 1), (795, 13247, 64)),
    ((256, 256, 1), (1053, 11424, 88)),
]


@pytest.mark.parametrize("tile,shape", TILE_SHAPES, ids=[f"{t[0]}x{t[1]}/{t[2]}-{m}x{n}x{k}" for t, (m, n, k) in TILE_SHAPES])
@pytest.mark.parametrize("bf16", [True, False])
def test_tile_shapes_against_fp32(tile, shape, bf16):
    M, N, K = shape
    dtype = torch.bfloat16 if bf16 else torch.float16
    plan = capi.gemm_plan(M, N, K)
    print(f"gemm {M}x{N}x{K} {dtype} plan {plan}", flush=True)
    assert plan[:3] == tile, plan  # the plan names what runs
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    a = torch.randn(M, K, generator=g, device="cuda", dtype=dtype)
    b = torch.randn(N, K, generator=g, device="cuda", dtype=dtype) / K**0.5
    bias = torch.randn(N, generator=g, device="cuda", dtype=dtype)
    out = dk.gemm(a, b, bias)
    assert_max_abs(out, gemm_f32_gpu(a, b, bias), dtype, f"gemm {M}x{N}x{K} plan {plan}")
    c = torch.full((M, N), float("nan"), device="cuda", dtype=dtype)
    rc = capi.lib().dk_gemm_tn(capi.dtype_code(dtype), a.data_ptr(), b.data_ptr(), None, c.data_ptr(), M, N, K, K, K, N,
                               ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0, capi.last_error()
    torch.cuda.synchronize()
    assert_max_abs(c, gemm_f32_gpu(a, b), dtype, f"gemm {M}x{N}x{K} unsplit, no bias")
