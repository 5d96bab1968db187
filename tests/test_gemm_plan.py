"""CPU tests of what gemm_tn runs, through ``dk_gemm_tn_plan`` /
``dk_gemm_tn_workspace_bytes`` (host arithmetic, no kernel launch).

M > 64 (``tile_plan`` in decodekernels_amd/csrc/gemm.hip): of eleven tile shapes
with 1, 2, 3, 4, 6 or 8 K splits (>= 512 columns each, <= 256 tiles, <= 768
workgroups, <= 64 MiB of partials), the one with the smallest modelled time,
ceil(workgroups / 256) x (slices x slice + tile) plus the cost of a split; a
slice costs more where K % 64 != 0.

M <= 64 (``decode_plan``): the skinny kernel or a 64-row tile of 64 or 128
columns, whichever is modelled faster (a tile where no skinny grid fits one
workgroup per CU, N > 32768). The skinny kernel's own plan
(``skinny_plan``: workgroup shape = waves along N, 16 columns each, x waves
along K, and K splits) is the widest unsplit grid of <= 256 workgroups when it
fills >= 3/4 of the 256 CUs and each workgroup re-reads <= 256 KiB of
activations; else, with a workspace, the grid of 2..8 K splits (>= 512 columns
each, <= 256 workgroups, within 10% of the fullest) with the fewest splits
whose workgroups re-read <= max(128 KiB, half their weight bytes) of
activations (else the fewest activation bytes); else the unsplit grid, or the
wide plan for N > 32768.

A plan that does not split is the same with and without a workspace.

This file restates that arithmetic and checks, over random shapes, that the
library plans exactly the same, plus the invariants the kernels rely on: every
split non-empty and a multiple of 64 columns, the workspace size, and a
workgroup shape the launcher instantiates. The Llama-3-8B, Qwen2.5 and Phi-3
projections map to plans measured fastest or within a few percent of it.
"""

import random

import pytest

from decodekernels_amd import capi

SHAPES = [(1, 8), (2, 4), (4, 2), (6, 2), (7, 2), (8, 1)]
KIB = 1024
MAX_WORKSPACE = 64 << 20

# (rows, columns, us per 64-column slice, the same where K % 64 != 0, us per tile)
TILES = [(256, 256, 1.18, 1.52, 9.44), (256, 192, 0.962, 1.26, 10.7), (192, 256, 0.971, 1.26, 9.13),
         (256, 128, 0.716, 1.21, 6.41), (128, 256, 0.883, 1.24, 7.19), (128, 128, 0.509, 0.847, 4.19),
         (128, 160, 0.638, 0.909, 6.5), (128, 64, 0.395, 0.706, 2.53), (64, 64, 0.283, 0.442, 1.33),
         (64, 128, 0.365, 0.678, 5.48), (192, 192, 0.894, 1.23, 6.33)]
DECODE_TILES = [(64, 64, 0.377, 0.377, 2.05), (64, 128, 0.680, 0.680, 2.55)]
# split, partials, odd
TILE_MODEL = (2.7, 6.28e6, 3.53)
DECODE_MODEL = (2.37, 9.55e6, 8.76)
SKINNY_STEP = dict(zip((1, 2, 4, 6, 7, 8), (0.631, 0.527, 0.622, 0.764, 1.35, 0.589)))
SKINNY_ROWS = (1.0, 1.59, 1.62)
SKINNY_BASE = (1.71, 1.80, 2.53)


def _wide(M, N, K):
    mt = 1 if M <= 16 else (2 if M <= 32 else 4)
    min_wgs = 384 if mt == 1 else 192
    wn = 8 if (M > 32 and N >= 24576) else (4 if N >= 64 * min_wgs else (2 if N >= 32 * min_wgs else 1))
    return (wn, 8 // wn, 1, K)


def _unsplit(N, K):
    for wn, wk in SHAPES:
        if -(-N // (16 * wn)) <= 256:
            return (wn, wk, 1, K)
    return None


def replica_skinny_plan(M, N, K, with_workspace=True, mistake=None):
    """(wn, wk, splits, k_split) as skinny_plan computes it. ``mistake`` plants
    an error: "fill" drops the 3/4-fill condition of the unsplit grid, "limit"
    compares activation bytes with the weight bytes instead of half of them."""
    u = _unsplit(N, K)
    if u is not None and M * K * 2 <= 256 * KIB and (mistake == "fill" or 4 * -(-N // (16 * u[0])) >= 3 * 256):
        return u
    cands = []
    if with_workspace and K > 0:
        for wn, wk in SHAPES:
            tiles = -(-N // (16 * wn))
            for s in range(2, 9):
                if K // s < 512:
                    break
                per = -(-K // s)
                ks = -(-per // 64) * 64
                if -(-K // ks) != s:
                    continue
                if tiles * s > 256:
                    break
                cands.append((wn, wk, s, ks, tiles * s))
    if cands:
        mx = max(c[4] for c in cands)
        near = [c for c in cands if 10 * c[4] >= 9 * mx]
        div = 1 if mistake == "limit" else 2
        ok = [c for c in near if M * c[3] * 2 <= max(128 * KIB, 16 * c[0] * c[3] * 2 // div)]
        best = min(ok, key=lambda c: (c[2], near.index(c))) if ok else min(near, key=lambda c: (M * c[3], c[2], near.index(c)))
        return best[:4]
    return u if u is not None else _wide(M, N, K)


def _split_us(model, s, M, N, mistake=None):
    split, partials, odd = model
    return split + s * (float(M) * N) * 8.0 / partials * (odd if N % 4 != 0 and mistake != "odd" else 1.0) if s > 1 else 0.0


def _tile_candidates(model, tiles, M, N, K, with_workspace, mistake=None):
    """(us, (rows, columns, splits, k_split)) of every tiled candidate, in the library's order."""
    for bm, bn, slice_us, ragged_us, tile_us in tiles:
        slice_us = slice_us if K % 64 == 0 or mistake == "ragged" else ragged_us
        n = -(-M // bm) * -(-N // bn)
        for s in (1, 2, 3, 4, 6, 8):
            ks = K
            if s > 1:
                if not with_workspace or n > 256 or n * s > 768 or K // s < 512 or s * M * N * 4 > MAX_WORKSPACE:
                    break
                ks = -(-(-(-K // s)) // 64) * 64
                if -(-K // ks) != s:
                    continue
            rounds = n * s / 256 if mistake == "rounds" else float(-(-(n * s) // 256))
            yield rounds * (float(-(-ks // 64)) * slice_us + tile_us) + _split_us(model, s, M, N, mistake), (bm, bn, s, ks)


def _plan(M, N, K, with_workspace, mistake):
    if M > 64:
        return min(_tile_candidates(TILE_MODEL, TILES, M, N, K, with_workspace, mistake), key=lambda c: c[0])[1]
    p = replica_skinny_plan(M, N, K, with_workspace, mistake)
    if K == 0:
        return p
    cands = list(_tile_candidates(DECODE_MODEL, DECODE_TILES, M, N, K, with_workspace, mistake))
    if _unsplit(N, K) is None:
        return min(cands, key=lambda c: c[0])[1]
    wn, wk, s, ks = p
    rows = 0 if M <= 16 else (1 if M <= 32 else 2)
    rounds = float(-(-N // (16 * wn)) * s) / 256
    t = 1.26 + max(1.0, rounds) * (float(-(-ks // 64)) / wk * (SKINNY_STEP[wn] * SKINNY_ROWS[rows]) + SKINNY_BASE[rows])
    t += _split_us(DECODE_MODEL, s, M, N, mistake)
    return min([(t, p), *cands], key=lambda c: c[0])[1]


def replica_plan(M, N, K, with_workspace=True, mistake=None):
    """gemm_tn's plan: (tile rows, tile columns, splits, k_split) or, for the
    skinny kernel, (wn, wk, splits, k_split). ``mistake`` plants an error:
    "rounds" counts part-filled rounds by their fill, "odd" drops the price of
    partials of odd widths, "ragged" that of a ragged K, "fill" / "limit" go to
    the skinny plan."""
    full = _plan(M, N, K, True, mistake)
    return full if with_workspace or full[2] == 1 else _plan(M, N, K, False, mistake)


def runs_tile(plan):
    """Whether a plan runs the tiled kernel (rows and columns of a tile, not waves)."""
    return plan[0] >= 64


def random_shapes(n, seed):
    """Sizes on both sides of M = 64, small and large, half of them up to N = 130000."""
    rng = random.Random(seed)
    for _ in range(n):
        M = rng.choice([rng.randint(1, 64), rng.randint(1, 64), rng.randint(65, 600), rng.randint(65, 5000)])
        N = rng.choice([rng.randint(1, 600), rng.randint(1, 8192), rng.randint(1, 40000), rng.randint(12000, 130000)])
        K = 8 * rng.choice([rng.randint(0, 64), rng.randint(0, 3000)])
        yield M, N, K


def test_library_plans_like_the_replica():
    for M, N, K in random_shapes(40000, 3):
        for ws in (True, False):
            assert capi.gemm_plan(M, N, K, ws) == replica_plan(M, N, K, ws), (M, N, K, ws)


def test_plan_invariants_and_workspace_size():
    L = capi.lib()
    tiles = {(bm, bn) for bm, bn, *_ in TILES}
    for M, N, K in random_shapes(40000, 4):
        a, b, s, ks = plan = capi.gemm_plan(M, N, K)
        if M > 64:
            assert (a, b) in tiles, (M, N, K)
        else:
            assert (a, b) in SHAPES or (a, b) in ((64, 64), (64, 128)), (M, N, K)
        nbytes = L.dk_gemm_tn_workspace_bytes(M, N, K)
        if s == 1:
            # the call that runs asks for no workspace, and none changes what runs
            assert ks == K and nbytes == 0 and capi.gemm_plan(M, N, K, False) == plan
            continue
        assert 2 <= s <= 8 and ks % 64 == 0 and ks >= 512, (M, N, K, s, ks)
        assert (s - 1) * ks < K <= s * ks, "a split is empty or K is not covered"
        assert nbytes == s * M * N * 4
        if runs_tile(plan):
            assert nbytes <= MAX_WORKSPACE and -(-M // a) * -(-N // b) * s <= 768
        else:
            assert -(-N // (16 * a)) * s <= 256, "a skinny split plan over-fills the CUs"
        # without a workspace the same size is planned unsplit
        assert capi.gemm_plan(M, N, K, False)[2] == 1


# (M, N, K) -> (tile rows, tile columns, splits), or (waves along N, waves along K,
# splits) of the skinny kernel, at the projections of Llama-3-8B, Qwen2.5-7B and
# Qwen2.5-0.5B and the language-model head: the fastest of all candidates from
# cold caches, or within 4% of it (7% and 12%: the small model's qkv at M = 64 and
# gate_up at M = 1).
PICKS = {
    # qkv, o, gate_up, down of Llama-3-8B
    (1, 6144, 4096): (2, 4, 1), (32, 6144, 4096): (64, 128, 4), (64, 6144, 4096): (64, 128, 4),
    (256, 6144, 4096): (128, 128, 2), (384, 6144, 4096): (192, 192, 4), (512, 6144, 4096): (128, 128, 1),
    (4096, 6144, 4096): (256, 192, 1),
    (16, 4096, 4096): (1, 8, 1), (64, 4096, 4096): (64, 64, 4), (128, 4096, 4096): (128, 64, 4),
    (1003, 4096, 4096): (128, 128, 1), (4096, 4096, 4096): (256, 256, 1),
    (1, 28672, 4096): (64, 128, 1), (64, 28672, 4096): (64, 128, 1), (128, 28672, 4096): (128, 128, 1),
    (256, 28672, 4096): (256, 128, 1), (512, 28672, 4096): (256, 256, 1), (4096, 28672, 4096): (256, 256, 1),
    (8, 4096, 14336): (1, 8, 1), (16, 4096, 14336): (2, 4, 2), (64, 4096, 14336): (64, 128, 8),
    (128, 4096, 14336): (128, 128, 8), (256, 4096, 14336): (256, 128, 8), (512, 4096, 14336): (256, 128, 4),
    # Qwen2.5-7B
    (64, 4608, 3584): (64, 64, 3), (1003, 4608, 3584): (128, 160, 1), (64, 3584, 3584): (64, 64, 4),
    (1, 37888, 3584): (64, 64, 1), (384, 37888, 3584): (192, 192, 1), (1003, 37888, 3584): (256, 256, 1),
    (64, 3584, 18944): (64, 128, 8), (512, 3584, 18944): (256, 128, 4), (2048, 3584, 18944): (256, 256, 2),
    # Qwen2.5-0.5B
    (64, 1152, 896): (1, 8, 1), (1003, 896, 896): (64, 64, 1), (1, 9728, 896): (4, 2, 1),
    (64, 9728, 896): (64, 64, 1), (96, 9728, 896): (128, 64, 1), (1003, 896, 4864): (128, 128, 4),
    # the head
    (1, 128256, 4096): (64, 128, 1), (64, 128256, 4096): (64, 128, 1), (512, 128256, 4096): (256, 256, 1),
}


@pytest.mark.parametrize("shape", sorted(PICKS))
def test_projections_get_the_measured_plans(shape):
    assert capi.gemm_plan(*shape)[:3] == PICKS[shape]


@pytest.mark.parametrize("mistake", ["fill", "limit", "rounds", "odd", "ragged"])
def test_planted_mistake_is_caught(mistake):
    """A replica with one condition changed must disagree with the library on
    some size: the comparison above can see each of them."""
    assert any(capi.gemm_plan(*s) != replica_plan(*s, mistake=mistake) for s in random_shapes(5000, 5))


def test_plan_validation():
    L = capi.lib()
    assert L.dk_gemm_tn_plan(0, 8, 64, 1, None) == capi.HIP_ERROR_INVALID_VALUE
    with pytest.raises(ValueError, match="positive"):
        capi.gemm_plan(0, 8, 64)
    with pytest.raises(ValueError, match="positive"):
        capi.gemm_plan(4, 8, -8)


# One shape per (row tiles, workgroup shape, split or not) that the skinny plan
# reaches, each with N not a multiple of the workgroup's columns. The plan of
# some of them is a tile; the skinny kernel then runs where the row strides
# rule the tiles out (as in tests/test_gemm_splitk.py, which runs every one of
# them against the oracle that way).
COVERAGE_SHAPES = [
    (1, 8, 520), (1, 8, 1032), (1, 4101, 520), (1, 2050, 1032), (1, 8200, 520), (1, 4101, 1032),
    (1, 20000, 520), (1, 8200, 1032), (1, 28600, 520), (1, 8200, 2056), (1, 28680, 520), (16, 6150, 8200),
    (17, 8, 520), (17, 8, 1032), (17, 4101, 520), (17, 2050, 1032), (17, 8200, 520), (17, 4101, 1032),
    (17, 20000, 520), (17, 8200, 1032), (17, 28600, 520), (17, 8200, 2056), (17, 28680, 520), (18, 9622, 1624),
    (33, 8, 520), (33, 8, 1032), (33, 4101, 520), (33, 2050, 1032), (35, 13089, 520), (33, 4101, 1032),
    (33, 20000, 520), (55, 12225, 2656), (33, 28600, 520), (42, 12474, 3128), (33, 28680, 520), (64, 8, 8200),
]
# The 64-row tiles at M <= 64: columns, split or not, below and from M = 32, ragged N.
DECODE_TILE_SHAPES = [
    (44, 506, 64), (23, 649, 64), (34, 2072, 1032), (8, 4147, 1056),
    (55, 16631, 64), (25, 16572, 64), (34, 8480, 1616), (2, 8323, 1544),
]


def test_coverage_shapes_reach_every_plan():
    reached = set()
    for M, N, K in COVERAGE_SHAPES:
        wn, wk, s, _ = replica_skinny_plan(M, N, K)
        assert N % (16 * wn) != 0, (M, N, K)
        reached.add((1 if M <= 16 else (2 if M <= 32 else 4), wn, wk, s > 1))
    assert reached == {(mt, wn, wk, split) for mt in (1, 2, 4) for wn, wk in SHAPES for split in (False, True)}
    tiles = set()
    for M, N, K in DECODE_TILE_SHAPES:
        bm, bn, s, _ = capi.gemm_plan(M, N, K)
        assert bm == 64 and N % bn != 0, (M, N, K)
        tiles.add((bn, s > 1, M < 32))
    assert tiles == {(bn, split, below) for bn in (64, 128) for split in (False, True) for below in (False, True)}
