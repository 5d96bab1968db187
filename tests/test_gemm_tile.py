"""The tile that runs a gemm_tn plan (``dk_gemm_tn_tile``): the library's choice
against a restatement of its time model on the CPU, and on the GPU one set of
shapes per tile -- edges, remainders, short and ragged K, K splits, rotated
walks -- against an fp32 GEMM at the parity bar.

The plan (``dk_gemm_tn_plan``) sets the workspace and the most K splits; the
tile keeps to both, so an unsplit plan runs unsplit whatever the tile.
"""

import ctypes
import random

import pytest
import torch

from decodekernels_amd import capi

# (rows, columns, us per 64-column slice, us per tile, part-filled rounds count whole)
TILES = [
    (256, 256, 1.233, 5.10, False), (256, 192, 1.026, 6.34, False), (192, 256, 0.993, 5.64, False),
    (256, 128, 0.820, 3.59, False), (128, 256, 0.821, 4.25, False), (128, 128, 0.516, 1.51, False),
    (128, 160, 0.622, 2.77, False), (128, 64, 0.344, 1.54, False), (64, 64, 0.184, 0.83, True),
    (64, 128, 0.368, 2.00, False), (192, 192, 0.900, 6.00, False), (192, 224, 1.134, 6.20, False),
    (256, 224, 1.415, 5.91, False),
]
# start, split, per_split, partials, memory, part_fill, last_round
MODEL = (2.61, 1.42, 0.234, 7.27e6, 4.99e6, 0.62, 1.148)
DECODE_TILES = [(64, 64, 0.207, 0.519, True), (64, 128, 0.370, 1.027, False)]
DECODE_MODEL = (2.4, 1.672, 0.222, 8.24e6, 6.393e6, 0.636, 1.0)


def _rotation(tiles_m, tiles_n, splits, K):
    return 1 if splits == 1 and tiles_m == 1 and tiles_n >= 128 and K >= 1536 and K % 64 == 0 else 0


def _fastest(model, tiles, M, N, K, max_splits, rounds_up=True):
    start, split, per_split, partials, memory, part_fill, last_round = model
    best, best_t = None, -1.0
    mn = float(M) * N
    mem = 2.0 * (float(M) * K + float(N) * K + mn) / memory
    mem4 = mem * mem * mem * mem
    for bm, bn, slice_us, tile_us, whole in tiles:
        tm, tn = -(-M // bm), -(-N // bn)
        for s in (1, 2, 3, 4, 6, 8):
            ks = K
            if s > 1:
                if s > max_splits or tm * tn > 256 or K // s < 512:
                    break
                ks = -(-(-(-K // s)) // 64) * 64
                if -(-K // ks) != s:
                    continue
            full, rem = divmod(tm * tn * s, 256)
            rounds = float(full)
            if rem > 0:
                part = 1.0 if whole and rounds_up else part_fill + (1.0 - part_fill) * float(rem) / 256
                rounds += (last_round if full > 0 and not whole else 1.0) * part
            t = start + float(-(-ks // 64)) * slice_us * rounds + tile_us * float(full + (rem > 0))
            if s > 1:
                t += split + per_split * s + s * mn * 8.0 / partials
            t = t * t * t * t + mem4
            if best_t < 0 or t < best_t:
                best, best_t = (bm, bn, s, _rotation(tm, tn, s, K)), t
    return best


def replica(M, N, K, with_workspace=True, **mistake):
    plan = capi.gemm_plan(M, N, K, with_workspace)
    if M > 64:
        return _fastest(MODEL, TILES, M, N, K, plan[2], **mistake)
    t64, t128 = -(-N // 64), -(-N // 128)
    if K >= 2048 and 192 <= t64 <= 256:
        return (64, 64, 1, _rotation(1, t64, 1, K))
    if K >= 2048 and plan[2] == 1 and t64 > 256 and 4 * t128 >= 768 * -(-t128 // 256):
        return (64, 128, 1, _rotation(1, t128, 1, K))
    if plan[2] >= 3:
        tile = _fastest(DECODE_MODEL, DECODE_TILES, M, N, K, plan[2], **mistake)
        wide_ok = tile[1] == 64 or M >= 32 or K >= 8192
        if wide_ok and -(-N // tile[1]) * tile[2] >= 128:
            return tile
    return (plan[0], plan[1], plan[2], _rotation(1, -(-N // plan[1]), plan[2], K) if plan[0] == 64 else 0)


def _random_shapes(n, seed):
    rng = random.Random(seed)
    for _ in range(n):
        M = rng.choice([rng.randint(1, 64), rng.randint(65, 600), rng.randint(65, 5000)])
        N = rng.choice([rng.randint(1, 2000), rng.randint(1, 30000), rng.randint(12000, 130000)])
        yield M, N, 8 * rng.choice([rng.randint(1, 64), rng.randint(1, 3000)])


def test_library_picks_like_the_replica():
    for M, N, K in _random_shapes(20000, 11):
        for ws in (True, False):
            tile = capi.gemm_tile(M, N, K, ws)
            assert tile == replica(M, N, K, ws), (M, N, K, ws)
            # within the plan's workspace, and unsplit where the plan is
            assert tile[2] <= capi.gemm_plan(M, N, K, ws)[2]


def test_planted_mistake_is_caught():
    assert any(capi.gemm_tile(*s) != replica(*s, rounds_up=False) for s in _random_shapes(5000, 12))


def test_tile_validation():
    with pytest.raises(ValueError, match="positive"):
        capi.gemm_tile(0, 8, 64)
    assert capi.lib().dk_gemm_tn_tile(4, 8, 64, 1, None) == capi.HIP_ERROR_INVALID_VALUE


# Tile, K splits, rotated -> shapes (M, N, K) that pick it: whole tiles, ragged M
# and N (odd N: scalar stores), K of one to five slices, K ending inside a slice.
SHAPES = {
    (64, 64, False, 0): [(165, 1, 8), (84, 1, 152), (65, 131, 24), (1, 37488, 136), (1, 34369, 80), (1, 37679, 8)],
    (64, 64, False, 1): [(24, 15886, 4672), (64, 15991, 2176), (59, 16292, 2688), (41, 38630, 2816)],
    (64, 64, True, 0): [(103, 1, 1456), (65, 7, 1488), (103, 7, 2048), (1, 2720, 2712), (256, 320, 1504)],
    (64, 128, False, 0): [
        (32, 17749, 8), (34, 17000, 72), (33, 16549, 136), (33, 16524, 216), (33, 16706, 264), (135, 8301, 672),
    ],
    (64, 128, False, 1): [(1, 25857, 2624), (5, 25198, 4288), (23, 27676, 3712), (51, 27272, 3264)],
    (64, 128, True, 0): [(1, 10240, 8192), (3, 10113, 8200), (32, 11709, 3328), (277, 1812, 5184)],
    (128, 64, False, 0): [
        (66, 9455, 8), (133, 5511, 8), (72, 8557, 72), (194, 4281, 136), (67, 8375, 136), (385, 2325, 16),
    ],
    (128, 64, False, 1): [(99, 9697, 1792), (111, 15145, 1728), (108, 10818, 3008), (123, 15164, 3584)],
    (128, 64, True, 0): [(65, 4180, 3584), (68, 4201, 3528), (257, 1748, 4544), (640, 960, 5552)],
    (128, 128, False, 0): [
        (72, 17476, 8), (157, 8460, 8), (257, 5486, 8), (67, 16867, 208), (137, 10887, 136), (132, 8229, 16),
    ],
    (128, 128, False, 1): [(101, 17903, 2432), (128, 28416, 1536), (120, 24116, 2112), (93, 26141, 3200)],
    (128, 128, True, 0): [(67, 2898, 6488), (68, 2749, 6768), (86, 2747, 7168), (385, 2331, 3112), (256, 4352, 3360)],
    (128, 160, False, 0): [
        (66, 34011, 8), (140, 16583, 8), (67, 33182, 208), (1280, 3680, 6760), (72, 33510, 72), (129, 17819, 200),
    ],
    (128, 160, False, 1): [(87, 32892, 2112), (118, 34385, 1792), (74, 39464, 2560), (98, 33702, 3712)],
    (128, 160, True, 0): [(129, 5740, 4544), (131, 5511, 5312), (138, 6207, 4552), (1354, 1540, 5440)],
    (128, 256, False, 0): [(263, 16610, 272), (264, 17761, 264), (257, 20614, 320), (259, 16199, 576)],
    (128, 256, True, 0): [(66, 17103, 4984), (67, 16458, 5760), (69, 21476, 5912), (257, 5729, 6520)],
    (192, 192, False, 0): [(130, 32809, 1288), (145, 33625, 1408), (1445, 12225, 392), (1397, 12206, 1152)],
    (192, 192, False, 1): [(156, 35872, 2112), (136, 33759, 2752), (137, 39374, 2688), (160, 36479, 2816)],
    (192, 192, True, 0): [(132, 8995, 5664), (136, 9479, 6848), (135, 16573, 6528), (1537, 2629, 6952)],
    (192, 256, False, 0): [
        (129, 35791, 136), (275, 22700, 136), (131, 36961, 576), (384, 26880, 4104), (130, 34397, 208),
        (259, 22417, 264),
    ],
    (192, 256, False, 1): [(144, 39011, 1792), (156, 38208, 1728), (186, 36458, 1536), (151, 39337, 1856)],
    (192, 256, True, 0): [
        (140, 5626, 6384), (137, 6259, 6432), (130, 6415, 6784), (192, 11520, 6008), (385, 8689, 6120),
    ],
    (256, 128, False, 0): [
        (140, 32026, 72), (133, 22341, 136), (142, 25547, 576), (132, 23152, 264), (512, 16256, 128),
        (257, 14131, 248),
    ],
    (256, 128, False, 1): [(205, 22543, 2048), (179, 26269, 2560), (231, 22504, 3200), (226, 32416, 2688)],
    (256, 128, True, 0): [(134, 7203, 6136), (135, 7240, 6720), (728, 2925, 5184), (230, 13347, 7024)],
    (256, 192, False, 0): [
        (196, 33045, 784), (195, 34882, 832), (390, 22181, 840), (256, 35904, 896), (407, 22700, 896),
    ],
    (256, 192, False, 1): [(200, 36411, 1792), (208, 37390, 1984), (256, 39090, 1728), (244, 35619, 2176)],
    (256, 192, True, 0): [(385, 5706, 5344), (386, 5459, 5640), (400, 5778, 5952), (204, 23697, 4480)],
    (256, 256, False, 0): [
        (392, 25337, 8), (129, 33092, 72), (265, 21840, 80), (389, 16817, 264), (257, 22915, 88), (199, 33686, 576),
    ],
}


@pytest.mark.parametrize("tile", sorted(SHAPES))
def test_shapes_pick_their_tile(tile):
    for shape in SHAPES[tile]:
        got = capi.gemm_tile(*shape)
        assert (got[:2], got[2] > 1, got[3]) == (tile[:2], tile[2], tile[3]), (shape, got)


@pytest.mark.gpu
@pytest.mark.parametrize("bf16", [True, False])
@pytest.mark.parametrize("tile", sorted(SHAPES))
def test_tile_against_fp32(tile, bf16):
    import decodekernels_amd as dk
    from parity import assert_max_abs, gemm_f32_gpu

    dtype = torch.bfloat16 if bf16 else torch.float16
    for M, N, K in SHAPES[tile]:
        print(f"gemm {M}x{N}x{K} {dtype} tile {tile}", flush=True)
        g = torch.Generator(device="cuda").manual_seed(M + N + K)
        # Rows 8 elements longer than K: what lies past a row must not be read into it.
        a = torch.randn(M, K + 8, generator=g, device="cuda", dtype=dtype)[:, :K]
        b = (torch.randn(N, K + 8, generator=g, device="cuda", dtype=dtype) / K**0.5)[:, :K]
        bias = torch.randn(N, generator=g, device="cuda", dtype=dtype)
        out = torch.full((M, N + 3), float("nan"), device="cuda", dtype=dtype)
        torch.ops.decode_kernels.gemm_tn(out[:, :N], a, b, bias)
        assert_max_abs(out[:, :N], gemm_f32_gpu(a, b, bias), dtype, f"gemm {M}x{N}x{K} tile {tile}")
        assert out[:, N:].isnan().all()
        c = dk.gemm(a.contiguous(), b.contiguous())
        assert_max_abs(c, gemm_f32_gpu(a, b), dtype, f"gemm {M}x{N}x{K} tile {tile}, no bias")
        if not tile[2]:  # unsplit: the entry point without a workspace gives the same bits
            d = torch.empty(M, N, device="cuda", dtype=dtype)
            rc = capi.lib().dk_gemm_tn(capi.dtype_code(dtype), a.data_ptr(), b.data_ptr(), None, d.data_ptr(), M, N, K,
                                       K + 8, K + 8, N, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
            assert rc == 0, capi.last_error()
            torch.cuda.synchronize()
            assert torch.equal(c, d)


@pytest.mark.gpu
@pytest.mark.parametrize("tile, shape", [((64, 64), (192, 3008, 16)), ((128, 160), (1280, 3680, 6760)),
                                         ((256, 128), (512, 16256, 128)), ((256, 256), (257, 22915, 88))])
def test_output_rows_of_any_alignment(tile, shape):
    """Stores of 16, 8, 4 and 2 bytes: output rows of every stride modulo 8
    starting at every element offset modulo 8, odd and even N; the elements
    around each row keep their values."""
    from parity import assert_max_abs, gemm_f32_gpu

    M, N, K = shape
    for n in (N, N - 1, N - 2):
        assert capi.gemm_tile(M, n, K)[:2] == tile
        g = torch.Generator(device="cuda").manual_seed(n)
        a = torch.randn(M, K, generator=g, device="cuda", dtype=torch.bfloat16)
        b = torch.randn(n, K, generator=g, device="cuda", dtype=torch.bfloat16) / K**0.5
        bias = torch.randn(n, generator=g, device="cuda", dtype=torch.bfloat16)
        want = gemm_f32_gpu(a, b, bias)
        for pad, at in [(0, 0), (0, 1), (1, 0), (2, 2), (3, 3), (4, 4), (5, 1), (6, 2), (7, 5), (8, 6), (8, 8)]:
            print(f"gemm {M}x{n}x{K} tile {tile} row stride {n + pad}, first element {at}", flush=True)
            flat = torch.full((at + M * (n + pad) + 8,), float("nan"), device="cuda", dtype=torch.bfloat16)
            out = flat[at : at + M * (n + pad)].view(M, n + pad)[:, :n]
            torch.ops.decode_kernels.gemm_tn(out, a, b, bias)
            assert_max_abs(out, want, torch.bfloat16, f"gemm {M}x{n}x{K}, row stride {n + pad}, first element {at}")
            assert int(flat.isnan().sum()) == at + M * pad + 8
