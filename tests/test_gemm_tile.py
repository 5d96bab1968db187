"""The tiles of gemm_tn, one set of sizes per tile -- edges, remainders, short and
ragged K, K splits, rotated walks (``dk_gemm_tn_tile``) -- against an fp32 GEMM at
the parity bar on the GPU; on the CPU, that each size runs the tile it stands for.
"""

import ctypes

import pytest
import torch

from decodekernels_amd import capi
from test_gemm_plan import TILES, random_shapes, runs_tile


def test_tile_is_the_plan_and_its_rotation():
    for M, N, K in random_shapes(10000, 11):
        for ws in (True, False):
            tile, plan = capi.gemm_tile(M, N, K, ws), capi.gemm_plan(M, N, K, ws)
            assert tile[:3] == plan[:3]
            one_row = runs_tile(plan) and M <= plan[0] and -(-N // plan[1]) >= 128
            assert tile[3] == (1 if one_row and plan[2] == 1 and K >= 1536 and K % 64 == 0 else 0), (M, N, K, ws)


def test_every_tile_runs():
    """Every compiled tile shape is picked, split and unsplit (the two of M <= 64 among them)."""
    kinds = {(tile[:2], tile[2]) for tile in SHAPES}
    assert kinds == {((bm, bn), split) for bm, bn, *_ in TILES for split in (False, True)}


def test_tile_validation():
    with pytest.raises(ValueError, match="positive"):
        capi.gemm_tile(0, 8, 64)
    assert capi.lib().dk_gemm_tn_tile(4, 8, 64, 1, None) == capi.HIP_ERROR_INVALID_VALUE


# Tile, K splits, rotated -> shapes (M, N, K) that pick it: whole tiles, ragged M
# and N (odd N: scalar stores), K of one to five slices, K ending inside a slice.
SHAPES = {
    (64, 64, False, 0): [(165, 1, 8), (84, 1, 152), (17, 858, 88), (7, 15371, 280), (155, 1970, 248), (65, 131, 24)],
    (64, 64, False, 1): [(32, 11709, 3328), (24, 15886, 4672), (64, 15991, 2176), (59, 16292, 2688), (41, 38630, 2816)],
    (64, 64, True, 0): [(103, 1, 1456), (65, 7, 1488), (103, 7, 2048), (256, 320, 1504)],
    (64, 128, False, 0): [(1, 37679, 8), (1, 34369, 80), (1, 37488, 136), (33, 16706, 264), (47, 17033, 256)],
    (64, 128, False, 1): [(1, 25857, 2624), (5, 25198, 4288), (23, 27676, 3712), (51, 27272, 3264)],
    (64, 128, True, 0): [(24, 20752, 3456), (37, 19352, 2416), (18, 18702, 5264), (277, 1812, 5184), (55, 9179, 6392)],
    (128, 64, False, 0): [
        (66, 9455, 8), (385, 2325, 16), (72, 8557, 72), (67, 8375, 136), (71, 14183, 248), (340, 3703, 264),
    ],
    (128, 64, False, 1): [(99, 9697, 1792), (111, 15145, 1728), (123, 15164, 3584)],
    (128, 64, True, 0): [(65, 4180, 3584), (68, 4201, 3528), (117, 5032, 3008), (210, 2638, 4192), (404, 1305, 4800)],
    (128, 128, False, 0): [
        (72, 17476, 8), (137, 10887, 136), (67, 16867, 208), (294, 10769, 112), (185, 11933, 304), (400, 5778, 5952),
    ],
    (128, 128, False, 1): [(101, 17903, 2432), (128, 28416, 1536), (120, 24116, 2112), (93, 26141, 3200)],
    (128, 128, True, 0): [(67, 2898, 6488), (68, 2749, 6768), (385, 2331, 3112), (131, 5511, 5312), (130, 6415, 6784)],
    (128, 160, False, 0): [
        (66, 34011, 8), (129, 17819, 200), (247, 19966, 96), (1851, 2337, 192), (244, 19598, 304), (135, 16573, 6528),
    ],
    (128, 160, False, 1): [(87, 32892, 2112), (118, 34385, 1792), (74, 39464, 2560), (98, 33702, 3712)],
    (128, 160, True, 0): [(138, 6207, 4552), (278, 3781, 4384), (66, 17103, 4984), (67, 16458, 5760)],
    (128, 256, False, 0): [
        (625, 12737, 16), (603, 12388, 112), (594, 13046, 136), (595, 12382, 1024), (638, 12664, 976),
        (578, 12876, 2944),
    ],
    (128, 256, True, 0): [(66, 19156, 3248), (67, 21368, 5120), (69, 21476, 5912)],
    (192, 192, False, 0): [
        (132, 34762, 8), (129, 33092, 72), (293, 18540, 192), (263, 16610, 272), (279, 23607, 248), (131, 36961, 576),
    ],
    (192, 192, False, 1): [
        (144, 39011, 1792), (156, 38208, 1728), (156, 35872, 2112), (136, 33759, 2752), (137, 39374, 2688),
        (160, 36479, 2816),
    ],
    (192, 192, True, 0): [(129, 5740, 4544), (132, 8995, 5664), (257, 5729, 6520), (192, 11520, 6008)],
    (192, 256, False, 0): [
        (292, 32535, 8), (274, 27602, 96), (389, 16817, 264), (384, 29893, 152), (783, 10211, 240), (290, 28796, 304),
    ],
    (192, 256, True, 0): [(133, 18632, 5312), (1295, 3784, 2824)],
    (256, 128, False, 0): [
        (208, 29413, 40), (203, 24821, 104), (132, 23152, 264), (213, 29248, 136), (171, 30010, 248),
        (197, 26551, 248),
    ],
    (256, 128, False, 1): [
        (204, 23697, 4480), (205, 22543, 2048), (213, 20560, 4416), (226, 32416, 2688), (231, 22504, 3200),
        (215, 20556, 4544),
    ],
    (256, 128, True, 0): [(1615, 880, 5632), (1354, 1540, 5440), (251, 10593, 6920)],
    (256, 192, False, 0): [
        (238, 32773, 288), (256, 35904, 896), (199, 33686, 576), (229, 38988, 280), (196, 33045, 784),
        (195, 34882, 832),
    ],
    (256, 192, False, 1): [(200, 36411, 1792), (208, 37390, 1984), (256, 39090, 1728), (244, 35619, 2176)],
    (256, 192, True, 0): [
        (386, 5612, 5696), (210, 11528, 6016), (197, 12064, 6376), (201, 11225, 7096), (1730, 1600, 6704),
    ],
    (256, 256, False, 0): [(392, 25337, 8), (434, 29246, 104), (227, 35369, 208), (1162, 9994, 144), (400, 27892, 296)],
    (256, 256, True, 0): [(194, 16468, 4128), (221, 16860, 4376), (197, 20604, 4904), (1280, 3680, 6760)],
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
@pytest.mark.parametrize("tile, shape", [((64, 64), (192, 3008, 16)), ((128, 160), (129, 17816, 200)),
                                         ((256, 128), (132, 23152, 264)), ((256, 256), (392, 25336, 8))])
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
