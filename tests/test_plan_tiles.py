"""Which tiles the matrix-core kernels run on where two were measured against each other: sizes on both sides of a line.  No GPU needed."""
import pytest

import morello_amd as M

TYPES = {"u8": (M.u8, M.i8, M.i32), "i8": (M.i8, M.i8, M.i32), "bf16": (M.bf16, M.bf16, M.f32)}


@pytest.mark.parametrize("types,b,c,f,hw,fs,tile", [
    ("u8", 22, 16, 176, 114, 3, "Tile<256, 256"),     # two steps; 256 x 256 pads the filters by 80, 128 x 64 by 16
    ("u8", 22, 48, 208, 40, 3, "Tile<256, 256"),
    ("u8", 7, 16, 272, 72, 3, "RA = 4, RB = 2"),      # ... by 240, 48
    ("u8", 27, 16, 288, 71, 3, "Tile<256, 256"),      # two steps, twenty rounds of 128 x 64
    ("u8", 27, 32, 288, 71, 3, "RA = 4, RB = 2"),     # three
    ("bf16", 22, 16, 176, 60, 5, "RA = 4, RB = 2"),
    ("u8", 16, 112, 160, 55, 3, "Tile<256, 256"),     # eight steps
    ("u8", 18, 208, 240, 71, 3, "Tile<256, 256"),     # several rounds of 128 x 128
    ("i8", 18, 176, 192, 79, 3, "Tile<256, 256"),     # ... of 128 x 192
    ("u8", 5, 208, 96, 85, 5, "Tile<128, 128"),       # 283 tiles of 128 x 128
    ("u8", 10, 288, 320, 28, 5, "RA = 4, RB = 4"),    # 186
    ("u8", 22, 208, 64, 46, 3, "Tile<64, 64"),        # 364 tiles of 128 x 64
    ("u8", 20, 208, 64, 40, 3, "RA = 4, RB = 2"),     # 250
    ("u8", 26, 208, 64, 46, 3, "RA = 4, RB = 2"),     # 430
])
def test_windows(types, b, c, f, hw, fs, tile):
    p = M.Conv([b, f, c, hw, hw, fs, fs], TYPES[types]).plan()
    assert p.kernels == ["k_gemm"] and tile in p.steps[0].kernel, p


KT = M.layout(0, 2, 1)


@pytest.mark.parametrize("types,b,m,k,n,nk,tile", [
    # 128 x 64 and 128 x 128 of row-major operands, the last column of tiles 8 or 16 wide
    ("bf16", 1, 1153, 832, 904, False, "RB = 2, SLOTS"),
    ("bf16", 1, 1153, 768, 904, False, "Tile<64, 64"),
    ("bf16", 2, 1153, 776, 456, False, "RB = 2, SLOTS"),
    ("u8", 2, 1153, 1680, 464, False, "RB = 2, SLOTS"),
    ("u8", 2, 1153, 1664, 464, False, "Tile<64, 64"),
    ("bf16", 1, 1985, 1792, 1160, False, "RB = 4, SLOTS"),
    ("bf16", 1, 1985, 1728, 1160, False, "Tile<128, 128"),
    ("u8", 1, 1985, 3584, 1168, False, "RB = 4, SLOTS"),
    ("u8", 1, 1985, 3456, 1168, False, "Tile<128, 128"),
    ("u8", 3, 300, 4608, 1808, False, "RB = 4, SLOTS"),
    # 128 x 128: rows of K in whole cache lines, and not
    ("i8", 1, 1985, 3584, 1264, False, "RB = 4, SLOTS"),
    ("i8", 1, 1985, 3600, 1280, False, "Tile<128, 128"),
    ("i8", 3, 626, 3584, 2144, True, "RB = 4, SLOTS"),
    ("i8", 3, 626, 3600, 2144, True, "Tile<128, 128"),
    ("i8", 3, 626, 3600, 2144, False, "Tile<128, 128"),
    ("i8", 3, 626, 7600, 2144, False, "RB = 4, SLOTS"),
    ("i8", 3, 184, 4112, 3664, False, "RB = 4, SLOTS"),    # (the other choice is 64 x 64)
    ("u8", 3, 626, 3600, 2144, False, "RB = 4, SLOTS"),
    ("bf16", 2, 1109, 1792, 1504, True, "RB = 4, SLOTS"),
    ("bf16", 2, 1109, 1768, 1504, True, "Tile<128, 128"),
    ("bf16", 2, 1109, 1768, 1504, False, "RB = 4, SLOTS"),
    ("bf16", 2, 1109, 2024, 1504, True, "RB = 4, SLOTS"),
    ("i8", 1, 814, 7296, 2400, True, "RB = 4, SLOTS"),     # at most 512 tiles of 64 x 64
    ("i8", 1, 814, 7312, 2400, True, "Tile<64, 64"),
    ("u8", 1, 814, 7312, 2400, True, "RB = 4, SLOTS"),
])
def test_middling_matmuls(types, b, m, k, n, nk, tile):
    p = M.Matmul([b, m, k, n], TYPES[types], [None, KT if nk else None, None]).plan()
    assert len(p.steps) == 1 and tile in p.steps[0].kernel, p


@pytest.mark.parametrize("types,m,k,n,kernel", [
    # Rows of N on the 64 x 64 tile fed straight into LDS, from seven steps of i8, six of u8, nine of bf16
    ("i8", 193, 768, 208, "k_gemm"), ("i8", 193, 896, 208, "k_gemm_ring"), ("u8", 193, 768, 208, "k_gemm_ring"), ("u8", 193, 640, 208, "k_gemm"),
    ("bf16", 422, 512, 880, "k_gemm"), ("bf16", 422, 520, 880, "k_gemm_ring"),
    # Slices of a long K that are not all equal: 230 tiles of 64 x 64, 90 and 75; two rows of tiles
    ("i8", 262, 9584, 2896, "k_gemm"), ("i8", 262, 6128, 2896, "k_gemm_ring"), ("u8", 932, 13392, 336, "k_gemm"), ("u8", 932, 10128, 336, "k_gemm_ring"),
    ("i8", 932, 13392, 304, "k_gemm_ring"), ("u8", 106, 9264, 2960, "k_gemm"), ("i8", 77, 11536, 2464, "k_gemm"), ("i8", 66, 9264, 640, "k_gemm_ring"),
])
def test_rows_of_n(types, m, k, n, kernel):
    p = M.Matmul([1, m, k, n], TYPES[types]).plan()
    assert p.kernels[0] == kernel, p
