"""Which kernels a Spec goes to where two routes meet, by its plan (no GPU): Specs that one of them cannot
take, or takes at many times the other's cost."""
import math

import numpy as np
import pytest

import morello_amd as M

KT = M.layout(0, 2, 1)


@pytest.mark.parametrize("batch,k", [(1 << 27, 1), ((1 << 27) + 1, 3)])
def test_operands_too_many_for_padded_copies_stay_as_they_are(batch, k):
    """2^27 right operands of up to 16 rows of a chunk each are 2^31 chunks, more than the copy numbers."""
    p = M.Matmul([batch, 1, k, 1], (M.u8, M.i8, M.i32)).plan()
    assert p.kernels[-1] == "k_matmul_generic"


@pytest.mark.parametrize("shape,dst,kernel,vec", [
    ([45, 1963, 4], (0, 2, 1), "k_move_gather", 1), ([1, 1024, 1024], (0, 1, 2, (1, 16)), "k_move_gather", 1),
    ([300, 200, 16], (1, 0, 2), "k_move_runs", 4), ([2, 64, 2050], (1, 0, 2), "k_move_runs", 2),
    ([7340, 12, 16], (1, 0, 2), "k_move_runs", 4), ([8, 6, 5, 6212], (1, 2, 0, 3), "k_move_runs", 4),   # 5.6 MB in runs of 64 bytes and more
])
def test_small_moves_take_no_tiles(shape, dst, kernel, vec):
    """An element (or vector) a thread up to 2^20 elements, and up to 16 MB in long runs: the tiles' arithmetic made
    these 1.5 to 2 times as long."""
    layout = M.layout(*[(d[0], M.Packed(d[1])) if isinstance(d, tuple) else d for d in dst])
    p = M.Move(shape, (M.f32, M.f32), layouts=[None, layout]).plan()
    threads = math.prod(shape) // vec
    assert p.kernels == [kernel] and p.steps[0].grid == ((threads + 255) // 256, 1, 1)


def test_large_moves_take_tiles():
    for shape, dst in (([45, 19630, 4], (0, 2, 1)), ([1, 2048, 16384], (0, 2, 1, (2, M.Packed(16))))):
        p = M.Move(shape, (M.f32, M.bf16), layouts=[None, M.layout(*dst)]).plan()
        assert p.steps[0].grid[0] <= math.prod(shape) // 2048


@pytest.mark.parametrize("types", [(M.f32, M.f32), (M.f32, M.bf16), (M.bf16, M.bf16)])
@pytest.mark.parametrize("inner", [8, 16])
def test_tiles_of_short_digits_fill_their_workgroups(types, inner):
    """Four digits of two leave a tile of 16 vectors, most of a workgroup idle (f32 [40000, 2, 2, 2, 8]: 62.5 us, 4.8
    without tiles), and past 2^24 of them more workgroups than a launch takes."""
    for n in (400000, (1 << 31) // (8 * inner) - 1):
        shape = [n, 2, 2, 2, inner]
        p = M.Move(shape, types, layouts=[None, M.layout(0, 3, 2, 1, 4)]).plan()
        assert p.kernels == ["k_move_runs"]
        assert p.steps[0].grid[0] * 192 <= math.prod(shape) // 4 + 256 and p.steps[0].grid[0] < 1 << 24


@pytest.mark.parametrize("types,shape", [
    ("bf16", [1, 1, 64000, 14]), ("bf16", [1, 44, 9600, 16]), ("f32", [1, 1, 64000, 64]), ("f32", [1, 4, 9792, 64]), ("bf16", [1, 1, 16000, 64]), ("u8", [1, 4, 320000, 3]),   # a long K, few columns
    ("f32", [12, 53, 76, 1533]), ("bf16", [1, 59, 64, 13690]), ("u8", [62, 3, 64, 4096]),   # a short K, thousands of blocks
])
def test_few_rows_leave_k_gemm_skinny_where_it_is_the_slower_one(types, shape):
    dts = {"bf16": (M.bf16, M.bf16, M.f32), "f32": (M.f32,) * 3, "u8": (M.u8, M.i8, M.i32)}[types]
    kernels = M.Matmul(shape, dts, layouts=[None, KT, None]).plan().kernels
    assert "k_gemm_skinny" not in kernels and "k_matmul_generic" not in kernels


def test_few_rows_stay_with_k_gemm_skinny():
    for dts, shape in (((M.bf16, M.bf16, M.f32), [1, 1, 4096, 4096]), ((M.u8, M.i8, M.i32), [1, 4, 32767, 30]), ((M.bf16, M.bf16, M.f32), [1, 4, 10176, 16]), ((M.f32,) * 3, [18643, 3, 16, 16]), ((M.f32,) * 3, [2, 30, 64, 4000]),
                       ((M.f32,) * 3, [1, 1, 4096, 1000]), ((M.bf16, M.bf16, M.f32), [60, 53, 256, 153])):
        assert M.Matmul(shape, dts, layouts=[None, KT, None]).plan().kernels == ["k_gemm_skinny"], shape


@pytest.mark.parametrize("types,shape", [("f32", [1, 794, 27, 2728]), ("f32", [1, 1536, 16, 1585]), ("bf16", [1, 370, 34, 2386]), ("u8", [21, 1, 1891, 400])])
def test_small_problems_leave_k_gemm_tiny_where_it_is_the_slower_one(types, shape):
    dts = {"bf16": (M.bf16, M.bf16, M.f32), "f32": (M.f32,) * 3, "u8": (M.u8, M.i8, M.i32)}[types]
    kernels = M.Matmul(shape, dts).plan().kernels
    assert "k_gemm_tiny" not in kernels and "k_matmul_generic" not in kernels


def test_copies_of_a_short_k_are_no_taller_than_it():
    """Right operands of one to three rows were copied into 16."""
    for shape, most in (([1, 16, 3, 4825541], 16 << 20), ([1, 17, 1, 2111355], 4 << 20), ([47805, 1, 2, 187], 24 << 20)):
        assert M.Matmul(shape, (M.u8, M.i8, M.i32)).plan().scratch_bytes <= most
    p = M.Matmul([1, 1001, 2050, 4425], (M.bf16, M.bf16, M.bf16)).plan()   # a long one still ends on a whole chunk
    assert p.kernels == ["k_pad_rows_pair", "k_gemm_ring"]
    assert M.Matmul([1, 4518, 3787, 4543], (M.u8, M.i8, M.i32)).plan().kernels == ["k_pad_rows_pair", "k_gemm_wide"]
    for layout in (None, KT):   # ... which falls into equal slices
        assert M.Matmul([1, 384, 2559, 60], (M.u8, M.i8, M.i32), layouts=[None, layout, None]).plan().kernels == ["k_pad_rows_pair", "k_gemm", "k_sum_splits"]


@pytest.mark.parametrize("layout", [None, KT])
def test_a_right_operand_of_one_column_is_one_row(layout):
    """It has rows along either dim; along K they are the shorter ones by far once padded to chunks."""
    for dts, shape, scratch in (((M.f32,) * 3, [39287853, 3, 16, 1], 0), ((M.bf16, M.bf16, M.f32), [50000, 16, 16, 1], 0),
                                ((M.u8, M.i8, M.i32), [50000, 16, 16, 1], 0), ((M.f32,) * 3, [1, 16, 33864, 1], 1 << 20)):
        p = M.Matmul(shape, dts, layouts=[None, layout, None]).plan()
        assert p.scratch_bytes <= scratch and not {"k_pad_rows", "k_pad_rows_pair"} & set(p.kernels), (shape, p)
        assert ("k_matmul_generic" in p.kernels) == (shape[0] > 1), (shape, p)   # many short dot products: 64 x 64 tiles are mostly padding
    # neither way whole chunks: a copy of one row, not of one row an element
    p = M.Matmul([1, 300, 4001, 1], (M.bf16, M.bf16, M.f32), layouts=[None, layout, None]).plan()
    assert p.scratch_bytes < 300 * 4096 * 2 + 4096 * 2 + (1 << 20)


def test_columns_of_two_bytes_are_turned_not_padded():
    assert M.Matmul([1, 17, 2, 12613142], (M.i8, M.i8, M.i32), layouts=[None, KT, None]).plan().scratch_bytes <= 32 << 20
    assert M.Matmul([1, 16, 3, 400000], (M.u8, M.i8, M.i32), layouts=[None, KT, None]).plan().kernels == ["k_pad_rows_pair", "k_gemm"]   # a fifth: still one pass


@pytest.mark.parametrize("shape", [[1, 8192, 8192, 8192], [1, 2560, 2560, 2560], [1, 1001, 2050, 4425], [1, 300, 520, 416], [1, 2, 2048, 16384]])
def test_plans_count_bf16_results_as_two_bytes(shape):
    b, m, k, n = shape
    for dt, es in ((M.bf16, 2), (M.f32, 4)):
        step = M.Matmul(shape, (M.bf16, M.bf16, dt), layouts=[None, KT, None]).plan().steps[-1]
        whole = 8 * ((k + 7) // 8)   # (a copied K ends on a whole chunk)
        assert step.bytes in [2 * (m + n) * kk + es * m * n for kk in (k, whole)], (step, dt)


def test_the_two_forms_of_k_conv_windows_are_told_apart():
    pixels = M.Conv([32, 64, 3, 112, 112, 7, 7], (M.u8, M.i8, M.i32)).plan().steps[0].kernel
    windows = M.Conv([8, 32, 3, 110, 110, 5, 5], (M.f32, M.f32, M.f32)).plan().steps[0].kernel
    assert "PIXELS = true" in pixels and "PIXELS" not in windows


def test_padded_copies_of_up_to_a_million_chunks_go_one_to_a_thread():
    step = M.Matmul([1, 1500, 1000, 1500], (M.u8, M.i8, M.i32)).plan().steps[0]
    assert step.family == "k_pad_rows_pair" and step.grid[0] == (1500 * 64 + 255) // 256
    step = M.Matmul([1, 5003, 4001, 5001], (M.bf16, M.bf16, M.f32)).plan().steps[0]
    assert step.family == "k_pad_rows_pair" and step.grid[0] <= 5003 * 632 // 1024 + 1


def _fused(spec, tile_m, parts):
    return M.Action(spec, M._binding.ActionC(M.ActionKind.Fused, tile_m, 0, 0, parts, 0, 0, 0, 0.0))


@pytest.mark.parametrize("b,m,keys,d", [(4, 1, 564, 128), (16, 103, 767, 80), (13, 346, 1088, 80), (40, 90, 1024, 128), (16, 2048, 2048, 128)])
def test_fused_without_a_query_block_is_the_rules_choice(b, m, keys, d):
    """... of the form and its queries per workgroup, with the shares of the keys that the action names (none: one)."""
    spec = M.ComposeMSM(b, m, d, keys, d, layouts=[None, None, KT, None])
    rules = spec.plan().steps[0]
    for parts in (0, 1, 2):
        p = _fused(spec, 0, parts).plan()
        assert p.steps[0].kernel == rules.kernel and p.steps[0].grid == (rules.grid[0], max(1, parts), 1)
        assert p.kernels == ["k_attn", "k_attn_merge"][:max(1, parts)] and (p.scratch_bytes > 0) == (parts == 2)


@pytest.mark.parametrize("tile_m", [16, 32, 48, 256])
def test_fused_takes_the_query_blocks_it_documents(tile_m):
    for m, keys in ((1, 564), (2048, 2048)):
        spec = M.ComposeMSM(4, m, 128, keys, 128, layouts=[None, None, KT, None])
        with pytest.raises(M.MorelloError):
            _fused(spec, tile_m, 1).plan()


@pytest.mark.parametrize("shape,wide", [([1, 2048, 16384], True), ([1, 8192, 3072], False), ([2, 8192, 3072], False), ([2, 8192, 2048], True),
                                        ([3, 4097, 2048], True), ([8, 1024, 1536], False), ([4, 1, 700, 4096], True),
                                        ([1, 2048, 6144], False), ([1, 2048, 10240], False), ([1, 2048, 12288], False), ([1, 8192, 8192], True), ([1, 1024, 32768], False)])
def test_wide_narrowing_vectors_where_rows_lie_8_kib_apart(shape, wide):
    """... or 16, 32 or 64.  Rows, not the entries of a batch: two of 8192 x 3072 are a multiple of 8 KiB apart and their rows 12."""
    r = len(shape)
    strips = M.layout(*range(r - 2), r - 1, r - 2, (r - 1, M.Packed(16)))
    p = M.Move(shape, (M.f32, M.bf16), layouts=[None, strips]).plan()
    per_workgroup = np.prod(shape) / p.steps[0].grid[0]   # 1024 vectors of eight elements, or of four
    assert p.kernels == ["k_move_runs"] and (per_workgroup > 5000) == wide, p


@pytest.mark.parametrize("layout", [None, KT])
@pytest.mark.parametrize("shape", [[1, 960, 1000, 1000], [1, 1000, 1000, 1000], [2, 4089, 1000, 99], [1, 384, 2559, 120], [1, 3910, 10085, 125],
                                   [1, 300, 270, 290], [1, 1217, 281, 334], [3, 770, 136, 132]])
def test_int8_up_to_a_round_of_tiles_is_read_in_place(shape, layout):
    """... the last tile of a round, few columns and a short K among them."""
    p = M.Matmul(shape, (M.u8, M.i8, M.i32), layouts=[None, layout, None]).plan()
    assert p.kernels[0] == "k_gemm_ring" and "RA = 2" in p.steps[0].kernel, p


@pytest.mark.parametrize("dts,b,c,f,hw,fs,slices", [
    ("bf16", 24, 320, 320, 10, 3, 3), ("bf16", 4, 256, 288, 24, 3, 4), ("bf16", 22, 256, 96, 19, 3, 3), ("bf16", 14, 384, 112, 26, 3, 2),   # long chains: equal slices
    ("bf16", 3, 384, 160, 15, 5, 15), ("bf16", 14, 384, 64, 12, 5, 15),                        # as many equal ones but two
    ("bf16", 5, 320, 112, 11, 5, 14), ("u8", 5, 384, 32, 13, 5, 9),   # many fewer
    ("bf16", 9, 192, 96, 24, 3, 3), ("bf16", 11, 128, 64, 15, 3, 2), ("bf16", 4, 128, 208, 15, 3, 2), ("u8", 4, 256, 48, 41, 3, 2),   # 27 steps, 18 under few results
    ("bf16", 5, 128, 48, 40, 3, 1), ("bf16", 16, 128, 32, 27, 3, 1), ("u8", 6, 256, 64, 33, 3, 1),                                   # 18 under many
    ("u8", 10, 224, 16, 33, 3, 1), ("u8", 14, 240, 16, 30, 3, 1), ("u8", 8, 224, 32, 11, 3, 2)])        # int8: two short slices of many tiles, of few
def test_slices_of_conv_windows(dts, b, c, f, hw, fs, slices):
    types = {"bf16": (M.bf16, M.bf16, M.f32), "u8": (M.u8, M.i8, M.i32)}[dts]
    p = M.Conv([b, f, c, hw, hw, fs, fs], types).plan()
    assert p.kernels == ["k_gemm", "k_sum_splits"][:1 + (slices > 1)] and p.steps[0].grid[1] == slices, p


@pytest.mark.parametrize("types,m,k,n,nk,in_place", [
    ("bf16", 678, 5488, 755, True, False), ("u8", 201, 10320, 2955, True, False), ("bf16", 474, 3768, 1108, True, True), ("bf16", 231, 3872, 3091, True, True),    # nothing to copy: 86, 81, 59 steps; 196 tiles
    ("bf16", 653, 5434, 782, True, False), ("bf16", 460, 4031, 1299, False, False), ("bf16", 1150, 4530, 497, True, True),                                         # equal slices, none
    ("bf16", 755, 4992, 741, False, False), ("bf16", 1415, 4448, 443, False, True),                                                                             # one copy: 78 and 70 steps
    ("u8", 905, 9285, 519, False, False), ("u8", 204, 9048, 2539, True, True),                                                                                   # int8 rows of N, of K
    ("bf16", 1031, 2937, 1194, True, False), ("bf16", 836, 2455, 1981, True, True), ("bf16", 1031, 2938, 1194, True, True), ("bf16", 1031, 2937, 1194, False, True),   # odd rows along K, words, along N
])
def test_long_k_of_more_than_half_a_round_of_tiles(types, m, k, n, nk, in_place):
    dts = {"bf16": (M.bf16, M.bf16, M.f32), "u8": (M.u8, M.i8, M.i32)}[types]
    p = M.Matmul([1, m, k, n], dts, layouts=[None, KT if nk else None, None]).plan()
    assert (p.kernels == ["k_gemm_ring"] and "RA = " in p.steps[0].kernel) == in_place, p


@pytest.mark.parametrize("types,m,k,n,start", [("bf16", 45, 398, 408, 1), ("bf16", 45, 514, 325, 4), ("u8", 40, 1020, 2804, 1), ("u8", 40, 1028, 2804, 4),
                                               ("bf16", 32, 398, 408, 4), ("bf16", 45, 399, 408, 1), ("bf16", 45, 400, 408, 16), ("f32", 45, 199, 408, 4)])
def test_few_rows_on_words(types, m, k, n, start):
    """One load a chunk, or for more than 32 rows over up to a unit of K a wave cut out of two."""
    dts = {"bf16": (M.bf16, M.bf16, M.f32), "u8": (M.u8, M.i8, M.i32), "f32": (M.f32,) * 3}[types]
    p = M.Matmul([1, m, k, n], dts, layouts=[None, KT, None]).plan()
    assert p.kernels == ["k_gemm_skinny"] and f"START = {start}," in p.steps[0].kernel, p


@pytest.mark.parametrize("b,m,keys,d,by_waves", [(8, 1651, 448, 64, False), (12, 1129, 534, 64, False), (25, 554, 640, 64, False), (29, 309, 832, 64, False), (8, 1046, 1030, 64, False),
                                                 (9, 955, 1090, 64, True), (14, 960, 1024, 64, False), (12, 960, 1280, 64, False), (14, 704, 1344, 64, True),   # ragged, and whole blocks of 64
                                                 (43, 290, 443, 64, True), (36, 398, 420, 64, True),                                                          # where the other form has 128 queries
                                                 (45, 326, 325, 64, False), (5, 1770, 512, 32, True), (9, 1598, 323, 32, False), (9, 620, 300, 128, True)])
def test_32_queries_a_workgroup(b, m, keys, d, by_waves):
    """Two of them to a compute unit only where the keys are many enough."""
    p = M.ComposeMSM(b, m, d, keys, d, layouts=[None, None, KT, None]).plan()
    assert p.kernels == ["k_attn"] and ("QB = 2, W = 8" in p.steps[0].kernel) == by_waves, p


@pytest.mark.parametrize("b,m,keys,d,shares", [(34, 1, 3264, 128, 4), (18, 2, 5760, 128, 8), (20, 1, 4032, 128, 8), (51, 4, 2759, 64, 3), (124, 1, 1152, 64, 1),   # 25 to 64 MB of K and V
                                               (47, 1, 896, 64, 1), (16, 1, 2800, 128, 6), (16, 1, 32768, 128, 16), (71, 2, 1885, 128, 3),                         # below, above
                                               (6, 1, 8679, 128, 17)])                                                                                             # not 34: a third trip of the merge
def test_shares_of_the_keys_in_decoding(b, m, keys, d, shares):
    """Workgroups enough to stream K and V from memory, not from a cache that a model's other layers have been through."""
    p = M.ComposeMSM(b, m, d, keys, d, layouts=[None, None, KT, None]).plan()
    assert p.kernels == ["k_attn", "k_attn_merge"][:1 + (shares > 1)] and p.steps[0].grid == (b, shares, 1), p


@pytest.mark.parametrize("types,m,k,n,in_place", [
    ("bf16", 47, 8192, 5696, False), ("bf16", 33, 3456, 14243, False), ("u8", 45, 3840, 8607, False), ("bf16", 43, 4224, 14336, False),   # three equal slices of K or more
    ("bf16", 50, 5184, 1329, True), ("bf16", 63, 4224, 3216, True), ("bf16", 56, 2816, 14053, True),                                      # ... of 14 and 27 MB of B; two
    ("u8", 40, 10496, 8431, False), ("bf16", 45, 3904, 8991, False), ("bf16", 63, 3904, 12191, True), ("bf16", 46, 3904, 15168, True),    # one left over: 132, 141, 191, 237 tiles
    ("bf16", 35, 8768, 5888, False), ("bf16", 55, 7736, 4661, True), ("bf16", 48, 9520, 5312, True), ("bf16", 52, 3712, 8704, False),     # many steps; whole ones
    ("bf16", 57, 4478, 12288, True)])                                                                                                     # rows of no whole chunks
def test_33_to_64_rows_over_a_long_k(types, m, k, n, in_place):
    dts = {"bf16": (M.bf16, M.bf16, M.f32), "u8": (M.u8, M.i8, M.i32)}[types]
    p = M.Matmul([1, m, k, n], dts, layouts=[None, KT, None]).plan()
    assert p.kernels[0] == ("k_gemm_ring" if in_place else "k_gemm"), p


@pytest.mark.parametrize("types,k,n,rows", [("bf16", 9152, 3008, 1), ("bf16", 5056, 5122, 1), ("bf16", 4592, 5804, 2), ("bf16", 3712, 9142, 2), ("bf16", 4096, 6144, 1), ("bf16", 4096, 6656, 2),
                                            ("bf16", 6528, 7726, 2), ("u8", 11424, 4800, 1), ("u8", 8192, 8192, 1), ("u8", 4096, 11008, 1), ("u8", 3360, 13907, 2), ("u8", 10144, 7518, 2)])
def test_rows_of_b_a_wavefront_for_two_rows_of_a(types, k, n, rows):
    dts = {"bf16": (M.bf16, M.bf16, M.f32), "u8": (M.u8, M.i8, M.i32)}[types]
    p = M.Matmul([1, 2, k, n], dts, layouts=[None, KT, None]).plan()
    assert p.kernels == ["k_gemv"] and f"ROWS = 2, COLS = {rows}]" in p.steps[0].kernel, p


@pytest.mark.parametrize("b,m,k,n,out,accum,in_place", [
    (1, 43, 1273, 4452, M.f32, False, False), (1, 43, 1084, 5269, M.f32, False, True), (1, 35, 971, 8647, M.f32, False, True), (1, 39, 1603, 3436, M.f32, False, True),   # few rows: odd, words, 136 tiles, slices
    (2, 581, 2761, 1178, M.bf16, False, False), (2, 887, 1961, 904, M.f32, False, False), (2, 1343, 1481, 639, M.f32, False, True), (2, 581, 2762, 1178, M.f32, False, True),   # 44, 31, 24 steps; words
    (2, 789, 1007, 1167, M.f32, False, False), (1, 2399, 1307, 925, M.bf16, False, False), (2, 598, 1019, 3125, M.f32, False, True), (2, 1101, 829, 1540, M.bf16, False, True),   # 128 x 128: 16, 21 steps, 250 tiles, 13 steps
    (1, 1749, 173, 1407, M.bf16, True, False), (1, 1749, 173, 1407, M.bf16, False, True), (1, 1749, 174, 1408, M.bf16, True, True)])                                          # onto bf16
def test_odd_rows_of_bf16_along_k(b, m, k, n, out, accum, in_place):
    p = M.Matmul([b, m, k, n], (M.bf16, M.bf16, out), accum=accum, layouts=[None, KT, None]).plan()
    assert (p.kernels[0] == "k_gemm_ring" and "RA = " in p.steps[0].kernel) == in_place, p
