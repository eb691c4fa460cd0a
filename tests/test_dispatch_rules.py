"""Which kernel a call takes: the rules by size, asked directly on the host (C++ functions of libchadq.so).  No GPU."""
import ctypes
import random

import pytest

from chadslab_amd import _lib

TILES = ["32x64", "64x64", "96x64", "128x64", "96x128", "128x128", "192x128", "256x128", "256x256",
         "short 32x64", "short 64x64", "short 128x128", "short 256x256"]


def _rule(symbol, result=ctypes.c_int):
    fn = _lib.load()[symbol]
    fn.restype = result
    return fn


def _tile(m, n, k, int4, guard):
    fn = _rule("_ZN5chadq14gemm_tile_pickEiiibb")
    fn.argtypes = [ctypes.c_int] * 3 + [ctypes.c_bool] * 2
    return TILES[fn(m, n, k, int4, guard)]


def test_gemm_tile_of_few_k_is_not_one_fitted_to_many():
    """Products of a few steps, each with its time on the tile given here and on the one that constants fitted to 512 k and more gave."""
    assert _tile(193, 12160, 128, False, False) == "short 128x128"  # 6.5 us, on 128 x 64 8.8
    assert _tile(2690, 256, 256, False, False) == "short 64x64"     # 4.3, on 96 x 64 5.1
    assert _tile(1865, 1728, 256, False, False) == "short 128x128"  # 8.1, on 192 x 128 9.8
    assert _tile(24, 1024, 1120, True, True) == "short 32x64"       # 5.2, with the other loop 5.8
    assert _tile(48, 1024, 512, True, False) == "short 64x64"       # 4.7, with the other loop 4.9
    # and many k still take the loop that is the faster one there
    assert _tile(48, 14336, 4096, True, False) == "64x64"
    assert _tile(512, 4096, 4096, True, False) == "128x64"
    assert _tile(1000, 4096, 14336, False, False) == "128x128"
    assert _tile(4096, 14336, 4096, True, False) == "256x256"


@pytest.mark.parametrize("int4", [True, False])
@pytest.mark.parametrize("guard", [True, False])
def test_gemm_tile_fits_the_rows_and_every_tile_is_somebodys(int4, guard):
    seen = set()
    for m in (1, 17, 32, 33, 64, 65, 70, 100, 129, 190, 250, 300, 385, 512, 700, 1000, 1500, 2049, 4096, 7000):
        for n in (1, 64, 257, 1024, 2048, 3000, 4096, 5000, 8192, 11008, 14336, 20000, 33000):
            for k in (32, 96, 256, 512, 800, 1024, 1504, 2048, 4096, 8192, 14336):
                tile = _tile(m, n, k, int4, guard)
                seen.add(tile)
                assert tile.endswith("32x64") == (m <= 32) and (m > 64 or tile.endswith(("32x64", "64x64")))
    assert seen == set(TILES) - (set() if int4 else {"short 256x256"})


def test_gemv_of_k_that_256_does_not_divide_takes_the_matrix_cores_where_they_are_faster():
    fn = _rule("_ZN5chadq20gemv_on_matrix_coresEiii", ctypes.c_bool)
    # us, streamed once per pair of rows (beyond 4096 k: per row) / on the matrix cores
    for m, n, k in ((3, 32, 14368), (4, 1024, 14368), (3, 2048, 8160), (4, 4096, 8160), (8, 512, 6176), (5, 32, 4064), (5, 1024, 4064),
                    (8, 512, 4064), (5, 128, 2080)):  # 9.9 / 38, 14.8 / 39.5, 9.7 / 23.8, 20.4 / 23.9, 13.2 / 19.2, 8.4 / 13, 9.0 / 13.4, 12.4 / 13.3, 8.1 / 8.9
        assert not fn(m, n, k), (m, n, k)
    for m, n, k in ((5, 32, 32), (16, 128, 96), (5, 2048, 2080), (8, 4096, 4064), (16, 1024, 4064), (4, 11008, 6176), (8, 8192, 8160), (16, 1024, 8160),
                    (3, 32000, 14368)):               # 7.2 / 3.7, 19 / 3.8, 11.1 / 9.0, 26 / 13.8, 24 / 13.5, 46 / 21, 71 / 24.6, 27.8 / 23.9, 207 / 81
        assert fn(m, n, k), (m, n, k)
    assert not any(fn(m, 4096, 4064) for m in range(1, 5)) and not any(fn(m, 32000, 14368) for m in (1, 2))


def test_few_token_experts_stage_activations_only_where_workgroups_have_items_enough():
    fn = _rule("_ZN5chadq19moe_few_through_ldsEiiiii", ctypes.c_bool)  # (tokens, experts, top k, items of an expert, blocks of 256 k of each)

    def gate_up(t, e, top_k, h, f):
        return fn(t, e, top_k, f // 16, h // 256)

    def down(t, e, top_k, h, f):
        parts = 4 if f >= 4096 else 2 if f >= 2048 else 1
        return fn(t, e, top_k, h // 32 * parts, -(-(f // 256) // parts))

    # whole calls, us, through LDS / straight to registers: 28 / 21, 40 / 32.5, 23 / 20 (one or two items per workgroup, or none)
    for size in ((2, 8, 1, 2304, 1536), (14, 4, 2, 1280, 4352), (3, 8, 1, 1280, 1280)):
        assert not gate_up(*size) and not down(*size)
    assert gate_up(4, 8, 2, 4096, 14336) and down(4, 8, 2, 4096, 14336)  # 135 / 150
    assert gate_up(6, 8, 2, 256, 12288)                                  # 40 / 43
    # never more LDS than leaves three workgroups on a compute unit: 18304 bytes are the kernel's own, dealt out in pieces of 1280
    for t in range(1, 17):
        for span in range(1, 65):
            x_bytes = 512 + t * (span * 512 + 16)
            assert fn(t, 16, 4, 100000, span) == (3 * -(-(18304 + x_bytes) // 1280) * 1280 <= 163840)


def test_expert_down_product_of_short_k_is_not_split_among_many_workgroups():
    fn = _rule("_ZN5chadq17moe_uneven_splitsEiiii")  # (pairs, H, F, experts)
    assert fn(4 * 375, 2304, 768, 8) == 1 and fn(4 * 422, 2560, 1536, 4) == 1  # 67.0 us (split 71.6), 85.4 (96.3)
    assert fn(2 * 256, 2304, 1280, 8) == 4                                     # 65.8 (69.6)
    assert fn(2 * 455, 2048, 8960, 8) == 3 and fn(4 * 455, 2304, 1280, 8) == 1


def test_splits_of_exact_products_count_the_workgroups_of_the_fullest_xcd():
    """us, in the parts that rounds of 256 (512) workgroups gave / in those given here."""
    fn = _rule("_ZN5chadq17gemm_exact_splitsEiii")
    fn.argtypes = [ctypes.c_int] * 3
    assert fn(552, 1280, 5120) != 5   # 35 tiles: 25 workgroups in 5 parts on each XCD that has 5 tiles, 15 more than the others; 32.1 / 20.7 in 4
    assert fn(265, 1344, 7168) != 7   # 31.6 / 20.5 in 6
    assert fn(266, 3520, 3072) != 3   # 31.6 / 22.0 in 2
    assert fn(22, 4480, 1024) == 2    # 4: 6.4 / 4.9
    assert fn(55, 128, 256) == 1 and fn(152, 384, 22016) == 8 and fn(4096, 2048, 2048) == 1


@pytest.mark.parametrize("d,hq,dh,ffn", [(2048, 8, 256, 16384), (256, 16, 128, 256), (1280, 4, 128, 6400), (512, 1, 256, 768)])
def test_prompt_workspace_covers_shorter_chunks(d, hq, dh, ffn):
    """A workspace for T tokens serves fewer as well, the last layer's single row among them, in however many parts they are summed."""
    lib = _lib.load()
    splits = _rule("_ZN5chadq17gemm_exact_splitsEiii")
    splits.argtypes = [ctypes.c_int] * 3
    size = [lib.chadq_prompt_i4g32_workspace_bytes(t, d, hq, dh, ffn) for t in range(1, 400)]
    assert size == sorted(size)
    most = 0
    for t in range(1, 400):
        parts = [splits(t, n, k) * t * n for n, k in (((hq + 2) * dh, d), (d, hq * dh), (d, ffn))] + [splits(1, n, k) * n for n, k in ((d, hq * dh), (d, ffn))]
        most = max(most, *parts)
        rest = t * (4 * d + 4 * hq * dh + 2 * max(d, hq * dh) + 2 * ffn)
        assert size[t - 1] >= 4 * most + rest


def test_exact_products_take_the_tile_that_reaches_the_compute_units():
    """us in tiles of 64 / 128 (/ 256) rows."""
    fn = _rule("_ZN5chadq15gemm_exact_tileEiiiibPfPi")
    fn.argtypes = [ctypes.c_int] * 4 + [ctypes.c_bool, ctypes.POINTER(ctypes.c_float), ctypes.POINTER(ctypes.c_int)]

    def tile(m, n, per, parts, gated):
        columns = ctypes.c_int()
        return fn(m, n, per, parts, gated, ctypes.byref(ctypes.c_float()), ctypes.byref(columns)), columns.value

    def rows(*size):
        return tile(*size)[0]

    assert rows(101, 128, 1, 8, False) == 64      # 4.7 / 7.6
    assert rows(158, 5120, 9, 1, False) == 64     # 12.1 / 27.9
    assert rows(432, 5120, 6, 1, False) == 128    # 24.4 / 21.8
    assert rows(101, 8192, 8, 1, True) == 64      # 11.7 / 25.9 / 32.7
    assert rows(256, 32768, 8, 1, True) == 256
    assert rows(64, 32768, 8, 1, True) == 64 and rows(32, 32768, 8, 1, True) == 32 and rows(9, 64, 1, 1, False) == 32
    assert tile(256, 2048, 16, 4, False) == (128, 64) and tile(385, 5120, 3, 3, False) == (128, 128) and tile(300, 32768, 1, 1, True) == (128, 128)


def test_prompt_projections_are_rotated_where_they_are_written_unless_parts_pay():
    fn = _rule("_ZN5chadq19gemm_exact_qkv_paysEiii", ctypes.c_bool)  # (tokens, (hq + 2) * dh, d)
    assert fn(256, 2560, 2048) and fn(212, 2560, 1792) and fn(4, 1280, 512)          # us a prompt 2085 / 2134, 313 / 325, 203 / 208
    assert not fn(24, 2560, 2048) and not fn(35, 640, 1024) and not fn(7, 1536, 1536)  # 1088 / 1058, 283 / 277


def test_gemm_is_summed_in_parts_where_few_tiles_walk_a_long_k():
    lib = _lib.load()

    def parts(m, n, k, int8=0):
        return lib.chadq_gemm_bf16_workspace_bytes(m, n, k, int8) // (4 * m * n) or 1

    # us in one part / in parts with the launch that adds them
    for m, n, k, int8 in ((81, 1280, 14080, 0), (40, 1340, 10752, 0), (62, 1536, 11264, 0), (250, 640, 9760, 1), (152, 1280, 14336, 1), (48, 4096, 14336, 0), (26, 5542, 11776, 0)):
        assert parts(m, n, k, int8) > 1, (m, n, k)  # 29.1 / 14.2, 22.6 / 11.4, 23.2 / 12.5, 25.3 / 13.3, 30.0 / 18.0, 35 / 15.7, 21.6 / 15.2
    for m, n, k in ((48, 14336, 4096), (512, 4096, 4096), (1000, 4096, 14336), (4096, 14336, 4096), (48, 1024, 512), (16, 512, 16384), (33, 64, 1056), (48, 2048, 1 << 22)):
        assert parts(m, n, k) == 1 and parts(m, n, k, 1) == 1, (m, n, k)
    # calls of qlinear in a row: 7.0 / 9.1, 7.9 / 9.0, 6.8 / 9.1, 8.8 / 9.5, 8.6 / 9.4; 7.2 / 8.7, 8.8 / 9.2
    for m, n, k in ((17, 512, 3584), (31, 64, 4032), (17, 512, 4096), (116, 128, 1952), (65, 512, 3584), (128, 64, 3584)):
        assert parts(m, n, k, 1) == 1, (m, n, k)
    assert parts(38, 107, 1728) == 1 and parts(49, 960, 2816) == 1
    assert lib.chadq_gemm_bf16_workspace_bytes(0, 512, 4096, 0) == 0 and lib.chadq_gemm_bf16_workspace_bytes(17, -1, 4096, 1) == 0


def test_parts_of_a_gemm_cover_k_and_none_is_empty():
    fn = _rule("_ZN5chadq16gemm_split_partsEiiibPNS_8GemmTileEPi")
    fn.argtypes = [ctypes.c_int] * 3 + [ctypes.c_bool] + [ctypes.POINTER(ctypes.c_int)] * 2
    r, tile, span = random.Random(11), ctypes.c_int(), ctypes.c_int()
    split = ends_early = 0
    for i in range(60000):
        int4, m, n = i % 2 == 0, int(17 * 30 ** r.random()), int(16 * 500 ** r.random())
        step = 32 if int4 else 16
        k = int(1024 / step * 16 ** r.random()) * step
        parts = fn(m, n, k, int4, ctypes.byref(tile), ctypes.byref(span))
        assert 1 <= parts <= 8 and (parts == 1 or TILES[tile.value] in ("32x64", "64x64", "128x64")), (m, n, k)
        assert parts * span.value >= k > (parts - 1) * span.value and (parts == 1 or span.value % 256 == 0), (m, n, k, int4, parts, span.value)
        split += parts > 1
        ends_early += parts > 1 and -(-(k // 256) // parts) * 256 * parts < k  # were it counted in whole blocks
    assert split > 5000 and ends_early > 500, (split, ends_early)


def test_gemv_is_summed_in_parts_where_few_rows_walk_a_long_k():
    lib = _lib.load()

    def parts(m, n, k, int8):
        return lib.chadq_gemv_workspace_bytes(m, n, k, int8) // ((8 if int8 else 4) * m * n) or 1

    for int8 in (0, 1):
        for m in (1, 4, 8, 16):
            assert parts(m, 512, 16384, int8) > 1 and parts(m, 2048, 2048, int8) == 1 and parts(m, 16384, 16384, int8) == 1 and parts(m, 512, 4064, int8) == 1
            for n in (1, 16, 100, 512, 1000, 2048):
                for k in (128, 256, 4096, 6400, 8192, 16384, 65536):
                    assert 1 <= parts(m, n, k, int8) <= 8
    # int8, us in one part / in parts: 6.6 / 7.8, 48.0 / 29.1, 20.3 / 22.2
    assert parts(1, 512, 6144, 1) == 1 and parts(16, 4096, 16384, 1) == 4 and parts(12, 6144, 6144, 1) == 1
    assert parts(1, 14336, 4096, 0) == 1 and parts(1, 16384, 2048, 1) == 1 and parts(6, 11008, 4096, 0) == 1
    assert lib.chadq_gemv_workspace_bytes(17, 512, 16384, 0) == 0 and lib.chadq_gemv_workspace_bytes(1, 512, 16400, 1) == 0


def test_host_module_answers_as_the_library_does():
    """Bytes asked through the host module, which the calls of ops.py use, and through the C ABI."""
    lib, native, r = _lib.load(), _lib.native(), random.Random(4)
    for _ in range(3000):
        size = (r.randint(-1, 300), r.randint(-2, 9000), r.randint(-2, 600) * 32, r.randint(0, 1))
        assert native.gemv_bytes(*size) == lib.chadq_gemv_workspace_bytes(*size)
        assert native.gemm_bytes(*size) == lib.chadq_gemm_bf16_workspace_bytes(*size)
    assert native.gemv_bytes(1, 512, 16384, 0) > 0 and native.gemm_bytes(48, 4096, 14336, 1) > 0
    assert native.gemm_bytes(1 << 40, 512, 16384, 0) == 0  # (the product refuses it)
    with pytest.raises(TypeError):
        native.gemv_bytes(1, 512, 16384)
