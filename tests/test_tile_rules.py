"""The rules of csrc/tile_rules.h, built with the host's compiler: which tiles the products run on."""
import ctypes as C
import shutil
import subprocess
from pathlib import Path

import pytest

from tests.test_gpu_expert_gemm import KERNELS_OF_NARROW
from tests.test_gpu_grouped_tiles import FEW_STEPS, KERNELS, PAST_THE_CACHE
from tests.test_gpu_linear import WAYS, WITH_A_NEXT_TILE
from tests.test_gpu_ring_tiles import RING_STEPS, RING_TILES

CSRC = Path(__file__).resolve().parent.parent / "amd_distributed_2025_amd" / "csrc"


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ not installed")
    src = tmp_path_factory.mktemp("rules") / "rules.cpp"
    src.write_text('#include "tile_rules.h"\n'
                   'extern "C" int bands(long long rows_hint, int groups, int n, int k) { return grouped_tile_bands(rows_hint, groups, n, k); }\n'
                   'extern "C" int past(int groups, long long rows_hint, int n, int k) { return weights_past_the_cache(groups, rows_hint, n, k); }\n'
                   'extern "C" int ring(long long rows_hint, int groups, int n, int k) { return grouped_ring(rows_hint, groups, n, k); }\n'
                   'extern "C" int far_ahead(long long rows_hint, int groups, int n) { return streams_far_ahead(rows_hint, groups, n); }\n'
                   'extern "C" int linear_ring_of(long long m, long long n, long long k) { return linear_ring(m, n, k); }\n'
                   'extern "C" int way(long long m, long long n, long long k) { return linear_way(m, n, k); }\n')
    lib = src.with_suffix(".so")
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Wno-unused-function", "-shared", "-fPIC", f"-I{CSRC}",
                    str(src), "-o", str(lib)], check=True)
    dll = C.CDLL(str(lib))
    dll.bands.argtypes = [C.c_longlong, C.c_int, C.c_int, C.c_int]
    dll.past.argtypes = [C.c_int, C.c_longlong, C.c_int, C.c_int]
    dll.ring.argtypes = [C.c_longlong, C.c_int, C.c_int, C.c_int]
    dll.far_ahead.argtypes = [C.c_longlong, C.c_int, C.c_int]
    dll.linear_ring_of.argtypes = [C.c_longlong] * 3
    dll.way.argtypes = [C.c_longlong] * 3
    return dll


OUT_OF_RANGE = 1 << 30


def kernel_of(rules, rows, groups, n, k):
    """The kernel of a grouped product, `rows` per group, as launch_grouped_dense and launch_grouped_gemm ask for it."""
    ring = rules.ring(rows * groups, groups, n, k)
    if ring:
        return "ring " + ["32 x 32", "32 x 64", "64 x 64", "64 x 128"][ring - 1]
    if rows >= 56:
        return f"tiles {32 * rules.bands(rows * groups, groups, n, k)}"
    if rules.far_ahead(rows * groups, groups, n):
        return "stream 32, four steps ahead"
    return "stream 32, two steps ahead" if rows <= 8 else "stream 64" if rows <= 48 else "stream 128"


@pytest.mark.parametrize("K", [1677712, 1677720, 1677728, 2097144])
def test_rows_of_a_tile_end_before_the_out_of_range_offset(rules, K):
    """Vectors past the end of a row are read at an offset of 2^30, which has to lie past the tile's rows: at
    320 rows that is so up to K = 1677720, at 256 up to 2097144."""
    picked = {rules.bands(rows * groups, groups, n, K) for rows in (60, 150, 200, 300, 320, 600, 1000) for groups in (1, 5, 32)
              for n in (32, 2048, 7168)}
    assert 0 not in picked
    assert all(bands * 32 * K * 2 < OUT_OF_RANGE for bands in picked), picked
    assert (10 in picked) == (320 * K * 2 < OUT_OF_RANGE)


def test_no_tile_beyond_the_range_of_its_offsets(rules):
    assert rules.bands(1500, 5, 7168, 2097152) == 0  # (the streaming kernel takes it)


@pytest.mark.parametrize("rows_hint,groups,n,k,bands", [
    (2013, 32, 7168, 7168, 4),               # 7 workgroups of 128 columns on every unit, where 256 leave half a round idle
    (8 * 64, 8, 4096, 4096, 4), (8 * 80, 8, 4096, 2048, 4),  # 256 workgroups for 256 units, where 256 columns make 128
    (32 * 100, 32, 2048, 4096, 6), (64 * 64, 64, 7168, 7168, 6),  # whole rounds of 256 columns
    (32 * 256, 32, 2048, 4096, 10), (32 * 256, 32, 4096, 2048, 10),
    (8 * 200, 8, 7168, 2048, 8), (8 * 64, 8, 2048, 7168, 2),
])
def test_tile_that_was_fastest_where_they_differ_most(rules, rows_hint, groups, n, k, bands):
    """Timed on the GPU: the tile picked here is the fastest of five or within 3 % of it."""
    assert rules.bands(rows_hint, groups, n, k) == bands


def test_every_count_of_rows_has_a_tile(rules):
    for rows_hint in (1, 56, 57, 10 ** 6, 2 ** 31 - 1):
        for groups in (1, 2, 1000, 65536):
            assert rules.bands(rows_hint, groups, 32, 8) in (2, 4, 6, 8, 10)


@pytest.mark.parametrize("K", [8, 200, 2048, 2112])
def test_the_kernels_that_the_gpu_tests_mean(rules, K):
    """(with few steps of K other tiles and no rings are picked, but a streaming kernel stays one)"""
    for groups, kernels in KERNELS.items():
        picked = {rows: kernel_of(rules, rows, groups, 7168, K) for rows in kernels}
        assert picked == kernels if K > 2000 else all(picked[r].split()[0] == k.split()[0] for r, k in kernels.items() if "ring" not in k)
    tested = {k for kernels in KERNELS.values() for k in kernels.values()}
    assert tested >= {f"tiles {t}" for t in (64, 128, 192, 256, 320)} | {f"stream {s}" for s in ("64", "128")}
    assert {f"stream 32, {n} steps ahead" for n in ("two", "four")} <= tested


def test_the_kernels_of_narrow_products_that_the_gpu_tests_mean(rules):
    for (groups, in_dim, out_dim), kernels in KERNELS_OF_NARROW.items():
        assert {rows: kernel_of(rules, rows, groups, out_dim, in_dim) for rows in kernels} == kernels


@pytest.mark.parametrize("K", FEW_STEPS)
def test_the_tile_that_the_ring_of_half_steps_is_tested_on(rules, K):
    assert rules.bands(800 * 3, 3, 7168, K) == 10


def test_weights_past_the_cache(rules):
    """From 256 MB on (MB of 2^20 bytes), also where the product of the sizes does not fit 64 bits, and from 192 MB in as
    many groups as there are rows."""
    big = 2 ** 31 - 1
    assert rules.past(64, 64, 1024, 2048) and not rules.past(64, 64, 1024, 2040) and rules.past(big, big, big, big)
    assert rules.past(64, 48, 1024, 2048) and not rules.past(64, 47, 1024, 2048) and not rules.past(256, 0, 7168, 7168)
    for (groups, N, K), kernels in PAST_THE_CACHE.items():
        for rows, kernel in kernels.items():
            assert rules.past(groups, rows * groups, N, K)
            assert kernel_of(rules, rows, groups, N, K) == kernel
            assert kernel.startswith("stream") or rows <= int(kernel.split()[1])  # (one row of tiles: else plain loads)


def test_the_second_tiles_that_the_gpu_tests_mean():
    """A launch has a workgroup for every tile of `rows_hint` rows and one more row of tiles per group: with the row
    counts of KERNELS for five groups, [704, 704, 650, 704, 704] is more than that for every tall tile."""
    for rows, kernel in KERNELS[5].items():
        if kernel.startswith("tiles"):
            tile = int(kernel.split()[1])
            workgroups = rows * 5 // tile + 5
            assert 5 * -(-650 // tile) > workgroups, (rows, tile)


SPLIT_32, SPLIT_64, TILES_64x128, TILES_128x128, PHASED_128, PHASED_192, PHASED_256, STREAM_WEIGHTS = range(8)  # LinearWay


def test_the_ways_that_the_gpu_tests_mean(rules):
    for name, shapes in WAYS.items():
        for m, n in shapes:
            for k in (512, 2048, 8192):
                assert rules.way(m, n, k) == globals()[name], (m, n, k)


@pytest.mark.parametrize("m,n", WITH_A_NEXT_TILE)
def test_the_tiles_with_a_next_one_that_the_gpu_tests_mean(rules, m, n):
    """phased_gemm_kernel: workgroup b of 256 takes tiles b, b + 256, ..., whose numbers run through an XCD's share of them
    (xcd_contiguous) and then down four tile rows before the next tile column (GROUP_M)."""
    assert all(rules.way(m, n, k) == PHASED_256 for k in (8, 64, 200, 448))
    tiles_m, tiles_n = -(-m // 256), -(-n // 256)
    total = tiles_m * tiles_n
    kinds, places = set(), set()
    for tile in range(total):
        xcd, share, rest = tile % 8, total // 8, total % 8
        number = xcd * share + min(xcd, rest) + tile // 8
        group, inside = divmod(number, 4 * tiles_n)
        column, row = divmod(inside, min(4, tiles_m - 4 * group))
        row += 4 * group
        places.add((row, column))
        if tile + 256 < total:
            rows = min(256, m - 256 * row)
            kinds.add("columns" if 256 * (column + 1) > n else "whole" if rows == 256 else "half" if rows >= 128 else "less")
    assert len(places) == total and kinds == WITH_A_NEXT_TILE[m, n]


@pytest.mark.parametrize("m,n,k,way", [(112, 1920, 1832, SPLIT_32), (255, 1728, 3968, SPLIT_64), (64, 7168, 2304, SPLIT_64),
                                       (59, 512, 4448, SPLIT_32), (867, 1216, 6104, TILES_64x128),
                                       (547, 2688, 5376, TILES_64x128), (825, 2624, 1792, TILES_128x128),
                                       (1586, 2688, 1536, PHASED_192), (2048, 2880, 360, PHASED_192),
                                       (3532, 1408, 3824, PHASED_192), (1646, 5056, 2800, PHASED_256),
                                       (2048, 4096, 1024, PHASED_128), (4096, 4096, 512, PHASED_256)])
def test_way_that_was_fastest_where_they_differ_most(rules, m, n, k, way):
    assert rules.way(m, n, k) == way


def test_ways_of_a_product_stay_in_the_range_of_their_kernels(rules):
    """K is split from two steps for each of four waves on, and a way whose 32-bit offsets reach over `rows` rows is
    picked only where rows of K elements end before the out-of-range offset. Large and extreme sizes have a way too."""
    rows_of = {SPLIT_32: 128, SPLIT_64: 128, TILES_64x128: 256, TILES_128x128: 256, PHASED_128: 256, PHASED_192: 256, PHASED_256: 256}
    for m in (1, 32, 33, 64, 65, 200, 1000, 5000, 2 ** 31 - 1):
        for n in (32, 1024, 7168, 24448, 24480, 40000, 2 ** 31 - 32):
            for k in (8, 448, 456, 7168, 2097144, 2097152, 4194296, 4194304, 2 ** 31 - 8):
                way = rules.way(m, n, k)
                assert way == STREAM_WEIGHTS or rows_of[way] * k * 2 < OUT_OF_RANGE, (m, n, k, way)
                if way in (SPLIT_32, SPLIT_64):
                    assert (k + 63) // 64 >= 8
                    assert (n // 32) * ((m + 31) // 32) < 2 ** 31  # workgroups
                if way == STREAM_WEIGHTS:
                    assert k >= 2097152


@pytest.mark.parametrize("tile", RING_TILES)
def test_rings_that_the_gpu_tests_mean(rules, tile):
    groups, n, rows = RING_TILES[tile]
    for k in [*RING_STEPS[tile], 1544, 2112]:
        assert rules.ring(rows * groups, groups, n, k) == tile, k
    assert rules.ring(30000 * groups, groups, n, 2048) == 0


@pytest.mark.parametrize("rows_hint,groups,n,k,tile", [
    (7, 48, 832, 3840, 1), (2, 8, 4096, 2048, 1), (4, 4, 2048, 7168, 1), (425, 36, 5728, 2432, 2), (357, 43, 2240, 2752, 2),
    (368, 8, 1024, 3648, 2), (1704, 48, 512, 2432, 3), (858, 6, 960, 2400, 3), (1379, 7, 832, 6528, 4), (468, 9, 2304, 5568, 4),
    (144, 64, 1024, 2048, 0), (144, 64, 2048, 1024, 0), (118, 53, 2240, 512, 0), (2792, 41, 512, 640, 0), (2468, 48, 1856, 1184, 0),
    (320, 8, 7168, 7168, 0), (224, 8, 7168, 1536, 0), (32, 8, 7168, 2048, 0), (1280, 32, 2048, 1536, 0), (128, 32, 2048, 2880, 0),
    (14, 55, 2048, 2816, 2), (36, 78, 960, 2496, 2), (12, 61, 2528, 2400, 2), (20, 31, 2368, 2560, 0), (35, 24, 5376, 7136, 2), (154, 70, 928, 2336, 0),
    (8192, 32, 2048, 4096, 0), (0, 3, 7168, 200, 1), (7, 48, 832, 1 << 23, 0),
    (4, 44, 1728, 8, 0), (275, 11, 512, 216, 1), (285, 5, 2816, 8, 0), (480, 10, 896, 360, 0),
])
def test_ring_that_was_fastest(rules, rows_hint, groups, n, k, tile):
    """(a tenth slower on tiles of 32 x 64, uniform or skewed: 8 groups of 40 rows, 7168 x 7168, of 28, 7168 x 1536, of 4,
    7168 x 2048; 32 of 40, 2048 x 1536; 5 %: 64 of 2.25, 1024 x 2048)"""
    assert rules.ring(rows_hint, groups, n, k) == tile


@pytest.mark.parametrize("groups", [8, 32, 64, 128])
@pytest.mark.parametrize("n,k", [(4096, 2048), (7168, 2880), (2048, 7168), (4096, 1024)])
def test_many_rows_are_not_cut_into_tiles_of_32(rules, groups, n, k):
    """Above 24 rows per group a group often has more than 32 of them, and a second row of tiles reads its weights again."""
    for rows in (25, 32, 40, 44, 50, 55):
        assert rules.ring(rows * groups, groups, n, k) in (0, 3, 4), rows
    assert all(rules.ring(rows * groups, groups, n, k) == 0 for rows in (45, 50, 55)) or groups * n < 65536


@pytest.mark.parametrize("m,n,k,tile", [
    (137, 4320, 5440, 3), (200, 4096, 4096, 3), (82, 6592, 2816, 3), (494, 2048, 2176, 3), (195, 3008, 832, 3),
    (255, 1728, 3968, 0), (349, 4032, 2752, 0), (160, 4544, 512, 0), (64, 7168, 2304, 0), (8192, 8192, 3696, 0), (2048, 2880, 360, 0),
    (15, 5888, 448, 1), (80, 2176, 448, 1), (33, 4608, 352, 0), (1, 32, 264, 1), (1, 32, 256, 0), (2, 1344, 64, 0), (100, 4096, 1 << 22, 0),
])
def test_plain_products_on_rings(rules, m, n, k, tile):
    assert rules.linear_ring_of(m, n, k) == tile
    from tests.test_gpu_ring_tiles import RING_LINEAR
    for rows, columns, inputs in RING_LINEAR:
        assert rules.linear_ring_of(rows, columns, inputs), (rows, columns, inputs)
