"""The rules of csrc/tile_rules.h, built with the host's compiler: which tiles the products run on."""
import ctypes as C
import shutil
import subprocess
from pathlib import Path

import pytest

from tests.test_gpu_expert_gemm import TILES_OF_NARROW
from tests.test_gpu_grouped_tiles import FEW_STEPS, PAST_THE_CACHE, ROWS_FOR_TILE

CSRC = Path(__file__).resolve().parent.parent / "amd_distributed_2025_amd" / "csrc"


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ not installed")
    src = tmp_path_factory.mktemp("rules") / "rules.cpp"
    src.write_text('#include "tile_rules.h"\n'
                   'extern "C" int bands(long long rows_hint, int groups, int n, int k) { return grouped_tile_bands(rows_hint, groups, n, k); }\n'
                   'extern "C" int past(int groups, int n, int k) { return weights_past_the_cache(groups, n, k); }\n')
    lib = src.with_suffix(".so")
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Wno-unused-function", "-shared", "-fPIC", f"-I{CSRC}",
                    str(src), "-o", str(lib)], check=True)
    dll = C.CDLL(str(lib))
    dll.bands.argtypes = [C.c_longlong, C.c_int, C.c_int, C.c_int]
    return dll


OUT_OF_RANGE = 1 << 30


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


@pytest.mark.parametrize("K", [2048, 2112])
def test_the_tiles_that_the_gpu_tests_mean(rules, K):
    for groups, tiles in ROWS_FOR_TILE.items():
        for rows, tile in tiles.items():
            if isinstance(tile, int):
                assert 32 * rules.bands(rows * groups, groups, 7168, K) == tile, (groups, rows)
    assert {t for tiles in ROWS_FOR_TILE.values() for t in tiles.values() if isinstance(t, int)} == {64, 128, 192, 256, 320}
    for (in_dim, out_dim), tiles in TILES_OF_NARROW.items():
        assert {rows: 32 * rules.bands(rows * 5, 5, out_dim, in_dim) for rows in tiles} == tiles


@pytest.mark.parametrize("K", FEW_STEPS)
def test_the_tile_that_the_ring_of_half_steps_is_tested_on(rules, K):
    assert rules.bands(800 * 3, 3, 7168, K) == 10


def test_weights_past_the_cache(rules):
    """From 256 MB on (MB of 2^20 bytes), also where the product of the sizes does not fit 64 bits."""
    assert rules.past(64, 1024, 2048) and not rules.past(64, 1024, 2040) and rules.past(2 ** 31 - 1, 2 ** 31 - 1, 2 ** 31 - 1)
    for (groups, K), tiles in PAST_THE_CACHE.items():
        assert rules.past(groups, 7168, K)
        for rows, tile in tiles.items():
            assert not tile or (32 * rules.bands(rows * groups, groups, 7168, K) == tile and rows <= tile)


def test_the_second_tiles_that_the_gpu_tests_mean():
    """A launch has a workgroup for every tile of `rows_hint` rows and one more row of tiles per group: with the row
    counts of ROWS_FOR_TILE for five groups, [704, 704, 650, 704, 704] is more than that for every tall tile."""
    for rows, tile in ROWS_FOR_TILE[5].items():
        if isinstance(tile, int):
            workgroups = rows * 5 // tile + 5
            assert 5 * -(-650 // tile) > workgroups, (rows, tile)
