"""The rules of csrc/tile_rules.h, built with the host's compiler: which tiles the products run on."""
import ctypes as C
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "amd_distributed_2025_amd" / "csrc"


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    src = tmp_path_factory.mktemp("rules") / "rules.cpp"
    src.write_text('#include "tile_rules.h"\n'
                   'extern "C" int bands(long long rows, int groups, int n, int k) { return grouped_tile_bands(rows, groups, n, k); }\n')
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
    picked = {rules.bands(rows, groups, n, K) for rows in (60, 150, 200, 300, 320, 600, 1000) for groups in (1, 5, 32)
              for n in (32, 2048, 7168)}
    assert 0 not in picked
    assert all(bands * 32 * K * 2 < OUT_OF_RANGE for bands in picked), picked
    assert (10 in picked) == (320 * K * 2 < OUT_OF_RANGE)


def test_no_tile_beyond_the_range_of_its_offsets(rules):
    assert rules.bands(300, 5, 7168, 2097152) == 0  # (the streaming kernel takes it)
