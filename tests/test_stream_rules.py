"""The rules of csrc/stream_rules.h, built with the host's compiler: which kernels the stages of a job run on."""
import ctypes as C
import shutil
import subprocess
from pathlib import Path

import pytest

from tests.test_gpu_block_streams import CASES
from tests.test_gpu_short_streams import LANES, RECV_CASES

CSRC = Path(__file__).resolve().parent.parent / "amd_distributed_2025_amd" / "csrc"
SEND_WAYS = ["by entry", "few", "block", "fanout", "wide fanout"]  # SendWay


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ not installed")
    src = tmp_path_factory.mktemp("rules") / "rules.cpp"
    src.write_text('#include "stream_rules.h"\n'
                   'extern "C" int way(long long tokens, int k, int ranks, int row_vecs, int vec16) {\n'
                   '  return send_way(tokens, k, ranks, row_vecs, vec16); }\n'
                   'extern "C" int piece(long long tokens, int k, int nvw, int vec16) { return block_piece(tokens, k, nvw, vec16); }\n'
                   'extern "C" int few(long long rows, int row_vecs, int nvw, int vec16, int compact) {\n'
                   '  return recv_few(rows, row_vecs, nvw, vec16, compact); }\n'
                   'extern "C" int through(long long rows, long long row_bytes) { return recv_through(rows, row_bytes); }\n'
                   'extern "C" int lanes(long long tokens, long long entries, int ranks, int row_vecs, int vec16) {\n'
                   '  return local_few_vecs(tokens, entries, ranks, row_vecs, vec16); }\n'
                   'extern "C" int keys(long long entries) { return few_keys(entries); }\n')
    lib = src.with_suffix(".so")
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Wno-unused-function", "-shared", "-fPIC", f"-I{CSRC}",
                    str(src), "-o", str(lib)], check=True)
    dll = C.CDLL(str(lib))
    dll.way.argtypes = [C.c_longlong] + [C.c_int] * 4
    dll.piece.argtypes = [C.c_longlong] + [C.c_int] * 3
    dll.few.argtypes = [C.c_longlong] + [C.c_int] * 4
    dll.through.argtypes = [C.c_longlong, C.c_longlong]
    dll.lanes.argtypes = [C.c_longlong, C.c_longlong] + [C.c_int] * 3
    dll.keys.argtypes = [C.c_longlong]
    return dll


def row(hidden):
    """Vectors of 16 bytes in a row, or its elements, and vectors per lane of a wave that moves it (row_geometry)."""
    vec16 = hidden % 8 == 0
    vecs = hidden // 8 if vec16 else hidden
    nvw = next((n for n in (1, 2, 4, 6, 8, 12, 14) if vecs <= 64 * n), 16) if vec16 else 16
    return vecs, vec16, nvw


def way_of(rules, tokens, k, ranks, hidden):
    vecs, vec16, nvw = row(hidden)
    way = SEND_WAYS[rules.way(tokens, k, ranks, vecs, vec16)]
    if way == "block":
        nvw = rules.piece(tokens, k, nvw, vec16)
        return way, nvw, -(-vecs // (64 * nvw))
    return way


@pytest.mark.parametrize("W,E,K,H,T", CASES)
def test_kernels_of_stage_1_that_the_gpu_tests_mean(rules, W, E, K, H, T):
    assert way_of(rules, T, K, W, H) == CASES[W, E, K, H, T]


@pytest.mark.parametrize("tokens,k,hidden,way", [
    (500, 1, 7167, "by entry"), (900, 1, 513, "by entry"), (500, 2, 1001, "by entry"), (300, 2, 4097, "by entry"),
    (200, 4, 4097, "by entry"), (120, 8, 7167, "by entry"), (435, 1, 1235, "by entry"), (858, 1, 4491, "by entry"),
    (728, 1, 2304, "by entry"), (918, 1, 6720, "by entry"), (100, 1, 7167, "few"), (60, 2, 7167, "few"), (100, 3, 1001, "few"),
    (30, 8, 7167, "few"), (80, 6, 1561, "few"), (1000, 1, 2048, "few"), (250, 2, 7168, "few"), (120, 8, 7168, "few"), (16, 2, 6144, "few"),
])
def test_way_of_short_streams_that_was_faster(rules, tokens, k, hidden, way):
    """Timed on the GPU: many pieces of rows that each rank all keys take up to 3.6 times as long as a wave per entry."""
    assert way_of(rules, tokens, k, 8, hidden) == way


@pytest.mark.parametrize("tokens,k,hidden,way", [
    (1967, 1, 2880, "by entry"), (2036, 1, 3328, "by entry"), (2303, 1, 2432, "by entry"), (2440, 1, 384, "by entry"), (2862, 1, 1856, "by entry"),
    (1823, 1, 704, "block"), (1917, 1, 1728, "block"), (1326, 1, 8000, "block"), (2518, 1, 5312, "block"), (3735, 1, 3712, "block"),
    (3642, 1, 576, "block"), (2067, 1, 1452, "by entry"), (2091, 1, 452, "by entry"), (3552, 1, 3060, "block"),
    (1292, 2, 2496, ("block", 6, 1)), (885, 2, 2560, ("block", 6, 1)), (1581, 2, 3264, ("block", 8, 1)), (1001, 2, 6848, ("block", 4, 4)),
    (671, 2, 5376, ("block", 4, 3)), (893, 3, 2240, ("block", 6, 1)), (560, 3, 3840, ("block", 8, 1)), (537, 3, 6784, ("block", 2, 7)),
])
def test_way_of_streams_of_few_entries_per_token_that_was_faster(rules, tokens, k, hidden, way):
    """Timed on the GPU, rows of two and three entries in pieces of two vectors per lane take up to 1.18 times as long as a wave per entry."""
    got = way_of(rules, tokens, k, 8, hidden)
    assert got == way if isinstance(way, tuple) or not isinstance(got, tuple) else got[0] == way


@pytest.mark.parametrize("tokens,k,hidden,way", [
    (464, 4, 2304, "wide fanout"), (492, 4, 2240, "wide fanout"), (509, 4, 4096, "wide fanout"), (301, 4, 3584, "wide fanout"), (523, 4, 2560, "block"), (773, 4, 3584, "block"),
    (919, 5, 4096, "wide fanout"), (1044, 7, 4096, "wide fanout"), (997, 8, 4096, "wide fanout"), (1518, 8, 4096, "wide fanout"),
    (953, 8, 3840, "wide fanout"), (399, 8, 4096, "block"), (1986, 8, 4096, "block"), (2043, 4, 4096, "block"), (156, 8, 4096, "block"),
    (1566, 8, 3072, "block"), (223, 5, 4096, "block"), (648, 7, 3328, "wide fanout"), (1105, 8, 3520, "wide fanout"), (1156, 4, 3584, "block"),
    (673, 8, 3072, "block"),
])
def test_way_of_streams_of_long_rows_that_was_faster(rules, tokens, k, hidden, way):
    """Timed on the GPU: four tokens in a pass over the keys take up to 1.15 times as long as a token at a time, or the other way round."""
    got = way_of(rules, tokens, k, 8, hidden)
    assert (got[0] if isinstance(got, tuple) else got) == way


def test_limits_of_the_kernels_of_stage_1(rules):
    """(each of them addresses what its way promises: a key per lane and slot, bytes of counts, 32-bit order keys)"""
    for tokens in (1, 2, 3, 63, 64, 65, 1023, 1024, 1025, 4095, 16320, 16321, 65280, 65281, 1 << 20):
        for k in (1, 2, 3, 4, 8, 15, 16, 17, 63, 64, 65):
            for ranks in (1, 8, 9, 64, 65536):
                for vecs, vec16 in ((1, 1), (256, 1), (513, 1), (896, 1), (1 << 22, 1), (37, 0), (7167, 0), (1 << 25, 0)):
                    way, entries = SEND_WAYS[rules.way(tokens, k, ranks, vecs, vec16)], tokens * k
                    pieces = -(-vecs // 256)
                    if way == "few":
                        assert entries <= 64 * rules.keys(entries) <= 1024 and k <= 64 and tokens * pieces <= 1 << 20
                    if way == "block":
                        assert entries <= 65280 and ranks <= 8 and 4 * k <= 64
                    if way == "fanout":
                        assert (ranks + 2) * entries < 2 ** 31 and tokens * pieces < 2 ** 30
                    if way == "wide fanout":
                        assert (ranks + 1) << max(1, (entries - 1).bit_length()) < 2 ** 31 and tokens * pieces < 2 ** 30
    assert rules.way(0, 2, 8, 896, 1) == 0 and SEND_WAYS[rules.way(0, 8, 8, 896, 1)] == "wide fanout"  # (which read nothing then)


def recv_way(rules, rows, hidden, layout):
    vecs, vec16, nvw = row(hidden)
    few = rules.few(rows, vecs, nvw, vec16, layout == "compact")
    if few:
        return "few, through" if few == 2 else "few, plain"
    return "scan, through" if rules.through(rows, 2 * hidden) else "scan, plain"


@pytest.mark.parametrize("hidden,rows,hint,layout", RECV_CASES)
def test_kernels_of_stage_2_that_the_gpu_tests_mean(rules, hidden, rows, hint, layout):
    assert recv_way(rules, hint, hidden, layout) == RECV_CASES[hidden, rows, hint, layout]


def test_ways_of_stage_2_that_there_are_kernels_for(rules):
    """Stores past L2 from the kernel that holds all keys are built for 8, 12 and 16 vectors per lane, plain ones of the scan
    only for rows of elements (with a plan)."""
    for hidden in [*range(8, 9000, 8), 12288, 16384, 65536, 37, 1025, 7167]:
        vecs, vec16, nvw = row(hidden)
        for rows in (0, 1, 256, 512, 513, 600, 1000, 1024, 1025, 5000):
            for layout in ("padded", "compact"):
                way = recv_way(rules, rows, hidden, layout)
                assert way != "few, through" or (vec16 and nvw in (8, 12, 16)), (hidden, rows)
                assert way != "scan, plain" or not vec16, (hidden, rows)
                assert way.startswith("scan") or rows <= 1024


@pytest.mark.parametrize("W,T,K,H", LANES)
def test_vectors_of_a_lane_that_the_gpu_tests_mean(rules, W, T, K, H):
    vecs, vec16, _ = row(H)
    tokens = W * T - W * (W - 1) // 2  # (rank r has r tokens less)
    assert rules.lanes(tokens, tokens * K, W, vecs, vec16) == LANES[W, T, K, H] and tokens * K <= 2048


@pytest.mark.parametrize("W,T,K,H,lanes", [
    (8, 60, 2, 7168, 4), (8, 100, 1, 7168, 4), (1, 900, 1, 7168, 4), (1, 1000, 1, 4096, 2), (1, 500, 2, 7168, 2), (4, 60, 4, 7168, 2),
    (2, 200, 2, 4096, 2), (1, 128, 8, 7168, 1), (8, 30, 4, 4096, 1), (8, 8, 4, 7168, 1), (1, 256, 1, 7168, 1), (1, 250, 8, 7168, 2),
    (8, 64, 2, 7167, 8), (8, 16, 8, 3001, 4), (1, 1000, 1, 7167, 8), (1, 200, 4, 3001, 4), (8, 60, 2, 1001, 4), (4, 20, 6, 4097, 4),
    (8, 8, 4, 7167, 4), (1, 16, 8, 7167, 1), (8, 4, 8, 7167, 1), (1, 16, 2, 257, 1), (1, 250, 8, 5001, 8),
])
def test_vectors_of_a_lane_that_were_fastest(rules, W, T, K, H, lanes):
    """Timed on the GPU, of one, two, four and eight: the fastest or within a tenth of it."""
    vecs, vec16, _ = row(H)
    assert rules.lanes(W * T, W * T * K, W, vecs, vec16) == lanes


def test_lanes_that_move_several_vectors_have_stores_for_a_megabyte_and_more(rules):
    """(there are no others: they store past L2)"""
    for W in (1, 2, 8):
        for K in (1, 2, 8):
            for vecs in (256, 257, 300, 512, 513, 896, 1025, 4096):
                least = next((T for T in range(W, 2048 // K + 1) if rules.lanes(T, T * K, W, vecs, 1) > 1), None)
                assert least is None or least * K * vecs * 16 >= 1 << 20, (W, K, vecs)
