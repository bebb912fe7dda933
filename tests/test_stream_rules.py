"""The rules of csrc/stream_rules.h, built with the host's compiler: which kernels the stages of a job run on."""
import ctypes as C
import shutil
import subprocess
from pathlib import Path

import pytest

from tests.test_gpu_block_streams import CASES
from tests.test_gpu_combine_block import CASES as COMBINE_CASES
from tests.test_gpu_large_streams import LONG_CASES, MAPPED_PAST_CASES, RECV_PAST_CASES
from tests.test_gpu_local_long import CASES as LOCAL_LONG_CASES
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
                   'extern "C" int vecs_of_stage_2(long long bytes, int row_vecs) { return planned_recv_vecs(bytes, row_vecs); }\n'
                   'extern "C" int long_of(long long tokens, int k, int ranks, int row_vecs, int vec16) {\n'
                   '  return long_tokens(send_way(tokens, k, ranks, row_vecs, vec16), tokens, k, ranks, row_vecs, vec16); }\n'
                   'extern "C" int vecs_of_stage_3(long long bytes, int row_vecs) { return planned_send_vecs(bytes, row_vecs); }\n'
                   'extern "C" int vecs_of_stage_4(int k, int row_vecs, int past) { return mapped_vecs(k, row_vecs, past); }\n'
                   'extern "C" int tokens_of_stage_4(long long tokens, long long rows, int k) { return combine_block(tokens, rows, k); }\n'
                   'extern "C" int tokens_of_jobs(long long tokens, int k, int ranks, int experts) {\n'
                   '  return local_long_tokens(tokens, k, ranks, experts); }\n'
                   'extern "C" int vecs_of_jobs(long long bytes, int row_vecs) { return local_long_vecs(bytes, row_vecs); }\n'
                   'extern "C" long long line(int which) {\n'
                   '  return which == 0 ? RECV_PAST_BYTES : which == 1 ? COMBINE_PAST_BYTES : which == 2 ? COMBINE_TOKENS : LOCAL_LONG_ENTRIES; }\n'
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
    dll.long_of.argtypes = [C.c_longlong] + [C.c_int] * 4
    dll.line.restype = C.c_longlong
    dll.tokens_of_stage_4.argtypes = [C.c_longlong, C.c_longlong, C.c_int]
    dll.tokens_of_jobs.argtypes = [C.c_longlong] + [C.c_int] * 3
    dll.vecs_of_stage_3.argtypes = dll.vecs_of_jobs.argtypes = [C.c_longlong, C.c_int]
    dll.vecs_of_stage_2.argtypes = [C.c_longlong, C.c_int]
    return dll


def row(hidden):
    """Vectors of 16 bytes in a row, or its elements, and vectors per lane of a wave that moves it (row_geometry)."""
    vec16 = hidden % 8 == 0
    vecs = hidden // 8 if vec16 else hidden
    nvw = next((n for n in (1, 2, 4, 6, 8, 12, 14) if vecs <= 64 * n), 16) if vec16 else 16
    return vecs, vec16, nvw


def way_of(rules, tokens, k, ranks, hidden):
    """(as dispatch_long_kernel finds them, which takes streams of 5120 entries and more over)"""
    vecs, vec16, nvw = row(hidden)
    way = SEND_WAYS[rules.way(tokens, k, ranks, vecs, vec16)]
    if way == "block":
        nvw = rules.piece(tokens, k, nvw, vec16)
        return way, nvw, -(-vecs // (64 * nvw))
    return way


@pytest.mark.parametrize("W,E,K,H,T", CASES)
def test_kernels_of_stage_1_that_the_gpu_tests_mean(rules, W, E, K, H, T):
    vecs, vec16, _ = row(H)
    own = rules.long_of(T, K, W, vecs, vec16)
    assert (("long", own) if own else way_of(rules, T, K, W, H)) == CASES[W, E, K, H, T]


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


@pytest.mark.parametrize("rows,hidden,vecs", [
    (6278, 7168, 2), (17530, 7168, 2), (21496, 7168, 1), (32613, 7168, 1), (32690, 5120, 1), (39957, 4096, 2), (32690, 4096, 2),
    (11900, 4096, 2), (32945, 2560, 2), (55992, 3072, 2), (17946, 2048, 1), (64029, 2048, 1),
])
def test_pieces_of_a_planned_stage_2(rules, rows, hidden, vecs):
    """Timed on the GPU: beyond the cache two vectors per lane of long rows take 2 % more of the four stages."""
    assert rules.vecs_of_stage_2(rows * hidden * 2, hidden // 8) == vecs


@pytest.mark.parametrize("tokens,k,hidden,own", [
    (722, 8, 136, 0), (755, 8, 336, 0), (1005, 6, 2792, 0), (613, 8, 448, 0), (2803, 6, 952, 0), (2235, 8, 728, 0), (2225, 8, 136, 0),
    (1015, 7, 416, 4), (816, 8, 2464, 4), (3590, 3, 512, 15), (2054, 8, 264, 8), (3131, 5, 80, 12), (3649, 5, 768, 8), (2675, 6, 1056, 6),
    (2055, 4, 2912, 9), (2637, 6, 1456, 10), (3212, 5, 2488, 7), (3594, 8, 3136, 8), (3731, 4, 7144, 4), (4084, 6, 5600, 4), (4096, 8, 7168, 4),
])
def test_tokens_of_a_workgroup_for_long_streams(rules, tokens, k, hidden, own):
    """Timed on the GPU: streams that stay with another kernel lose up to 13 % here, too few or too many tokens in a workgroup up to 40 %."""
    vecs, vec16, _ = row(hidden)
    assert rules.long_of(tokens, k, 8, vecs, vec16) == own


def test_limits_of_the_kernel_of_long_streams(rules):
    """(64 entries in a workgroup, keys that 1024 lanes count in bytes, whole vectors, eight ranks)"""
    for tokens in (1, 79, 80, 640, 1023, 1024, 2048, 2112, 2113, 4080, 5120, 16320, 16321, 65280, 65281, 261120, 261121):
        for k in (1, 2, 3, 5, 8, 16, 17, 63, 64, 65):
            for vecs in (1, 128, 129, 256, 257, 400, 401, 512, 513, 896, 1 << 20):
                own, entries = rules.long_of(tokens, k, 8, vecs, 1), tokens * k
                assert rules.long_of(tokens, k, 9, vecs, 1) == rules.long_of(tokens, k, 8, vecs, 0) == 0
                assert 0 <= own * k <= 64 and (not own or 5120 <= entries <= 255 * 1024)
                assert own or not 65280 < entries <= 255 * 1024 or k > 64


def test_long_streams_of_stage_1_that_the_gpu_tests_mean(rules):
    for (W, E, K, H, T), own in LONG_CASES.items():
        vecs, vec16, _ = row(H)
        assert rules.long_of(T, K, W, vecs, vec16) == own, (W, E, K, H, T)


def test_large_streams_that_the_gpu_tests_mean(rules):
    """(those that stages 2 and 4 read past the caches, and on pieces of one vector per lane and of two)"""
    for (hidden, rows), vecs in RECV_PAST_CASES.items():
        assert rows * hidden * 2 >= rules.line(0) and rules.vecs_of_stage_2(rows * hidden * 2, hidden // 8) == vecs, (hidden, rows)
    for (hidden, k, tokens), vecs in MAPPED_PAST_CASES.items():
        assert tokens * (k + 1) * hidden * 2 >= rules.line(1) and rules.vecs_of_stage_4(k, hidden // 8, 1) == vecs, (hidden, k, tokens)
    assert {k > 2 for (_, k, _), vecs in MAPPED_PAST_CASES.items() if vecs == 2} == {True, False}


@pytest.mark.parametrize("k,hidden,past,vecs", [
    (8, 7168, 1, 1), (4, 2880, 0, 1), (3, 4096, 0, 1), (3, 4096, 1, 2), (2, 4096, 0, 2), (1, 4096, 0, 2), (1, 512, 1, 1), (5, 4096, 1, 1),
])
def test_vectors_of_stage_4_that_were_faster(rules, k, hidden, past, vecs):
    """(timed on the GPU)"""
    assert rules.vecs_of_stage_4(k, hidden // 8, past) == vecs


@pytest.mark.parametrize("megabytes,hidden,vecs", [(470, 7168, 8), (336, 5120, 8), (275, 7168, 8), (235, 7168, 4), (268, 4096, 4), (29, 7168, 4)])
def test_pieces_of_a_planned_stage_3(rules, megabytes, hidden, vecs):
    """Timed on the GPU (megabytes of 10^6): eight vectors per lane of rows of more than 8 KB beyond the cache, else four."""
    assert rules.vecs_of_stage_3(megabytes * 10 ** 6, hidden // 8) == vecs


def test_tokens_of_stage_4_that_the_gpu_tests_mean(rules):
    for (T, K, H, W), tokens in COMBINE_CASES.items():
        assert rules.tokens_of_stage_4(T, T * K, K) == tokens, (T, K)
    for T in (1, 256, 257, 767, 768, 4096, 32768, 32769, 1 << 20):
        for K in (1, 2, 8, 9):
            tokens = rules.tokens_of_stage_4(T, T * K, K)
            assert tokens <= rules.line(2) and (tokens == 0) == (T <= 256 or T * K <= 512 or K > 8)


def test_movers_of_jobs_that_the_gpu_tests_mean(rules):
    for (E, K, H, T), (tokens, vecs) in LOCAL_LONG_CASES.items():
        assert rules.tokens_of_jobs(T, K, 1, E) == tokens and rules.vecs_of_jobs(T * K * H * 2, H // 8) == vecs, (E, K, H, T)
    for T in (0, 1, 255, 256, 257, 511, 512, 513, 4096, 16384, 32767, 32768, 32769):
        for K in (1, 2, 3, 8, 63, 64, 65):
            tokens = rules.tokens_of_jobs(T, K, 8, 512)
            assert (tokens == 0) == (not 1 <= T * K <= 32768 or K > 64) and tokens * K <= rules.line(3)
    assert rules.tokens_of_jobs(300, 8, 9, 9) == rules.tokens_of_jobs(300, 8, 8, 513) == 0
    for megabytes, hidden, vecs in ((235, 7168, 4), (146, 4096, 4), (92, 7168, 2), (24, 2048, 2), (300, 512, 1), (300, 1024, 2)):
        assert rules.vecs_of_jobs(megabytes * 10 ** 6, hidden // 8) == vecs
