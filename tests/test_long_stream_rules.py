"""Which kernel, and how many tokens or vectors of it, long and large streams get (`csrc/stream_rules.h`, compiled for the host), at the sizes
that the GPU tests run and at the ends of each rule."""
import ctypes as C
import shutil
import subprocess
from pathlib import Path

import pytest

from tests.test_gpu_stream_limits import COMBINE_CASES, LOCAL_CASES, LONG_CASES, MAPPED_PAST_CASES, RECV_PAST_CASES, SEND_CASES

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
                   '  return which == 0 ? RECV_PAST_BYTES : which == 1 ? COMBINE_PAST_BYTES : which == 2 ? COMBINE_TOKENS : LOCAL_LONG_ENTRIES; }\n')
    lib = src.with_suffix(".so")
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Wno-unused-function", "-shared", "-fPIC", f"-I{CSRC}", str(src), "-o", str(lib)],
                   check=True)
    dll = C.CDLL(str(lib))
    dll.way.argtypes = dll.long_of.argtypes = [C.c_longlong] + [C.c_int] * 4
    dll.line.restype = C.c_longlong
    dll.tokens_of_stage_4.argtypes = [C.c_longlong, C.c_longlong, C.c_int]
    dll.tokens_of_jobs.argtypes = [C.c_longlong] + [C.c_int] * 3
    dll.vecs_of_stage_2.argtypes = dll.vecs_of_stage_3.argtypes = dll.vecs_of_jobs.argtypes = [C.c_longlong, C.c_int]
    return dll


def row(hidden):
    """Vectors of 16 bytes in a row, or its elements."""
    return (hidden // 8, 1) if hidden % 8 == 0 else (hidden, 0)


def test_stage_1_that_the_gpu_tests_mean(rules):
    for (W, E, K, H, T), kernel in [*SEND_CASES.items(), *LONG_CASES.items()]:
        own = rules.long_of(T, K, W, *row(H))
        assert (own or SEND_WAYS[rules.way(T, K, W, *row(H))]) == kernel, (W, E, K, H, T)


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
    assert rules.long_of(tokens, k, 8, *row(hidden)) == own


@pytest.mark.parametrize("tokens,k,hidden,own", [
    (1836, 5, 1144, 0), (1627, 6, 1336, 0), (1736, 5, 1416, 0), (1046, 8, 944, 0), (1892, 5, 1608, 0), (1443, 6, 2024, 0), (2573, 7, 1528, 0), (2290, 8, 1304, 0),
    (1024, 8, 944, 4), (2049, 5, 1144, 9), (1836, 5, 512, 8), (1836, 5, 3208, 4), (2060, 4, 1144, 9), (2400, 7, 1544, 5),
])
def test_streams_just_past_a_batch_of_keys(rules, tokens, k, hidden, own):
    """Timed on the GPU: with five and more entries per token another pass over the keys costs up to 10 % more than dispatch_block_kernel."""
    assert rules.long_of(tokens, k, 8, *row(hidden)) == own


def test_limits_of_the_kernel_of_long_streams(rules):
    """(64 entries in a workgroup, keys that 1024 lanes count in bytes, whole vectors, eight ranks)"""
    for tokens in (1, 79, 80, 640, 1023, 1024, 2048, 2112, 2113, 4080, 5120, 16320, 16321, 65280, 65281, 261120, 261121):
        for k in (1, 2, 3, 5, 8, 16, 17, 63, 64, 65):
            for vecs in (1, 128, 129, 256, 257, 400, 401, 512, 513, 896, 1 << 20):
                own, entries = rules.long_of(tokens, k, 8, vecs, 1), tokens * k
                assert rules.long_of(tokens, k, 9, vecs, 1) == rules.long_of(tokens, k, 8, vecs, 0) == 0
                assert 0 <= own * k <= 64 and (not own or 5120 <= entries <= 255 * 1024)
                assert own or not 65280 < entries <= 255 * 1024 or k > 64


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
    for (E, K, H, T), (tokens, vecs) in LOCAL_CASES.items():
        assert rules.tokens_of_jobs(T, K, 1, E) == tokens and rules.vecs_of_jobs(T * K * H * 2, H // 8) == vecs, (E, K, H, T)
    for T in (0, 1, 255, 256, 257, 511, 512, 513, 4096, 16384, 32767, 32768, 32769):
        for K in (1, 2, 3, 8, 63, 64, 65):
            tokens = rules.tokens_of_jobs(T, K, 8, 512)
            assert (tokens == 0) == (not 1 <= T * K <= 32768 or K > 64) and tokens * K <= rules.line(3)
    assert rules.tokens_of_jobs(300, 8, 9, 9) == rules.tokens_of_jobs(300, 8, 8, 513) == 0
    for megabytes, hidden, vecs in ((235, 7168, 4), (146, 4096, 4), (92, 7168, 2), (24, 2048, 2), (300, 512, 1), (300, 1024, 2)):
        assert rules.vecs_of_jobs(megabytes * 10 ** 6, hidden // 8) == vecs
