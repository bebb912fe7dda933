"""Products of about one tile per unit (`sliced_gemm_kernel`): every tile it is launched with, on walks of K shorter than its ring, as
long, and longer, with rows and columns that end inside a tile, and with more tiles than the caller's row count lets expect."""
import ctypes as C
import shutil
import subprocess
from pathlib import Path

import pytest
import torch

from amd_distributed_2025_amd import HIPAllToAll, MoEConfig, gemm_rs

DEV = "cuda:0"
DT = pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
TILES = ["32x64", "64x64", "64x128", "128x128", "192x128"]  # SlicedTile, from 1 on
STEPS = [8, 64, 72, 128, 136, 192, 200, 264, 328, 512]
# tile -> groups, out_dim, rows per group that the caller promises; K
GROUPED = {"64x64": (3, 160, 70, [264, 320, 328, 384, 1000, 2048]), "64x128": (3, 2080, 200, STEPS), "128x128": (3, 2080, 400, STEPS),
           "192x128": (3, 2080, 550, STEPS)}
# weights that are read past the caches (rows of one tile per group)
STREAMED = {"64x64": (8, 1024, 60, 16384), "64x128": (8, 3072, 58, 5632), "128x128": (8, 2048, 115, 8192), "192x128": (8, 2048, 150, 8192)}
# rows, out_dim, K
PLAIN = {"32x64": [(m, n, k) for m, n in [(1, 1056), (65, 2016)] for k in [8, 64, 128, 192, 200]] + [(70, 5024, 1544), (96, 5440, 2048), (33, 7008, 512)],
         "64x64": [(m, n, k) for m, n in [(513, 1056), (300, 2016)] for k in [8, 64, 128, 192, 200]] + [(200, 4064, 1544), (511, 2016, 2048)],
         "64x128": [(m, n, k) for m, n in [(700, 2016), (321, 4128)] for k in STEPS] + [(700, 2016, 2048)]}


@pytest.fixture(scope="module")
def chosen(tmp_path_factory):
    """The tile of a grouped product, and of a plain one, as launch_grouped_dense and launch_linear ask for it; and whether weights stream."""
    if shutil.which("g++") is None:
        pytest.skip("g++ not installed")
    src = tmp_path_factory.mktemp("rules") / "rules.cpp"
    src.write_text('#include "tile_rules.h"\n'
                   'extern "C" int grouped(long long hint, int groups, int n, int k) {\n'
                   '  const RingTile ring = grouped_ring(hint, groups, n, k);\n'
                   '  return grouped_slices(ring, hint >= 56ll * groups && !ring ? grouped_tile_bands(hint, groups, n, k) : 0, hint, groups, n);\n'
                   '}\n'
                   'extern "C" int plain(long long m, long long n, long long k) {\n'
                   '  const RingTile ring = linear_ring(m, n, k);\n'
                   '  return linear_slices(ring, ring ? STREAM_WEIGHTS : linear_way(m, n, k), m, n, k);\n'
                   '}\n'
                   'extern "C" int past(int groups, long long hint, int n, int k) { return weights_past_the_cache(groups, hint, n, k); }\n')
    lib = src.with_suffix(".so")
    csrc = Path(__file__).resolve().parent.parent / "amd_distributed_2025_amd" / "csrc"
    subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Wno-unused-function", "-shared", "-fPIC", f"-I{csrc}", str(src), "-o", str(lib)],
                   check=True)
    dll = C.CDLL(str(lib))
    dll.grouped.argtypes, dll.plain.argtypes = [C.c_longlong, C.c_int, C.c_int, C.c_int], [C.c_longlong] * 3
    dll.past.argtypes = [C.c_int, C.c_longlong, C.c_int, C.c_int]
    return dll


def test_the_sizes_here_reach_every_tile(chosen):
    for tile, (groups, n, rows, ks) in GROUPED.items():
        for k in ks:
            assert TILES[chosen.grouped(rows * groups, groups, n, k) - 1] == tile, (tile, k)
    for tile, (groups, n, rows, k) in STREAMED.items():
        assert TILES[chosen.grouped(rows * groups, groups, n, k) - 1] == tile and chosen.past(groups, rows * groups, n, k), tile
        assert rows <= int(tile.split("x")[0])
    for tile, shapes in PLAIN.items():
        for shape in shapes:
            assert TILES[chosen.plain(*shape) - 1] == tile, (tile, shape)


def check_grouped(tile, groups, N, rows, K, counts, bias, dt):
    """Small integers, whose float32 sums every order gives exactly; one rounding, with a bias two."""
    print(f"slices {tile} K={K} counts={counts} bias={bias} {dt}", flush=True)
    T = max(counts)
    a = HIPAllToAll(MoEConfig(groups, 1, K, T, dt, dt), 0, 1, device=torch.device(DEV))
    g = torch.Generator(device=DEV).manual_seed(K + T)
    x = torch.randint(-1, 2, (groups, T, K), generator=g, device=DEV, dtype=torch.int8).to(dt)
    w = torch.randint(-1, 2, (groups, N, K), generator=g, device=DEV, dtype=torch.int8).to(dt)
    b = torch.randint(-9, 10, (groups, N), generator=g, device=DEV).to(dt) if bias else None
    num = torch.tensor(counts, dtype=torch.int32, device=DEV)
    flat = torch.cat([x[e, :c] for e, c in enumerate(counts)] + [x[0, :5]]).contiguous()  # (and rows of nobody)
    out = a.expert_gemm(x, num, w, b, rows_hint=rows * groups, out=torch.full((groups, T, N), 7.0, dtype=dt, device=DEV))
    packed = a.expert_gemm(flat, num, w, b, rows_hint=rows * groups, out=torch.full((len(flat), N), 7.0, dtype=dt, device=DEV))
    at = 0
    for e, c in enumerate(counts):
        want = (x[e, :c].double() @ w[e].double().T).to(dt)
        if bias:
            want = (want.double() + b[e].double()).to(dt)
        assert torch.equal(out[e, :c], want), e
        assert (out[e, c:] == 7).all()
        assert torch.equal(packed[at:at + c], want), e
        at += c
    assert (packed[at:] == 7).all()


@pytest.mark.gpu
@DT
@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("tile,K", [(tile, k) for tile, (*_, ks) in GROUPED.items() for k in ks])
def test_grouped_products(tile, K, bias, dt):
    groups, N, rows, _ = GROUPED[tile]
    # (in the second, more tiles than workgroups, and first rows at the end of a tile before them)
    for counts in ([385, 0, 193], [700, 641, 577]):
        check_grouped(tile, groups, N, rows, K, counts, bias, dt)


@pytest.mark.gpu
@pytest.mark.parametrize("tile", STREAMED)
def test_weights_past_the_caches(tile):
    groups, N, rows, K = STREAMED[tile]
    check_grouped(tile, groups, N, rows, K, [rows, 0, 1, rows, 33, rows, 3 * rows, 16], True, torch.bfloat16)


@pytest.mark.gpu
@pytest.mark.parametrize("tile", GROUPED)
def test_the_tile_changes_no_bit(tile):
    groups, N, rows, _ = GROUPED[tile]
    print(f"slices bits {tile}", flush=True)
    for K in (1544, 2048):  # (2048: groups start their walk apart)
        a = HIPAllToAll(MoEConfig(groups, 1, K, 385, torch.bfloat16, torch.bfloat16), 0, 1, device=torch.device(DEV))
        g = torch.Generator(device=DEV).manual_seed(K)
        x = torch.randn(groups, 385, K, generator=g, device=DEV).bfloat16()
        w = (torch.randn(groups, N, K, generator=g, device=DEV) / K ** 0.5).bfloat16()
        num = torch.tensor([385, 31, 193], dtype=torch.int32, device=DEV)
        got, base = (a.expert_gemm(x, num, w, None, rows_hint=hint, out=torch.zeros(groups, 385, N, dtype=x.dtype, device=DEV))
                     for hint in (rows * groups, 30000 * groups))
        assert torch.equal(got, base), K


@pytest.mark.gpu
@DT
@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("tile", PLAIN)
def test_plain_products(tile, bias, dt):
    """Small integers again, with NaNs around the operands and sentinels around the result."""
    for m, n, k in PLAIN[tile]:
        print(f"slices plain {m} {n} {k} {bias} {dt}", flush=True)
        g = torch.Generator(device=DEV).manual_seed(m + n + k)
        x, w = (torch.full((r + 2, k), float("nan"), dtype=dt, device=DEV) for r in (m, n))
        x[1:m + 1] = torch.randint(-1, 2, (m, k), generator=g, device=DEV).to(dt)
        w[1:n + 1] = torch.randint(-1, 2, (n, k), generator=g, device=DEV).to(dt)
        b = torch.randint(-9, 10, (n,), generator=g, device=DEV).to(dt) if bias else None
        out = torch.full((m + 2, n), 7.0, dtype=dt, device=DEV)
        gemm_rs.local_product((x[1:m + 1], w[1:n + 1], b), out=out[1:m + 1])
        want = (x[1:m + 1].double() @ w[1:n + 1].double().T).to(dt)
        if bias:
            want = (want.double() + b.double()).to(dt)
        assert torch.equal(out[1:m + 1], want), (m, n, k)
        assert (out[0] == 7).all() and (out[m + 1] == 7).all()
