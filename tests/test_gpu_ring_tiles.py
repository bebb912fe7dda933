"""Grouped products of few tiles (`ring_gemm_kernel`): every tile it is launched with, on walks of K shorter than the ring, as
long, and longer, with rows and columns that end inside a tile."""
import pytest
import torch

from amd_distributed_2025_amd import HIPAllToAll, MoEConfig, gemm_rs

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
# tile (RingTile) -> groups, out_dim, rows per group that the caller promises (test_tile_rules.py holds the rule to that)
RING_TILES = {1: (3, 96, 8), 2: (5, 2080, 9), 3: (3, 160, 70), 4: (6, 2080, 80)}
RING_STEPS = {1: [136, 192, 256, 264, 320, 384, 448, 512, 520, 576, 1000, 2048], 2: [264, 320, 328, 384, 448, 456, 1000, 2048],
              3: [264, 320, 328, 384, 1000, 2048], 4: [456, 512, 520, 576, 640, 1000, 2048]}


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("tile,K", [(tile, K) for tile in RING_TILES for K in RING_STEPS[tile]])
def test_rings_on_small_integers(tile, K, bias, dt):
    """Small integers, whose sums every order gives exactly (below 2^11 but for a rounding of bfloat16)."""
    groups, N, rows = RING_TILES[tile]
    print(f"ring tile={tile} K={K} bias={bias} {dt}", flush=True)
    T = 100
    a = HIPAllToAll(MoEConfig(groups, 1, K, T, dt, dt), 0, 1, device=torch.device(DEV))
    g = torch.Generator(device=DEV).manual_seed(K + tile)
    counts = [65, 0, 97, 1, 100, 32][:groups]
    x = torch.randint(-1, 2, (groups, T, K), generator=g, device=DEV).to(dt)
    w = torch.randint(-1, 2, (groups, N, K), generator=g, device=DEV).to(dt)
    b = torch.randint(-9, 10, (groups, N), generator=g, device=DEV).to(dt) if bias else None
    num = torch.tensor(counts, dtype=torch.int32, device=DEV)
    flat = torch.cat([x[e, :c] for e, c in enumerate(counts)] + [x[0, :5]]).contiguous()  # (and rows of nobody)
    hint = rows * groups
    out = a.expert_gemm(x, num, w, b, rows_hint=hint, out=torch.full((groups, T, N), 7.0, dtype=dt, device=DEV))
    packed = a.expert_gemm(flat, num, w, b, rows_hint=hint, out=torch.full((len(flat), N), 7.0, dtype=dt, device=DEV))
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


@pytest.mark.parametrize("tile", RING_TILES)
def test_rings_keep_the_bits(tile):
    """The row count picks the tile and changes no bit: against a count at which none of these runs."""
    groups, N, rows = RING_TILES[tile]
    print(f"ring bits tile={tile}", flush=True)
    for K in (1544, 2048, 2112):
        a = HIPAllToAll(MoEConfig(groups, 1, K, 130, torch.bfloat16, torch.bfloat16), 0, 1, device=torch.device(DEV))
        g = torch.Generator(device=DEV).manual_seed(K)
        x = torch.randn(groups, 130, K, generator=g, device=DEV).bfloat16()
        w = (torch.randn(groups, N, K, generator=g, device=DEV) / K ** 0.5).bfloat16()
        num = torch.tensor([130, 31, 64, 0, 66, 2][:groups], dtype=torch.int32, device=DEV)
        got, base = (a.expert_gemm(x, num, w, None, rows_hint=hint, out=torch.zeros(groups, 130, N, dtype=x.dtype, device=DEV))
                     for hint in (rows * groups, 30000 * groups))
        assert torch.equal(got, base), K


RING_LINEAR = [(1, 32, 264), (31, 64, 320), (33, 96, 328), (100, 2016, 448), (256, 1024, 384),
               (65, 7168, 768), (129, 4320, 1000), (200, 4064, 4096), (511, 2048, 1544), (250, 3936, 777 * 8)]


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("m,n,k", RING_LINEAR)
def test_plain_products(m, n, k, dt):
    """Small integers again, with stray NaNs around the operands and sentinels around the result."""
    print(f"ring linear {m} {n} {k} {dt}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(m + n + k)
    x, w = torch.full((m + 2, k), float("nan"), dtype=dt, device=DEV), torch.full((n + 2, k), float("nan"), dtype=dt, device=DEV)
    x[1:m + 1] = torch.randint(-1, 2, (m, k), generator=g, device=DEV).to(dt)
    w[1:n + 1] = torch.randint(-1, 2, (n, k), generator=g, device=DEV).to(dt)
    b = torch.randint(-9, 10, (n,), generator=g, device=DEV).to(dt)
    out = torch.full((m + 2, n), 777.0, dtype=dt, device=DEV)
    gemm_rs.local_product((x[1:m + 1], w[1:n + 1], b), out=out[1:m + 1])
    want = ((x[1:m + 1].double() @ w[1:n + 1].double().T).to(dt).double() + b.double()).to(dt)
    assert torch.equal(out[1:m + 1], want)
    assert (out[0] == 777).all() and (out[m + 1] == 777).all()
