"""The tiles of the grouped product (`moe_a2a_expert_gemm` and its compact form): blocks of 32, 64 or 128 rows that
stream the weights, 64 x 128, 128 x 128 and 192, 256 or 320 rows x 256 columns, which of them from the caller's row
count. The row count must change no bit of the result, and K may start anywhere in a group's walk (rows a multiple of
4 KB apart do)."""
import pytest
import torch

from amd_distributed_2025_amd import HIPAllToAll, MoEConfig

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
# rows per group -> the kernel, by groups, at N = 7168 and every K below (csrc/tile_rules.h; test_tile_rules.py holds the
# kernels to that)
KERNELS = {3: {20: "stream 32, four steps ahead", 0: "ring 32 x 32", 50: "ring 64 x 128", 60: "tiles 64", 100: "tiles 128",
               150: "tiles 192", 600: "tiles 256", 800: "tiles 320"},
           5: {8: "stream 32, two steps ahead", 20: "stream 64", 50: "stream 128", 100: "tiles 192", 230: "tiles 256",
               300: "tiles 320"}}


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("groups,counts", [
    (3, [1, 193, 257]), (3, [700, 0, 31]), (3, [192, 256, 320]), (3, [64, 65, 63]),
    (5, [321, 1, 0, 33, 640]), (5, [320, 319, 289, 288, 641]),
    (5, [704, 704, 650, 704, 704]),  # more rows than any of the row counts: workgroups take a second tile, some a third
])
@pytest.mark.parametrize("K", [8, 200, 2048, 2112])  # one short step; a tail; a walk that starts apart; one that does not
def test_every_kernel_gives_the_same_bits(groups, counts, K, bias, dt):
    print(f"tiles groups={groups} counts={counts} K={K} bias={bias} {dt}", flush=True)
    N, T = 7168, 704
    a = HIPAllToAll(MoEConfig(groups, 1, K, T, dt, dt), 0, 1, device=torch.device(DEV))
    g = torch.Generator(device=DEV).manual_seed(K + sum(counts))
    x = torch.randn(groups, T, K, generator=g, device=DEV).to(dt)
    w = (torch.randn(groups, N, K, generator=g, device=DEV) / K ** 0.5).to(dt)
    b = torch.randn(groups, N, generator=g, device=DEV).to(dt) if bias else None
    num = torch.tensor(counts, dtype=torch.int32, device=DEV)
    flat = torch.cat([x[e, :c] for e, c in enumerate(counts)] + [x[0, :5]]).contiguous()  # (and rows of nobody)

    def run(rows, hint):
        out = torch.full((*rows.shape[:-1], N), 7.0, dtype=dt, device=DEV)
        return a.expert_gemm(rows, num, w, b, rows_hint=hint, out=out)

    base = run(x, next(iter(KERNELS[groups])) * groups)  # (streams the weights in blocks of 32 rows)
    ulp = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dt]  # of one rounding, to either side
    for e, c in enumerate(counts):
        want = x[e, :c].double() @ w[e].double().T
        # K float32 sums and a rounding; with a bias a second one, and the first is of the sum without it
        bound = ulp * want.abs() + 2.0 ** -24 * K * (x[e, :c].double().abs() @ w[e].double().abs().T)
        if bias:
            want = want + b[e].double()
            bound = (1 + ulp) * bound + ulp * want.abs()
        assert ((base[e, :c].double() - want).abs() <= bound + 2.0 ** -24).all(), f"group {e}"
        assert (base[e, c:] == 7).all()
    for rows in KERNELS[groups]:
        got = run(x, rows * groups)
        assert torch.equal(got, base), f"row count {rows} per group"
        got = run(flat, rows * groups)
        at = 0
        for e, c in enumerate(counts):
            assert torch.equal(got[at:at + c], base[e, :c]), f"compact, row count {rows} per group, group {e}"
            at += c
        assert (got[at:] == 7).all()


FEW_STEPS = [64, 128, 136, 192, 328, 392]  # one to seven steps of 64, the last one whole or not


@pytest.mark.parametrize("K", FEW_STEPS)
def test_few_steps_on_the_ring_of_half_steps(K):
    """320 rows: weights go round a ring of five half steps. Walks shorter than the ring, as long, and longer,
    on small integers, whose sums every order gives exactly; tiles of one to ten bands of 32 rows."""
    print(f"ring of halves K={K}", flush=True)
    counts, N = [289, 330, 61], 7168
    a = HIPAllToAll(MoEConfig(3, 1, K, 704, torch.bfloat16, torch.bfloat16), 0, 1, device=torch.device(DEV))
    g = torch.Generator(device=DEV).manual_seed(K)
    x = torch.randint(-1, 2, (3, 704, K), generator=g, device=DEV).bfloat16()
    w = torch.randint(-1, 2, (3, N, K), generator=g, device=DEV).bfloat16()
    num = torch.tensor(counts, dtype=torch.int32, device=DEV)
    for rows in (1, 32, 65, 97, 129, 161, 193, 225, 257, 320):
        num[2] = rows
        out = a.expert_gemm(x, num, w, None, rows_hint=800 * 3, out=torch.full((3, 704, N), 7.0, dtype=x.dtype, device=DEV))
        for e, c in enumerate([*counts[:2], rows]):
            assert torch.equal(out[e, :c], (x[e, :c].double() @ w[e].double().T).float().bfloat16()), (rows, e)
            assert (out[e, c:] == 7).all()


# groups, N, K -> rows per group and the kernel, for weights of 256 MB and more, which are read with loads that leave nothing
# in the caches: every kernel of the grouped product has such a form
PAST_THE_CACHE = {(3, 7168, 6272): {20: "stream 32, four steps ahead", 50: "ring 64 x 128", 60: "tiles 64", 100: "tiles 128",
                                    150: "tiles 192"},
                  (5, 7168, 3752): {8: "ring 32 x 64", 30: "ring 64 x 64", 230: "tiles 256", 300: "tiles 320"},
                  (8, 1024, 16384): {1: "ring 32 x 32"},
                  (64, 2048, 1024): {2: "stream 32, two steps ahead", 20: "stream 64", 50: "stream 128"}}


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("groups,N,K", PAST_THE_CACHE)
def test_weights_that_the_cache_cannot_hold(groups, N, K, dt):
    """Small integers, whose sums every order gives exactly (|sums| < 2^11 here, which float16 holds; bfloat16
    rounds them once)."""
    print(f"past the cache groups={groups} N={N} K={K} {dt}", flush=True)
    T = 330
    a = HIPAllToAll(MoEConfig(groups, 1, K, T, dt, dt), 0, 1, device=torch.device(DEV))
    g = torch.Generator(device=DEV).manual_seed(K)
    x = torch.randint(-1, 2, (groups, T, K), generator=g, device=DEV).to(dt)
    w = torch.randint(-1, 2, (groups, N, K), generator=g, device=DEV).to(dt)
    b = torch.randint(-9, 10, (groups, N), generator=g, device=DEV).to(dt)
    counts = ([257, 0, 33, 321, 1] + [0, 64, 2, 31] * 15)[:groups]
    num = torch.tensor(counts, dtype=torch.int32, device=DEV)
    want = [((x[e, :c].double() @ w[e].double().T).to(dt).double() + b[e].double()).to(dt) for e, c in enumerate(counts)]
    for rows in PAST_THE_CACHE[groups, N, K]:
        out = a.expert_gemm(x, num, w, b, rows_hint=rows * groups, out=torch.full((groups, T, N), 7.0, dtype=dt, device=DEV))
        for e, c in enumerate(counts):
            assert torch.equal(out[e, :c], want[e]), (rows, e)
            assert (out[e, c:] == 7).all()


@pytest.mark.parametrize("M,N,K", [(1, 32, 2048), (33, 96, 4096), (64, 2080, 2048), (8, 1024, 6144), (64, 64, 8192)])
def test_few_rows_whose_walks_of_K_start_apart(M, N, K):
    """`moe_a2a_linear` on at most 64 rows of a multiple of 2048 inputs: small integers, whose sums every order
    gives exactly (|sums| <= K < 2^24, and those a bfloat16 cannot hold are rounded once)."""
    from amd_distributed_2025_amd import gemm_rs

    print(f"linear M={M} N={N} K={K}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    x = torch.randint(-1, 2, (M, K), generator=g, device=DEV).bfloat16()
    w = torch.randint(-1, 2, (N, K), generator=g, device=DEV).bfloat16()
    got = gemm_rs.local_product((x, w, None))
    assert torch.equal(got, (x.double() @ w.double().T).float().bfloat16())


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("M,N,K", [(1586, 2432, 200), (2048, 2048, 64), (1025, 2080, 8), (2047, 2080, 136)])
def test_one_round_of_square_tiles(M, N, K, dt):
    """128 x 128 tiles on both sides of one per unit (247, 256, 153, 272 of them), small integers, whose sums
    both types hold."""
    from amd_distributed_2025_amd import gemm_rs

    print(f"linear M={M} N={N} K={K} {dt}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    x = torch.randint(-1, 2, (M, K), generator=g, device=DEV).to(dt)
    w = torch.randint(-1, 2, (N, K), generator=g, device=DEV).to(dt)
    b = torch.randint(-9, 10, (N,), generator=g, device=DEV).to(dt)
    got = gemm_rs.local_product((x, w, b))
    assert torch.equal(got.double(), x.double() @ w.double().T + b.double())
