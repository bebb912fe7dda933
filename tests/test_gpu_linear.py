"""`moe_a2a_linear`: the product a rank forms in the reference's gemm-rs task before the
reduce-scatter, `matmul(input, weight.T) + bias` (gemm-rs/reference.py:54-57).

Shapes are the per-rank ones of gemm-rs/task.yml (k there is the job's; a rank holds k/8).
Exact cases pin indexing, the bias and the K tail; random operands are held to the bound
that float32 accumulation in any order and the two roundings allow around the float64
value, which is far inside the task's own rtol = atol = 1e-2 (gemm-rs/reference.py:66)."""
import numpy as np
import pytest
import torch

from amd_distributed_2025_amd import _binding, all2all, gemm_rs
from oracle import moe_a2a_oracle as orc
from tests.helpers import bits, from_bits, reach_the_binding

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

TASK_TESTS, TASK_BENCHMARKS = gemm_rs.TASK_TESTS, gemm_rs.TASK_BENCHMARKS  # gemm-rs/task.yml:66-76, :80-85


def check_against_bound(out, inp, weight, bias, name, rows):
    ib, wb = bits(inp[rows]), bits(weight)
    bb = None if bias is None else bits(bias)
    exact, tol = orc.linear_bound(ib, wb, bb, name)
    got = orc.b16_to_f32(bits(out[rows]), name).astype(np.float64)
    err = np.abs(got - exact)
    worst = np.unravel_index(np.argmax(err - tol), err.shape)
    assert (err <= tol).all(), f"at {worst}: off by {err[worst]:.3e}, allowed {tol[worst]:.3e}"
    want = orc.linear(ib, wb, bb, name)
    assert (np.abs(orc.b16_to_f32(want, name).astype(np.float64) - exact) <= tol).all()
    same = float((want == bits(out[rows])).mean())
    return same


@pytest.mark.parametrize("m,n,k,has_bias,seed", TASK_TESTS + TASK_BENCHMARKS)
def test_task_shapes(m, n, k, has_bias, seed):
    print(f"linear m={m} n={n} k={k}/8 bias={has_bias}", flush=True)
    data = gemm_rs.generate_input(0, 8, m, n, k, has_bias, seed, device=DEV)
    inp, weight, bias = data
    out = torch.full((m, n), float("nan"), dtype=inp.dtype, device=DEV)
    got = gemm_rs.local_product(data, out=out)
    torch.cuda.synchronize()
    assert got.data_ptr() == out.data_ptr() and not torch.isnan(out).any()
    rng = np.random.default_rng(seed)
    rows = np.sort(rng.choice(m, size=min(m, 96), replace=False))  # a sample of rows, every column
    rows[0], rows[-1] = 0, m - 1
    same = check_against_bound(out.cpu(), inp.cpu(), weight.cpu(), None if bias is None else bias.cpu(), "bf16",
                               torch.from_numpy(rows))
    print(f"  {same:.4f} of the sampled results equal the float32 oracle to the bit", flush=True)
    assert same > 0.97
    # the task's own check against the torch expression on the device
    want = torch.matmul(inp, weight.T)
    if bias is not None:
        want = want + bias
    assert torch.allclose(out, want, rtol=1e-2, atol=1e-2)


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
# from 8 steps of K, where tiles would leave units without work: a workgroup's 4 or 8 waves split K, 32 rows at a time
@pytest.mark.parametrize("m,n,k", [(1, 32, 512), (64, 96, 520), (33, 2880, 1000), (16, 64, 1600), (64, 96, 1544),
                                   (32, 32, 3000), (65, 64, 520), (70, 64, 1000), (200, 160, 1096),
                                   # tiles of 64 x 128 (short K, few rows) ...
                                   (1, 32, 8), (64, 64, 64), (70, 96, 72), (129, 160, 360), (300, 2880, 200),
                                   # ... of 192 x 128 ...
                                   (1000, 4128, 1096),
                                   # ... and of 256 x 256; ragged last tiles in both directions and a K tail each. (WAYS
                                   # below has shapes of every way, and tests/test_tile_rules.py holds them to it.)
                                   (3000, 2944, 72), (2050, 4128, 200), (4100, 2080, 8), (3900, 4000, 1032)])
def test_small_integers_with_bias_are_exact(m, n, k, dt):
    print(f"linear integers m={m} n={n} k={k} {dt}", flush=True)
    rng = np.random.default_rng(m * n + k)
    x = rng.integers(-1, 2, (m, k))
    w = rng.integers(-1, 2, (n, k))
    b = rng.integers(-8, 9, n)
    # stray values around the operands: a K tail or a row bound that reads past its end meets NaNs
    pad = torch.full((m + 2, k), float("nan"), dtype=dt, device=DEV)
    pad[1:m + 1] = torch.from_numpy(x).to(dt)
    wpad = torch.full((n + 2, k), float("nan"), dtype=dt, device=DEV)
    wpad[1:n + 1] = torch.from_numpy(w).to(dt)
    bias = torch.from_numpy(b).to(dt).to(DEV)
    out = torch.full((m + 2, n), 777.0, dtype=dt, device=DEV)
    gemm_rs.local_product((pad[1:m + 1], wpad[1:n + 1], bias), out=out[1:m + 1])
    torch.cuda.synchronize()
    prod = (x.astype(np.float64) @ w.T.astype(np.float64)).astype(np.int64)  # exact: small integers
    want = prod + b[None, :]
    assert np.abs(want).max() <= 256 and np.abs(prod).max() <= 256  # integers both 16-bit types hold
    assert np.array_equal(out[1:m + 1].float().cpu().numpy(), want.astype(np.float32))
    assert (out[0] == 777.0).all() and (out[m + 1] == 777.0).all()
    no_bias = gemm_rs.local_product((pad[1:m + 1], wpad[1:n + 1], None))
    assert np.array_equal(no_bias.float().cpu().numpy(), prod.astype(np.float32))


def test_bias_is_added_to_the_rounded_product():
    # 1 + 2^-8 is not a bf16 value: the product 257 * 2^-8 rounds to 1.0 (ties to even) before the
    # bias 2^-7 is added, so the result is 1 + 2^-7; adding first would give 1 + 2^-8 + 2^-7 -> 1.015625
    dt = torch.bfloat16
    x = torch.zeros(1, 8, dtype=dt, device=DEV)
    w = torch.zeros(32, 8, dtype=dt, device=DEV)
    x[0, 0], x[0, 1] = 1.0, 2.0 ** -8
    w[:, 0], w[:, 1] = 1.0, 1.0
    bias = torch.full((32,), 2.0 ** -7, dtype=dt, device=DEV)
    out = gemm_rs.local_product((x, w, bias))
    want = torch.matmul(x, w.T) + bias
    assert torch.equal(out, want) and float(out[0, 0]) == 1.0 + 2.0 ** -7
    name = "bf16"
    assert np.array_equal(orc.linear(bits(x.cpu()), bits(w.cpu()), bits(bias.cpu()), name), bits(out.cpu()))


def test_both_bindings_give_the_same_bits(monkeypatch):
    """Each of them is called, and gives what the native call gives."""
    data = gemm_rs.generate_input(0, 8, 512, 4096, 12288, True, 663, device=DEV)
    native = _binding.host_calls()["linear"](all2all._raw_stream, *data)
    assert native is not None  # (taken, not refused)
    for binding in ("ctypes", "ext"):
        with monkeypatch.context() as m:
            called = reach_the_binding(m, binding)
            assert torch.equal(gemm_rs.local_product(data, binding=binding), native)
            assert called == {"linear"}
    with monkeypatch.context() as m:
        called = reach_the_binding(m, "ext")
        out = torch.full_like(native, float("nan"))
        assert gemm_rs.local_product(data, out=out, binding="ext") is out and torch.equal(out, native)
        assert called == {"linear"}


def test_arguments_are_checked():
    x = torch.zeros(4, 64, dtype=torch.bfloat16, device=DEV)
    w = torch.zeros(32, 64, dtype=torch.bfloat16, device=DEV)
    with pytest.raises(ValueError):
        gemm_rs.local_product((x, w[:, :32], None))
    with pytest.raises(ValueError):
        gemm_rs.local_product((x, w.float(), None))
    with pytest.raises(Exception, match="invalid|argument"):
        gemm_rs.local_product((x, torch.zeros(40, 64, dtype=torch.bfloat16, device=DEV), None))  # n % 32
    with pytest.raises(ValueError):
        gemm_rs.local_product((x.cpu(), w.cpu(), None))
    assert gemm_rs.custom_kernel((x, w, None)).shape == (4, 32)


@pytest.mark.parametrize("m,n,k,has_bias,seed", [(64, 2880, 2880, True, 2035), (512, 4608, 36864, False, 1597),
                                                 (2048, 4096, 7168, False, 716), (4096, 2880, 2880, True, 136)])
def test_ranks_of_a_job_sum_to_the_whole_product(m, n, k, has_bias, seed):
    """The task as a whole on one GPU: the 8 ranks' local products over their slices of K, summed by the
    stand-in reduce-scatter, against the float64 product over all of K plus 8 times the bias (every rank
    adds it before the sum, gemm-rs/reference.py:55-59), at the task's tolerance (reference.py:66) and at
    the bound the roundings to bf16 allow."""
    W = 8
    world = [gemm_rs.generate_input(r, W, m, n, k, has_bias, seed, device=DEV) for r in range(W)]
    outs = gemm_rs.run_job(world)
    whole = torch.zeros(m, n, dtype=torch.float64, device=DEV)
    size = torch.zeros(m, n, dtype=torch.float64, device=DEV)   # sum of the magnitudes that get rounded
    for inp, weight, bias in world:
        part = inp.double() @ weight.double().T
        if bias is not None:
            size += part.abs()
            part = part + bias.double()
        whole += part
        size += part.abs()
    size += whole.abs()
    for r, out in enumerate(outs):
        assert out.shape == (m // W, n) and out.dtype == torch.bfloat16
        rows = slice(r * (m // W), (r + 1) * (m // W))
        assert torch.allclose(out.double(), whole[rows], rtol=1e-2, atol=1e-2), f"rank {r}"
        # and far inside it: every value that is rounded to bf16 on the way (each rank's product, its sum
        # with the bias, the total) may be off by 2^-9 of its size; float32 sums add far less
        err = (out.double() - whole[rows]).abs()
        assert (err <= 2.0 ** -8 * size[rows] + 1e-9).all(), f"rank {r}: {float(err.max()):.3e}"
    # the ranks share the bias (drawn from the job's seed) and differ in their operands
    if has_bias:
        assert torch.equal(world[0][2], world[W - 1][2])
    assert not torch.equal(world[0][0], world[1][0])


def _random_shapes(seed):
    rng = np.random.default_rng(seed)
    shapes = []
    for lo_m, hi_m, hi_n, count in ((1, 65, 70, 12), (65, 1400, 70, 10), (1500, 4200, 140, 10)):
        for _ in range(count):
            k = 8 * int(rng.choice([rng.integers(1, 9), rng.integers(9, 64), rng.integers(64, 200)]))
            shapes.append((int(rng.integers(lo_m, hi_m)), 32 * int(rng.integers(hi_n // 2, hi_n)), k))
    return shapes


@pytest.mark.parametrize("m,n,k", _random_shapes(20251))
def test_random_shapes_of_small_integers_are_exact(m, n, k):
    """Shapes drawn at random across the ranges that pick each kernel and tile (few rows with K split over
    waves, tiles of 64 x 128, 128 x 128 and 256 x 256), ragged in every direction: small integers with a
    bias must come out exactly, with stray NaNs around the operands and sentinels around the result."""
    print(f"linear random shape m={m} n={n} k={k}", flush=True)
    dt = torch.bfloat16
    rng = np.random.default_rng(m * 7919 + n * 31 + k)
    x = rng.integers(-1, 2, (m, k))
    w = rng.integers(-1, 2, (n, k))
    b = rng.integers(-8, 9, n)
    pad = torch.full((m + 2, k), float("nan"), dtype=dt, device=DEV)
    pad[1:m + 1] = torch.from_numpy(x).to(dt)
    wpad = torch.full((n + 2, k), float("nan"), dtype=dt, device=DEV)
    wpad[1:n + 1] = torch.from_numpy(w).to(dt)
    bias = torch.from_numpy(b).to(dt).to(DEV)
    out = torch.full((m + 2, n), 777.0, dtype=dt, device=DEV)
    gemm_rs.local_product((pad[1:m + 1], wpad[1:n + 1], bias), out=out[1:m + 1])
    torch.cuda.synchronize()
    prod = (x.astype(np.float64) @ w.T.astype(np.float64)).astype(np.int64)
    want = prod + b[None, :]
    assert np.abs(want).max() <= 256 and np.abs(prod).max() <= 256
    assert np.array_equal(out[1:m + 1].float().cpu().numpy(), want.astype(np.float32))
    assert (out[0] == 777.0).all() and (out[m + 1] == 777.0).all()


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("k", [8, 64, 72, 128, 136, 192, 264, 320])
@pytest.mark.parametrize("m,n", [(3329, 3104), (1100, 4128), (1921, 3872)], ids=["256", "192", "128"])
def test_products_of_one_to_five_steps(m, n, k, dt):
    """The kernel behind the tiles of 256 x 256, 192 x 128 and 128 x 128 asks for rows up to two steps of 64 ahead and
    runs its last three steps apart: every number of steps around that, with a whole and a cut last one, and
    last tiles of one row and of 32 columns. Small integers are exact in every order."""
    print(f"linear steps m={m} n={n} k={k} {dt}", flush=True)
    gen = torch.Generator(device=DEV)
    gen.manual_seed(m + k)
    x = torch.randint(-1, 2, (m, k), device=DEV, generator=gen)
    w = torch.randint(-1, 2, (n, k), device=DEV, generator=gen)
    pad = torch.full((m + 2, k), float("nan"), dtype=dt, device=DEV)
    pad[1:m + 1] = x.to(dt)
    wpad = torch.full((n + 2, k), float("nan"), dtype=dt, device=DEV)
    wpad[1:n + 1] = w.to(dt)
    out = torch.full((m + 2, n), 777.0, dtype=dt, device=DEV)
    gemm_rs.local_product((pad[1:m + 1], wpad[1:n + 1], None), out=out[1:m + 1])
    want = x.double() @ w.double().T
    assert torch.equal(out[1:m + 1].double(), want)
    assert (out[0] == 777.0).all() and (out[m + 1] == 777.0).all()


# products of more tiles of 256 x 256 than units, and what the tiles are of which a workgroup has a next one: whole, of too
# few columns, of 128 to 255 rows, of less (tests/test_tile_rules.py works it out)
WITH_A_NEXT_TILE = {(4100, 4128): {"whole"}, (5120, 7200): {"whole", "columns"}, (4738, 4128): {"whole", "columns", "half"},
                    (4736, 4128): {"whole", "columns", "half"}, (4863, 4128): {"whole", "columns", "half"},
                    (4735, 4128): {"whole", "columns", "less"}, (4613, 4128): {"whole", "columns", "less"}}


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("k", [8, 64, 200, 448])
@pytest.mark.parametrize("m,n", WITH_A_NEXT_TILE, ids=["289 of 256", "580 of 256", *[f"{m}x{n}" for m, n in list(WITH_A_NEXT_TILE)[2:]]])
def test_more_tiles_than_workgroups(m, n, k, bias, dt):
    """Workgroups take a second and a third tile, whose first rows are asked for ahead of the results of the tile
    before, and waited for by counting the stores of that one: as many as whole bands, half as many, none. Small integers, whose sums (|x @ w.T + b| <= 448 + 20 here at
    most, and in fact far below 256) both types hold."""
    print(f"linear m={m} n={n} k={k} bias={bias} {dt}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(m + n + k)
    x = torch.randint(-1, 2, (m, k), generator=g, device=DEV).to(dt)
    w = torch.randint(-1, 2, (n, k), generator=g, device=DEV).to(dt)
    b = torch.randint(-20, 21, (n,), generator=g, device=DEV).to(dt) if bias else None
    want = x.float() @ w.float().T
    assert want.abs().max() < 236
    for _ in range(2):
        out = torch.full((m, n), float("nan"), dtype=dt, device=DEV)
        gemm_rs.local_product((x, w, b), out=out)
        assert torch.equal(out.float(), want if b is None else want + b.float())


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("m", [1, 32, 33, 64])
@pytest.mark.parametrize("k", [512, 520, 768, 832, 1472, 1536, 1592, 2048, 2112, 2624, 3208, 4096])
def test_few_rows_whatever_a_wave_has_to_walk(m, k, dt):
    """Two to seven steps of 64 for each of the four or eight waves that share K, even and odd, the last one whole or
    not, with a bias. Small integers, whose sums every order gives exactly and float32 holds; rounded once before the bias
    and once after."""
    n = 96
    print(f"linear m={m} n={n} k={k} {dt}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(m + k)
    x = torch.randint(-1, 2, (m, k), generator=g, device=DEV).to(dt)
    w = torch.randint(-1, 2, (n, k), generator=g, device=DEV).to(dt)
    b = torch.randint(-9, 10, (n,), generator=g, device=DEV).to(dt)
    out = torch.full((m + 2, n), 777.0, dtype=dt, device=DEV)
    gemm_rs.local_product((x, w, b), out=out[1:m + 1])
    want = ((x.double() @ w.double().T).to(dt).double() + b.double()).to(dt)
    assert torch.equal(out[1:m + 1], want)
    assert (out[0] == 777.0).all() and (out[m + 1] == 777.0).all()


# rows and columns that csrc/tile_rules.h gives to each way of cutting a product (tests/test_tile_rules.py asks it), from
# eight steps of K on: last row blocks of one row and whole ones, last column tiles of 32 columns and whole ones
WAYS = {"SPLIT_32": [(65, 96), (64, 4096), (96, 2720), (97, 32), (321, 480)],
        "SPLIT_64": [(64, 7168), (129, 1728), (192, 2048), (449, 992)],
        "TILES_64x128": [(547, 2688), (513, 3104), (193, 7200)],
        "TILES_128x128": [(825, 2624), (769, 4128)],
        "PHASED_128": [(1024, 8192), (1921, 3872)],
        "PHASED_192": [(1536, 3360), (2113, 2336), (2017, 2688), (1345, 4000)],
        "PHASED_256": [(1646, 5056), (2305, 4000)]}


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("k", [512, 520, 1472, 1544, 2048, 4096])
@pytest.mark.parametrize("way,m,n", [(way, *mn) for way, shapes in WAYS.items() for mn in shapes])
def test_every_way_of_cutting_a_product(way, m, n, k, dt):
    """Four and eight waves on a workgroup's K, a cut last step, rows 4 KB apart; several row blocks of 32 and of 64 rows
    beside each other. Small integers, whose sums every order gives exactly and float32 holds; rounded once before the
    bias and once after. Stray NaNs around the operands, sentinels around the result."""
    print(f"linear {way} m={m} n={n} k={k} {dt}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(m + n + k)
    pad = torch.full((m + 2, k), float("nan"), dtype=dt, device=DEV)
    pad[1:m + 1] = torch.randint(-1, 2, (m, k), generator=g, device=DEV).to(dt)
    wpad = torch.full((n + 2, k), float("nan"), dtype=dt, device=DEV)
    wpad[1:n + 1] = torch.randint(-1, 2, (n, k), generator=g, device=DEV).to(dt)
    b = torch.randint(-9, 10, (n,), generator=g, device=DEV).to(dt)
    out = torch.full((m + 2, n), 777.0, dtype=dt, device=DEV)
    gemm_rs.local_product((pad[1:m + 1], wpad[1:n + 1], b), out=out[1:m + 1])
    want = ((pad[1:m + 1].double() @ wpad[1:n + 1].double().T).to(dt).double() + b.double()).to(dt)
    assert torch.equal(out[1:m + 1], want)
    assert (out[0] == 777.0).all() and (out[m + 1] == 777.0).all()
