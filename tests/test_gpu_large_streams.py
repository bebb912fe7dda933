"""Streams that the caches do not hold: rows read past them, in pieces of one, two, four or eight vectors per lane
(`csrc/stream_rules.h`). Results are the ones of the other kernels, bit for bit."""
import numpy as np
import pytest
import torch

from amd_distributed_2025_amd import HIPAllToAll, LocalWorld, WORKLOADS, _lib, generate_world
from amd_distributed_2025_amd.task import MoEConfig
from tests.helpers import bits, run_oracle
from tests.test_gpu_long_streams import run_long
from tests.test_gpu_parity import DEV, EDGE

pytestmark = pytest.mark.gpu


# rows of each stream: 42 to 49 MB, above the lines of the expert, of stage 3 and of stage 2
@pytest.mark.parametrize("hidden_dim,tokens,K,dtype", [
    (1032, 2560, 8, "bf16"),   # 129 vectors: a piece of one vector, one lane of it used
    (2048, 2816, 4, "fp16"),   # 256: whole pieces of one
    (2056, 2816, 4, "bf16"),   # 257: pieces of two, and one lane of the last
    (4104, 704, 8, "fp16"),    # 513
])
def test_streams_of_more_than_40_mb(hidden_dim, tokens, K, dtype):
    print(f"{tokens * K} rows of {hidden_dim}", flush=True)
    assert tokens * K * hidden_dim * 2 > 40 << 20
    spec = dict(world_size=2, num_experts=16, experts_per_token=K, hidden_dim=hidden_dim, max_num_tokens=tokens,
                num_tokens="full", routing="uniform", weights="softmax", dtype=dtype)
    run_long(generate_world(spec, 3), long_stream_rows=0)


# ranks, experts, entries per token, hidden, tokens -> tokens of a workgroup of dispatch_long_kernel
LONG_CASES = {
    (8, 16, 1, 8, 5120): 20,     # the shortest it takes, one entry per token; a vector per row
    (3, 15, 5, 520, 1024): 4,    # 65 vectors, experts per rank no power of two
    (2, 6, 6, 1032, 2561): 10,   # 60 entries in a workgroup, the last of which owns one token
    (8, 8, 7, 64, 2311): 9,      # an expert per rank
    (4, 256, 64, 16, 1021): 1,   # 64 entries of a token, more entries than the kernel before it takes
    (5, 20, 3, 3208, 1800): 4,   # 401 vectors: twice as many workgroups
    (4, 8, 4, 4104, 2000): 2,    # 513: four times
    (2, 4, 2, 8, 32641): 32,     # 65282 entries
    (1, 2, 1, 7168, 5121): 11,
}


@pytest.mark.parametrize("W,E,K,hidden_dim,tokens", LONG_CASES)
def test_stage_one_of_long_streams(W, E, K, hidden_dim, tokens):
    print(f"stage 1, {W} ranks x {tokens} tokens x {K} of {hidden_dim}", flush=True)
    spec = dict(world_size=W, num_experts=E, experts_per_token=K, hidden_dim=hidden_dim, max_num_tokens=tokens,
                num_tokens="full", routing="zipf" if K < E else "uniform", weights="softmax", dtype="bf16")
    world = generate_world(spec, 9)[:1]
    cfg, d = world[0][0], world[0][1]
    ids = d.indices.to(DEV)
    ids[tokens // 2] = E + 3  # names no expert: behind all ranks' rows
    a = HIPAllToAll(cfg, 0, W, device=DEV)
    x = d.x.to(DEV)
    counts, buf, meta = a.dispatch_send(x, ids)
    torch.cuda.synchronize()
    flat = ids.flatten().long()
    dest = torch.where(flat < E, flat // (E // W), W)
    order = torch.argsort(dest, stable=True)
    rows = order.numel()
    assert torch.equal(counts.long(), torch.bincount(dest, minlength=W + 1)[:W])
    assert torch.equal(buf[:rows], x[order // K])
    want = torch.stack([flat[order], torch.zeros_like(order), order // K, order % K, torch.zeros_like(order)], 1).int()
    assert torch.equal(meta[:rows], want)


@pytest.mark.parametrize("hidden_dim", [8, 520, 1024, 1032, 4096, 4104, 7168])
@pytest.mark.parametrize("layout", ["padded", "compact"])
def test_a_few_rows_in_a_launch_for_hundreds_of_megabytes(hidden_dim, layout):
    """The expert and stage 3 size their launches and choose their kernels by the caller's row count, which may lie above the
    rows that there are: below and above 24, 256 and 384 MB the same rows give the same results."""
    nle, tokens = 3, 37
    cfg = MoEConfig(nle, 2, hidden_dim, tokens, torch.bfloat16, torch.bfloat16)
    results = []
    for megabytes in (0, 25, 50, 300, 400):
        a = HIPAllToAll(cfg, 0, 1, device=DEV, layout=layout, compact_rows=96 if layout == "compact" else None)
        gen = torch.Generator(device=DEV)
        gen.manual_seed(7)
        rows = tokens * 2
        hint = max(rows, (megabytes << 20) // (2 * hidden_dim))
        recv = torch.randn(rows, hidden_dim, device=DEV, generator=gen).to(torch.bfloat16)
        meta = torch.zeros(rows, 5, dtype=torch.int32, device=DEV)
        meta[:, 0] = torch.arange(rows, device=DEV) * 7 % nle
        meta[:, 2] = torch.arange(rows, device=DEV) // 2
        meta[:, 3] = torch.arange(rows, device=DEV) % 2
        counts = torch.tensor([rows], dtype=torch.int32, device=DEV)
        num, ex, em = a.dispatch_recv(counts, recv, meta, rows)
        ex_rows, plan = ex.shape[0], a._ws["send_back_plan"]
        ey, back = torch.zeros_like(ex), torch.zeros_like(recv)
        back_meta, back_counts = torch.zeros_like(meta), torch.zeros_like(counts)
        p, st = _lib_pointer, torch.cuda.current_stream().cuda_stream
        print(f"{layout}, {hidden_dim}, launches for {megabytes} MB", flush=True)
        if layout == "compact":
            _lib.call("moe_a2a_expert_scale_compact", a.shape, p(ex), p(num), hint, ex_rows, _lib.BF16, _lib.BF16, p(ey), st)
            _lib.call("moe_a2a_combine_send_compact", a.shape, p(ey), p(em), p(num), hint, ex_rows, rows, p(back),
                      p(back_meta), p(back_counts), p(plan), st)
        else:
            _lib.call("moe_a2a_expert_scale", a.shape, p(ex), p(num), hint, _lib.BF16, _lib.BF16, p(ey), st)
            _lib.call("moe_a2a_combine_send", a.shape, p(ey), p(em), p(num), hint, rows, p(back), p(back_meta), p(back_counts),
                      p(plan), st)
        torch.cuda.synchronize()
        order = torch.argsort(meta[:, 0], stable=True)
        assert torch.equal(back, recv[order]) and torch.equal(back_meta, meta[order])  # (rank 0: times one)
        results.append((ey, back_counts))
    for ey, back_counts in results[1:]:
        assert torch.equal(ey, results[0][0]) and torch.equal(back_counts, results[0][1])


def _lib_pointer(t):
    return t.data_ptr()


def run_compact(world, binding="ctypes", exact_hints=True):
    cfg, W = world[0][0], len(world)
    lw = LocalWorld(cfg, W, device=DEV, layout="compact", long_stream_rows=0, binding=binding, exact_hints=exact_hints)
    ys = lw.run([d.to(DEV) for _, d, _, _ in world])
    torch.cuda.synchronize()
    want = run_oracle(world)
    for r in range(W):
        g, a = lw.trace[r], lw.ranks[r]
        num = want[r].expert_num_tokens
        R = int(num.sum())
        assert np.array_equal(g["expert_num_tokens"].cpu().numpy(), num), r
        assert np.array_equal(a.expert_offsets.cpu().numpy(), np.concatenate([[0], np.cumsum(num)])), r
        assert np.array_equal(bits(g["expert_x"][:R]), want[r].expert_rows), r
        assert np.array_equal(g["expert_meta"][:R].cpu().numpy(), want[r].expert_meta_rows), r
        assert np.array_equal(bits(ys[r]), want[r].y), r


@pytest.mark.parametrize("name", ["C1", "C2", "C3", "C4", "C5"] + sorted(EDGE))
def test_planned_places_in_the_compact_layout(name):
    print(f"compact, planned, {name}", flush=True)
    spec = WORKLOADS[name] if name in WORKLOADS else dict(dict(routing="uniform", weights="rand"), **EDGE[name])
    run_compact(generate_world(spec, 17))


@pytest.mark.parametrize("W,nle,K,tokens", [(2, 256, 8, 1500), (4, 3, 5, 2600), (1, 64, 8, 1025), (3, 257, 2, 300)])
@pytest.mark.parametrize("exact_hints", [True, False])
def test_planned_places_of_many_tiles(W, nle, K, tokens, exact_hints):
    """Several tiles of 1024 rows, more rows than the first batch of a tile (8192), up to 256 experts (257: the scan), hints above
    and, under skewed routing, below the rows that arrive; the extension's wrapper."""
    print(f"compact, planned, {W} x {nle} experts, {tokens} tokens x {K}", flush=True)
    spec = dict(world_size=W, num_experts=W * nle, experts_per_token=K, hidden_dim=16, max_num_tokens=tokens,
                num_tokens="full", routing="zipf", weights="rand", dtype="bf16")
    run_compact(generate_world(spec, 5), exact_hints=exact_hints, binding="ext" if exact_hints else "ctypes")


def test_planned_places_of_a_shape_that_could_hold_far_more():
    """128 experts that could each take 1.2 million rows, of which 4100 arrive: more than the experts' pieces could be numbered."""
    W, nle, H, R = 8, 128, 7168, 4100
    a = HIPAllToAll(MoEConfig(W * nle, 1, H, 150000, torch.bfloat16, torch.bfloat16), 3, W, device=DEV, layout="compact", compact_rows=4200)
    gen = torch.Generator(device=DEV)
    gen.manual_seed(1)
    recv = torch.randn(R, H, device=DEV, generator=gen).to(torch.bfloat16)
    meta = torch.randint(0, 1000, (R, 5), device=DEV, generator=gen, dtype=torch.int32)
    meta[:, 0] = 3 * nle + torch.randint(0, nle, (R,), device=DEV, generator=gen, dtype=torch.int32)
    counts = torch.tensor([R - 70] + [10] * 7, dtype=torch.int32, device=DEV)
    num, ex, em = a.dispatch_recv(counts, recv, meta, R)
    torch.cuda.synchronize()
    order = torch.argsort(meta[:, 0], stable=True)
    assert torch.equal(ex[:R], recv[order]) and torch.equal(em[:R], meta[order])
    want = torch.bincount(meta[:, 0] - 3 * nle, minlength=nle)
    assert torch.equal(num.long(), want) and torch.equal(a.expert_offsets[1:].long(), want.cumsum(0))


# hidden, rows -> vectors per lane; more than the 40 MB from which stage 2 reads rows past the caches
RECV_PAST_CASES = {(1032, 20500): 1, (2048, 10300): 1, (2056, 10300): 2, (7168, 3000): 2, (7168, 21200): 1}


@pytest.mark.parametrize("hidden_dim,rows", RECV_PAST_CASES)
@pytest.mark.parametrize("layout", ["padded", "compact"])
@pytest.mark.parametrize("plan", [True, False])
def test_stage_2_of_large_streams(hidden_dim, rows, layout, plan):
    print(f"stage 2, {rows} rows of {hidden_dim}, {layout}, plan {plan}", flush=True)
    W, nle = 2, 3
    a = HIPAllToAll(MoEConfig(W * nle, 1, hidden_dim, rows, torch.bfloat16, torch.bfloat16), 1, W, device=DEV, reuse_placement=plan,
                    layout=layout, compact_rows=rows + 5 if layout == "compact" else None)
    a.long_stream_rows = 0
    gen = torch.Generator(device=DEV)
    gen.manual_seed(rows)
    recv = torch.randint(-30000, 30000, (rows + 9, hidden_dim), device=DEV, generator=gen, dtype=torch.int16).view(torch.bfloat16)
    meta = torch.randint(0, 1000, (rows + 9, 5), device=DEV, generator=gen, dtype=torch.int32)
    meta[:, 0] = nle + torch.randint(0, nle, (rows + 9,), device=DEV, generator=gen, dtype=torch.int32)
    counts = torch.tensor([rows - 700, 700], dtype=torch.int32, device=DEV)  # (nine rows more than arrived lie in the buffers)
    num, ex, em = a.dispatch_recv(counts, recv, meta, rows)
    torch.cuda.synchronize()
    le = meta[:rows, 0] - nle
    assert torch.equal(num.long(), torch.bincount(le, minlength=nle))
    first = 0
    for e in range(nle):
        of, n = torch.nonzero(le == e).flatten(), int(num[e])
        got, got_meta = (ex[first:first + n], em[first:first + n]) if layout == "compact" else (ex[e, :n], em[e, :n])
        assert torch.equal(got.view(torch.int16), recv[of].view(torch.int16)) and torch.equal(got_meta, meta[of]), e
        first += n


# hidden, entries per token, tokens -> vectors per lane; rows and results of more than the 80 MB from which stage 4 reads past the caches
MAPPED_PAST_CASES = {(2048, 1, 10300): 2, (7168, 2, 2000): 2, (4104, 3, 2560): 2, (2056, 4, 4100): 2, (512, 4, 16500): 1, (3080, 6, 1950): 1,
                     (1032, 8, 4600): 1}


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("hidden_dim,K,tokens", MAPPED_PAST_CASES)
def test_stage_4_of_large_streams(hidden_dim, K, tokens, dtype):
    """With a table against the kernels that scan, which other files hold to the oracle. A third of the rows names other tokens' entries, and some lie past
    the counts."""
    print(f"stage 4, {tokens} tokens x {K} of {hidden_dim} {dtype}", flush=True)
    a = HIPAllToAll(MoEConfig(16, K, hidden_dim, tokens, dtype, dtype), 0, 2, device=DEV)
    a.long_stream_rows = 0
    gen = torch.Generator(device=DEV)
    gen.manual_seed(tokens)
    S = tokens * K
    order = torch.randperm(S, device=DEV, generator=gen)
    meta = torch.stack([order, order, order // K, order % K, order], 1).int()
    meta[::3, 2] += tokens
    rows = torch.randn(S, hidden_dim, device=DEV, generator=gen).to(dtype)
    weights = torch.rand(tokens, K, device=DEV, generator=gen)
    counts = torch.tensor([S - 900, 800], dtype=torch.int32, device=DEV)
    start = torch.randn(tokens, hidden_dim, device=DEV, generator=gen).to(dtype)
    for accumulate in (True, False):
        got = [start.clone() for _ in range(2)]
        for y, unique in zip(got, (True, False)):
            a.combine_recv(y, weights, counts, rows, meta, accumulate=accumulate, unique_pairs=unique)
        torch.cuda.synchronize()
        assert "entry_row" in a._ws and torch.equal(*[y.view(torch.int16) for y in got]), accumulate
