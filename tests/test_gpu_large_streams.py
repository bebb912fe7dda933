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


@pytest.mark.parametrize("W,E,K,hidden_dim,tokens", [
    (8, 16, 1, 8, 5120),     # the shortest it takes, one entry per token; a vector per row, 20 tokens a workgroup
    (3, 15, 5, 520, 1024),   # 65 vectors, experts per rank no power of two
    (2, 6, 6, 1032, 2561),   # 60 entries in a workgroup, the last of which owns one token
    (8, 8, 7, 64, 2311),     # an expert per rank, nine tokens each
    (4, 256, 64, 16, 81),    # a token per workgroup, with 64 entries
    (5, 20, 3, 3208, 1800),  # 401 vectors: twice as many workgroups
    (2, 4, 2, 8, 32641),     # 65282 entries, more than the kernel before it takes
    (1, 2, 1, 7168, 5121),
])
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
    for megabytes in (0, 25, 300, 400):
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
