"""Jobs whose streams are short: the kernels that hold every key of a stream in one wave (stages 1, 2 and 4, and jobs on one GPU), at the numbers of
entries where another number of keys per lane or another kernel takes over, against the oracle bit for bit."""
import numpy as np
import pytest
import torch

from amd_distributed_2025_amd import HIPAllToAll, LocalWorld, MoEConfig, custom_kernel_job, generate_world
from oracle import moe_a2a_oracle as orc
from tests.helpers import bits, run_oracle
from tests.test_gpu_local import config, rank_data
from tests.test_gpu_parity import run_and_compare

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def job(world_size, num_experts, topk, hidden, tokens, routing="uniform", dtype="bf16", seed=5):
    return generate_world(dict(world_size=world_size, num_experts=num_experts, experts_per_token=topk, hidden_dim=hidden,
                               max_num_tokens=tokens, num_tokens="full", routing=routing, weights="softmax", dtype=dtype), seed)


@pytest.mark.parametrize("entries", [1, 64, 127, 128, 129, 256, 257, 512, 513, 768, 769, 1024, 1025])
def test_numbers_of_entries(entries):
    """One entry per token, two ranks: as many rows leave as there are tokens and about as many arrive."""
    print(f"entries {entries}", flush=True)
    run_and_compare(job(2, 6, 1, 72, entries))


@pytest.mark.parametrize("hidden", [64, 2048, 2056, 4104, 37])
@pytest.mark.parametrize("world_size,num_experts,topk,tokens", [(4, 24, 5, 100), (8, 64, 8, 32), (4, 8, 3, 170), (2, 64, 64, 4)])
@pytest.mark.parametrize("routing", ["uniform", "zipf"])
def test_shapes(world_size, num_experts, topk, tokens, hidden, routing):
    print(f"shape {world_size} {num_experts} {topk} {tokens} {hidden} {routing}", flush=True)
    world = job(world_size, num_experts, topk, hidden, tokens, routing, "fp16" if hidden == 2048 else "bf16")
    _, want = run_and_compare(world)
    lw = LocalWorld(world[0][0], world_size, device=DEV, layout="compact")
    ys = lw.run([d.to(DEV) for _, d, _, _ in world])
    torch.cuda.synchronize()
    for r, t in enumerate(want):
        n = int(t.expert_num_tokens.sum())
        assert np.array_equal(bits(lw.trace[r]["expert_x"][:n]), t.expert_rows), r
        assert np.array_equal(lw.trace[r]["expert_meta"][:n].cpu().numpy(), t.expert_meta_rows), r
        assert np.array_equal(bits(ys[r]), t.y), r


@pytest.mark.parametrize("hint", [1, 60, 250, 256, 300, 512, 600])
@pytest.mark.parametrize("layout", ["padded", "compact"])
def test_a_stream_longer_than_the_hint(layout, hint):
    """The hint picks the kernel; the rows behind it are moved all the same."""
    print(f"hint {hint} {layout}", flush=True)
    world = job(4, 32, 6, 24, 95, "zipf")
    want = run_oracle(world)
    lw = LocalWorld(world[0][0], 4, device=DEV, layout=layout)
    counts_of = lw._exchange_hints
    lw._exchange_hints = lambda phase, sent: [[max(1, hint // 4) for _ in row] for row in counts_of(phase, sent)]
    ys = lw.run([d.to(DEV) for _, d, _, _ in world])
    torch.cuda.synchronize()
    for r, t in enumerate(want):
        assert np.array_equal(lw.trace[r]["expert_num_tokens"].cpu().numpy(), t.expert_num_tokens), r
        assert np.array_equal(bits(lw.trace[r]["back_buf"][: int(t.expert_num_tokens.sum())]), t.back_buf), r
        assert np.array_equal(bits(ys[r]), t.y), r


@pytest.mark.parametrize("arrive", [3, 64, 65, 250])
@pytest.mark.parametrize("accumulate", [True, False])
def test_rows_of_one_token(arrive, accumulate):
    """More rows of one token than the list of a wave holds (64) are added up in arrival order too."""
    print(f"rows of one token {arrive} {accumulate}", flush=True)
    T, K, H = 4, 3, 200
    rng = np.random.default_rng(arrive)
    cfg = MoEConfig(8, K, H, 128, torch.bfloat16, torch.bfloat16)
    a = HIPAllToAll(cfg, 0, 2, device=DEV)
    meta = np.zeros((arrive + 5, 5), np.int32)
    meta[:, 2], meta[:, 3] = np.where(np.arange(arrive + 5) < arrive, 1, 2), rng.integers(-1, K + 1, arrive + 5)
    buf = torch.from_numpy(rng.standard_normal((arrive + 5, H)).astype(np.float32)).bfloat16()
    weights = rng.random((T, K), np.float32)
    y = torch.from_numpy(rng.standard_normal((T, H)).astype(np.float32)).bfloat16()
    counts = torch.tensor([arrive, 5], dtype=torch.int32)
    names = (meta[:, 3] >= 0) & (meta[:, 3] < K)  # (a row whose k names no weight is not added)
    want = orc.combine_recv(bits(buf)[names], meta[names], weights, T, "bf16", y_init=bits(y) if accumulate else None)
    got = a.combine_recv(y.to(DEV), torch.from_numpy(weights).to(DEV), counts.to(DEV), buf.to(DEV),
                         torch.from_numpy(meta).to(DEV), accumulate=accumulate)
    torch.cuda.synchronize()
    assert np.array_equal(bits(got), want)


@pytest.mark.parametrize("tokens", [[256], [257], [1024], [1025], [2048], [0, 255, 1], [0, 100, 0, 157], [300, 0, 724, 0],
                                    [0, 0, 0, 0, 0, 0, 3, 1022], [100, 0, 948, 0, 1000]])
def test_jobs_on_one_gpu(tokens):
    """Entries where another number of keys per lane takes over, and ranks without tokens, one entry per token."""
    print(f"jobs {tokens}", flush=True)
    W = len(tokens)
    cfg = config(3 * W, 1, 40, max(tokens))
    data = [rank_data(cfg, t, 11 * r) for r, t in enumerate(tokens)]
    want = [y.clone() for y in LocalWorld(cfg, W, device=DEV).run(data)]
    ys = custom_kernel_job([(cfg, d, r, W) for r, d in enumerate(data)])
    for r in range(W):
        assert torch.equal(ys[r], want[r]), f"rank {r}"


@pytest.mark.parametrize("world_size", [1, 3])
@pytest.mark.parametrize("hidden", [2064, 4104, 5000, 7168, 1001])
def test_jobs_whose_lanes_move_several_vectors(world_size, hidden):
    """More than 1024 entries and two workgroups per unit: lanes move one, two or four vectors of a row."""
    print(f"several vectors {world_size} {hidden}", flush=True)
    cfg = config(4 * world_size, 2, hidden, 600)
    data = [rank_data(cfg, 540 if world_size == 1 else t, 7 * r) for r, t in enumerate([200, 341, 0][:world_size])]
    want = [y.clone() for y in LocalWorld(cfg, world_size, device=DEV).run(data)]
    ys = custom_kernel_job([(cfg, d, r, world_size) for r, d in enumerate(data)])
    for r in range(world_size):
        assert torch.equal(ys[r], want[r]), f"rank {r}"


# hidden, rows, promised rows, layout -> the kernel of stage 2 and how it stores (csrc/stream_rules.h; test_stream_rules.py
# holds the cases to that)
RECV_CASES = {
    (512, 300, 300, "padded"): "few, plain", (512, 300, 0, "padded"): "few, plain", (512, 300, 0, "compact"): "few, plain",
    (4096, 1023, 1023, "padded"): "few, plain", (4096, 1024, 1024, "padded"): "few, through", (5120, 820, 820, "compact"): "few, through",
    (8192, 512, 512, "padded"): "few, through", (8192, 700, 600, "compact"): "few, through", (6144, 700, 700, "padded"): "few, through",
    (7168, 580, 580, "padded"): "few, plain", (7168, 600, 600, "padded"): "scan, through", (7168, 1024, 1024, "compact"): "scan, through",
    (7168, 700, 600, "padded"): "scan, through", (7168, 590, 800, "compact"): "scan, through", (8200, 600, 600, "padded"): "few, plain",
    (72, 1025, 1025, "padded"): "scan, through", (2049, 512, 512, "padded"): "few, plain", (2049, 513, 513, "padded"): "scan, plain",
    (264, 4097, 4097, "padded"): "scan, through", (512, 4096, 4096, "compact"): "scan, through", (512, 5003, 5003, "compact"): "scan, through",
    (2049, 513, 513, "compact"): "few, plain", (1001, 1024, 1024, "padded"): "few, plain", (3001, 900, 700, "padded"): "scan, plain"}


@pytest.mark.parametrize("hidden,rows,hint,layout", RECV_CASES)
def test_kernels_of_stage_2(hidden, rows, hint, layout):
    """Placement, counts and meta rows, and with them the order of the way back, which stage 3 takes from stage 2's plan."""
    print(f"stage 2 {hidden} {rows} {hint} {layout}", flush=True)
    W, nle = 3, 5
    rng = np.random.default_rng(hidden + rows)
    a = HIPAllToAll(MoEConfig(W * nle, 1, hidden, rows // W + 1, torch.bfloat16, torch.bfloat16), 1, W, device=DEV, layout=layout)
    source = np.sort(rng.integers(0, W, rows))
    meta = np.stack([nle + rng.integers(0, nle, rows), source, np.arange(rows), np.zeros(rows), np.zeros(rows)], 1).astype(np.int32)
    buf = torch.from_numpy(rng.integers(-30000, 30000, (rows, hidden), dtype=np.int16))
    counts = torch.from_numpy(np.bincount(source, minlength=W).astype(np.int32)).to(DEV)
    num, ex, em = a.dispatch_recv(counts, buf.to(DEV).view(torch.bfloat16), torch.from_numpy(meta).to(DEV), hint)
    back_counts, back, back_meta = a.combine_send(em, ex, num)
    expert = meta[:, 0] - nle
    assert np.array_equal(num.cpu().numpy(), np.bincount(expert, minlength=nle))
    got_x, got_m = ex.cpu().view(torch.int16), em.cpu().numpy()
    at = 0
    for le in range(nle):
        mine = np.flatnonzero(expert == le)
        x, m = (got_x[at:at + len(mine)], got_m[at:at + len(mine)]) if layout == "compact" else (got_x[le, :len(mine)], got_m[le, :len(mine)])
        assert torch.equal(x, buf[torch.from_numpy(mine)]) and np.array_equal(m, meta[mine]), le
        at += len(mine)
    order = np.lexsort((np.arange(rows), expert, source))
    assert torch.equal(back_counts, counts) and np.array_equal(back_meta[:rows].cpu().numpy(), meta[order])
    assert torch.equal(back[:rows].cpu().view(torch.int16), buf[torch.from_numpy(order)])
    # (of other tensors: by a scan)
    back.zero_(), back_meta.zero_()
    back_counts, back, back_meta = a.combine_send(em.clone(), ex.clone(), num.clone())
    assert torch.equal(back_counts, counts) and np.array_equal(back_meta[:rows].cpu().numpy(), meta[order])
    assert torch.equal(back[:rows].cpu().view(torch.int16), buf[torch.from_numpy(order)])


# ranks, tokens of each, entries per token, hidden -> vectors of a row that a lane moves (csrc/stream_rules.h; test_stream_rules.py
# holds the cases to that)
LANES = {(1, 16, 8, 7168): 1, (2, 100, 1, 513): 1, (8, 16, 4, 7168): 1, (3, 60, 2, 7168): 2, (1, 300, 1, 7168): 2, (8, 40, 2, 7168): 4,
         (1, 900, 1, 7168): 4, (2, 20, 3, 7167): 4, (1, 1000, 1, 513): 4, (5, 30, 6, 4100): 4, (8, 26, 1, 7167): 8, (1, 300, 4, 5001): 8,
         (2, 300, 2, 2049): 8}


@pytest.mark.parametrize("world_size,tokens,topk,hidden", LANES)
@pytest.mark.parametrize("dtypes", ["bf16 fp16", "fp16 fp16"])
def test_lanes_that_move_several_vectors_of_short_jobs(world_size, tokens, topk, hidden, dtypes):
    print(f"lanes {world_size} {tokens} {topk} {hidden} {dtypes}", flush=True)
    din, dout = ({"bf16": torch.bfloat16, "fp16": torch.float16}[d] for d in dtypes.split())
    cfg = config(8 * world_size, topk, hidden, tokens, din, dout)
    data = [rank_data(cfg, tokens - r, 5 * r) for r in range(world_size)]
    want = [y.clone() for y in LocalWorld(cfg, world_size, device=DEV).run(data)]
    ys = custom_kernel_job([(cfg, d, r, world_size) for r, d in enumerate(data)])
    for r in range(world_size):
        assert torch.equal(ys[r], want[r]), f"rank {r}"
