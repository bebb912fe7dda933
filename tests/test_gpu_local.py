"""Jobs whose ranks share the GPU: `dispatch` / `combine` of a job of one rank and `custom_kernel` go straight
from tokens to experts' rows and back. Every bit has to be what the halves with an exchange between them give
(which other files check against the oracle)."""
import pytest
import torch

from amd_distributed_2025_amd import HIPAllToAll, LocalWorld, MoEConfig, RankTestData, custom_kernel, custom_kernel_job, set_peer_inputs
from tests.helpers import reach_the_binding

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def rank_data(cfg, T, seed, spoil=None, device=DEV):
    """Distinct experts per token; `spoil`: "ids" puts ids outside [0, E) in, "twins" repeats experts."""
    gen = torch.Generator(device=device)
    gen.manual_seed(seed)
    E, K = cfg.num_experts, cfg.experts_per_token
    d = object.__new__(RankTestData)
    d.num_tokens, d.rank = T, 0
    d.indices = torch.rand(T, E, generator=gen, device=device).argsort(dim=1)[:, :K].int().contiguous()
    if spoil == "ids":
        hit = torch.rand(T, K, generator=gen, device=device) < 0.2
        stray = torch.tensor([-1, E, E + 7, -2 ** 31], dtype=torch.int32, device=device)
        d.indices[hit] = stray[torch.randint(0, 4, (int(hit.sum()),), generator=gen, device=device)]
    elif spoil == "twins":
        d.indices = torch.randint(0, min(E, 2), (T, K), generator=gen, device=device).int()
    d.weights = torch.randn(T, K, generator=gen, device=device).softmax(dim=1)
    d.x = torch.randn(T, cfg.hidden_dim, generator=gen, device=device).to(cfg.in_dtype)
    return d


def config(E, K, H, T, din=torch.bfloat16, dout=torch.bfloat16):
    return MoEConfig(num_experts=E, experts_per_token=K, hidden_dim=H, max_num_tokens=T, in_dtype=din, out_dtype=dout)


@pytest.mark.parametrize("binding", ["ctypes", "ext"])
@pytest.mark.parametrize("layout", ["padded", "compact"])
@pytest.mark.parametrize("E,K,H,T,spoil", [
    (8, 2, 256, 16, None), (1, 1, 8, 1, None), (5, 3, 101, 7, None),       # one launch; element by element
    (64, 8, 2048, 256, None), (64, 8, 64, 257, None),                      # 2048 entries and 8 more: ranked, planned
    (64, 7, 4104, 40, "ids"), (300, 6, 520, 1000, "ids"),                  # ids outside the range, both ways
    (40, 9, 1032, 33, None), (64, 64, 128, 20, "ids"), (64, 33, 72, 90, None),  # more than eight entries per token
    (1024, 4, 96, 700, None), (5, 3, 101, 900, "ids"), (16, 8, 512, 300, "twins"), (4, 4, 264, 64, "twins"),
])
def test_one_rank_matches_the_halves(E, K, H, T, spoil, layout, binding, monkeypatch):
    print(f"one rank E={E} K={K} H={H} T={T} {spoil} {layout} {binding}", flush=True)
    if binding == "ext":  # (with the other one the native calls do the plain forms)
        called = reach_the_binding(monkeypatch, binding)
    cfg = config(E, K, H, T + 3)  # (room for more tokens than come)
    d = rank_data(cfg, T, 17 + K, spoil)
    direct = HIPAllToAll(cfg, 0, 1, device=DEV, layout=layout, binding=binding)
    halves = HIPAllToAll(cfg, 0, 1, device=DEV, layout=layout, binding=binding, reuse_placement=False)
    got = []
    for a in (direct, halves):
        for name, shape, dt in (("expert_x", (a.compact_rows,) if layout == "compact" else (E, a.max_recv), cfg.in_dtype),
                                ("expert_meta", None, torch.int32)):
            shape = (got_shape := shape or ((a.compact_rows,) if layout == "compact" else (E, a.max_recv))) + \
                ((H,) if name == "expert_x" else (5,))
            a._buf(name, shape, dt).fill_(77)  # rows that nothing fills stay as they are
        num, ex, em = a.dispatch(d.x, d.indices)
        ey = a.expert_scale(ex, num)
        y = torch.ones(T + 2, H, dtype=cfg.out_dtype, device=DEV)
        a.combine(y, d.weights, em, ey, num)
        torch.cuda.synchronize()
        got.append((num, ex, em, y, a.expert_offsets))
    assert direct._dispatched_for is not None and halves._dispatched_for is None
    for what, p, q in zip(("counts", "rows", "meta", "result", "offsets"), *got):
        assert (p is None and q is None) or torch.equal(p, q), what
    if binding == "ext":
        halves_too = {"dispatch_send", "combine_recv"} | ({"dispatch_recv", "combine_send"} if layout == "padded" else {"dispatch_recv_compact", "combine_send_compact"})
        assert called >= {"local_dispatch", "local_combine"} | halves_too


def test_combine_of_other_tensors_takes_the_halves():
    cfg = config(8, 2, 64, 20)
    d = rank_data(cfg, 20, 3)
    a = HIPAllToAll(cfg, 0, 1, device=DEV)
    num, ex, em = a.dispatch(d.x, d.indices)
    ey = a.expert_scale(ex, num)
    y = torch.zeros(20, 64, dtype=cfg.out_dtype, device=DEV)
    a.combine(y, d.weights, em, ey, num)
    y2 = torch.zeros_like(y)
    a.combine(y2, d.weights, em.clone(), ey, num.clone())  # (their rows' places are in the meta rows)
    assert torch.equal(y, y2)


@pytest.mark.parametrize("din,dout", [(torch.bfloat16, torch.bfloat16), (torch.float16, torch.bfloat16)], ids=["bf16", "fp16-bf16"])
@pytest.mark.parametrize("W,E,K,H,tokens,spoil", [
    (8, 8, 2, 256, [16] * 8, None), (8, 64, 6, 1032, [5, 1, 128, 77, 128, 3, 64, 9], None),
    (4, 12, 8, 101, [30, 1, 9, 17], None),                      # more entries per token than experts on a rank
    (2, 8, 8, 64, [40, 33], "twins"), (4, 8, 4, 72, [50, 2, 50, 31], "twins"), (2, 2, 4, 64, [20, 20], "twins"),
    (8, 256, 8, 520, [160] * 8, "ids"), (64, 128, 3, 64, [2] * 64, None), (1, 16, 4, 264, [70], "ids"),
    (1, 32, 12, 264, [300], None), (3, 9, 2, 7168, [11, 1, 40], None),
    # ranked by the mover: experts with more entries than room, ids outside the range, up to 2048 entries and just above
    (1, 4, 4, 264, [64], "twins"), (2, 16, 4, 72, [60, 50], "twins"), (8, 64, 8, 520, [32] * 8, "ids"),
    # tables of up to eight ranks up to 2048 workgroups, and behind
    (8, 16, 2, 64, [257] * 8, None), (2, 4, 2, 72, [1024, 1024], "ids"), (3, 9, 1, 101, [900, 249, 1000], None),
    (8, 64, 8, 64, [32] * 7 + [33], None), (7, 63, 9, 96, [32, 1, 60, 7, 33, 64, 30], None),
])
def test_custom_kernel_matches_the_halves(W, E, K, H, tokens, spoil, din, dout):
    print(f"job W={W} E={E} K={K} H={H} {tokens[:4]} {spoil} {din}", flush=True)
    cfg = config(E, K, H, max(tokens), din, dout)
    data = [rank_data(cfg, t, 100 * r + K, spoil) for r, t in enumerate(tokens)]
    want = [y.clone() for y in LocalWorld(cfg, W, device=DEV).run(data)]
    inputs = [(cfg, d, r, W) for r, d in enumerate(data)]
    ys = custom_kernel_job(inputs)
    set_peer_inputs(inputs)
    try:
        for r in sorted({0, W // 2, W - 1}):
            assert torch.equal(custom_kernel(inputs[r]), want[r]), f"rank {r} alone"
    finally:
        set_peer_inputs(None)
    for r in range(W):
        assert torch.equal(ys[r], want[r]), f"rank {r}"


def test_job_in_a_captured_graph_and_on_two_streams():
    """No buffer outlives a call: replays after other jobs, and jobs on another stream, keep their results."""
    cfg = config(32, 4, 512, 64)
    jobs = [[(cfg, rank_data(cfg, 64, 10 * j + r), r, 4) for r in range(4)] for j in range(2)]
    want = [[y.clone() for y in custom_kernel_job(job)] for job in jobs]
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = custom_kernel_job(jobs[0])
    side = torch.cuda.Stream()
    for _ in range(3):
        graph.replay()
        with torch.cuda.stream(side):
            other = custom_kernel_job(jobs[1])
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(captured, want[0]))
        assert all(torch.equal(a, b) for a, b in zip(other, want[1]))
        for y in captured:
            y.fill_(3.0)


@pytest.mark.parametrize("tokens", [[16] * 4, [1, 30, 7, 2]])
def test_results_of_a_job_share_no_storage(tokens):
    """A caller that keeps or saves one rank's result keeps that result alone."""
    cfg = config(16, 2, 264, max(tokens))
    ys = custom_kernel_job([(cfg, rank_data(cfg, t, r), r, 4) for r, t in enumerate(tokens)])
    assert len({y.untyped_storage().data_ptr() for y in ys}) == 4
    assert all(y.untyped_storage().nbytes() == y.numel() * y.element_size() for y in ys)


@pytest.mark.parametrize("W,E,K,tokens,spoil", [
    (5, 35, 3, [201, 7, 1, 350, 130], None), (9, 18, 1, [3, 0, 1, 2, 5, 0, 7, 1, 2], None),  # loads across two and more ranks
    (4, 64, 7, [100, 33, 0, 171], "ids"), (2, 8, 8, [4000, 4191], None), (2, 8, 8, [4096, 4097], None),  # 65528 and 65544 entries
    (2, 8, 8, [4000, 4400], "ids"), (64, 64, 3, [11] * 64, "twins"),
])
def test_planned_jobs(W, E, K, tokens, spoil):
    """Jobs with a plan launch of their own: ranks that begin inside a load of four entries, both counts of an expert
    in one word (up to 65535 entries) and in two."""
    print(f"planned W={W} E={E} K={K} {tokens[:4]} {spoil}", flush=True)
    cfg = config(E, K, 16, max(tokens))
    data = [rank_data(cfg, t, 7 * r + K, spoil) for r, t in enumerate(tokens)]
    want = [y.clone() for y in LocalWorld(cfg, W, device=DEV).run(data)]
    ys = custom_kernel_job([(cfg, d, r, W) for r, d in enumerate(data)])
    for r in range(W):
        assert torch.equal(ys[r], want[r]), f"rank {r}"
