"""The work that users of this framework have it do, as cases that can be timed.

Four kinds of call, all through the package's public surface:

  rank    one rank's share of an expert-parallel job: `dispatch_send`, `dispatch_recv`, the stand-in
          expert, `combine_send`, `combine_recv` of `HIPAllToAll`, one process per GPU as in a real job.
          The exchanges between the halves belong to the user's fabric: the rows that they deliver are
          in hand. A job of one rank runs `dispatch()`, the expert and `combine()`, the reference's own
          surface, and there the exchange with itself is part of the call.
  layer   the same one-rank call with a real expert: two `expert_gemm` layers (hidden -> inter -> hidden)
          where the job above has its stand-in. This is an MoE layer of a model on one GPU.
  job     `custom_kernel` / `custom_kernel_job`: every rank of a job stepped on this GPU, what the
          reference's harness calls.
  linear  `gemm_rs.local_product`: one rank's product of a tensor-parallel linear layer.

Inputs are made on the GPU from the seed: N(0, 1) rows, softmax weights, distinct experts per token,
uniform or skewed (Zipf, exponent 1.2); the values of the products are those of their task.
"""
from __future__ import annotations

import math

import torch

from amd_distributed_2025_amd import (HIPAllToAll, LocalWorld, MoEConfig, RankTestData, custom_kernel,
                                      custom_kernel_job, set_peer_inputs)
from amd_distributed_2025_amd import gemm_rs

DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}
META_BYTES = 20
ZIPF_S = 1.2
# The largest listed cases bound the drawn ones.
MAX_ROW_ELEMENTS = 4096 * 8 * 7168      # rows sent per rank times their length
MAX_JOB_ELEMENTS = 256 * 8 * 7168       # the same for a job whose ranks share the GPU
MAX_FLOPS = 2 * 8192 * 8192 * 3696
MAX_WEIGHT_BYTES = 2 << 30
MAX_WORLD_BYTES = 24 << 30              # workspaces of all ranks of a job while its inputs are made


def _rank(name, **kw):
    return dict(name=name, kind="rank", layout="padded", binding="ctypes", routing="uniform", inter=0, bias=False, **kw)


def listed():
    return [
        # a single GPU, a handful of short rows: nothing but launches and host time
        _rank("rank_one_gpu_tiny", world=1, experts=8, topk=2, hidden=256, tokens=16, dtype="bf16"),
        # a decode step of an expert-parallel job, ragged token count, through the torch extension
        dict(_rank("rank_decode_ragged", world=8, experts=128, topk=4, hidden=2880, tokens=125, dtype="fp16"),
             binding="ext"),
        # the headline shape: 256 experts over 8 GPUs, 256 tokens per GPU
        _rank("rank_headline", world=8, experts=256, topk=8, hidden=7168, tokens=256, dtype="bf16"),
        # the same under skewed routing, experts' rows back to back to save memory
        dict(_rank("rank_skewed_compact", world=8, experts=256, topk=8, hidden=7168, tokens=256, dtype="bf16"),
             routing="zipf", layout="compact"),
        # a prefill: thousands of tokens per GPU
        _rank("rank_prefill", world=2, experts=64, topk=8, hidden=7168, tokens=4096, dtype="bf16"),
        # the reference's harness: its smallest benchmark shape, all ranks, and its largest, one rank's result
        dict(name="job_smallest", kind="job", world=8, experts=8, topk=2, hidden=6144, tokens=16, dtype="fp16",
             routing="uniform", every_rank=True),
        dict(name="job_largest", kind="job", world=8, experts=256, topk=8, hidden=7168, tokens=256, dtype="fp16",
             routing="uniform", every_rank=False),
        # an MoE layer on one GPU: a decode step, bound by the experts' weights
        dict(_rank("layer_decode", world=1, experts=64, topk=6, hidden=2048, tokens=24, dtype="fp16"),
             kind="layer", inter=1024, layout="compact"),
        # and a prefill with biases, bound by the matrix cores
        dict(_rank("layer_prefill", world=1, experts=32, topk=4, hidden=4096, tokens=2048, dtype="bf16"),
             kind="layer", inter=2048, bias=True),
        # one rank's products of the gemm-rs task: few rows, short inner dimension with bias, the largest
        dict(name="linear_few_rows", kind="linear", m=64, n=7168, k=2304, bias=False, dtype="bf16"),
        dict(name="linear_short_k", kind="linear", m=2048, n=2880, k=360, bias=True, dtype="bf16"),
        dict(name="linear_largest", kind="linear", m=8192, n=8192, k=3696, bias=False, dtype="bf16"),
    ]


# ------------------------------------------------------------------------------ drawn cases


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _hidden(rng, lo, hi, step):
    """A row length: multiples of 64 mostly, of `step` now and then."""
    h = _log(rng, lo, hi)
    s = 64 if rng.random() < 0.7 else step
    return max(s, h // s * s)


def _draw_rank(rng):
    world = rng.choice([1, 2, 4, 8, 8])
    experts = world * _log(rng, 1, 32)
    topk = rng.randint(1, min(8, experts))
    hidden = _hidden(rng, 256, 7168, 8 if rng.random() < 0.8 else 1)
    most = min(4096, MAX_ROW_ELEMENTS // (topk * hidden),
               MAX_WORLD_BYTES // (4 * hidden * world * (experts + world * min(topk, experts // world))))
    return dict(kind="rank", world=world, experts=experts, topk=topk, hidden=hidden, tokens=_log(rng, 1, max(1, most)),
                dtype=rng.choice(["bf16", "fp16"]), routing=rng.choice(["uniform", "uniform", "zipf"]),
                layout=rng.choice(["padded", "padded", "compact"]), binding=rng.choice(["ctypes", "ext"]),
                inter=0, bias=False)


def _draw_layer(rng):
    experts = _log(rng, 4, 64)
    topk = rng.randint(1, min(8, experts))
    hidden, inter = _hidden(rng, 512, 7168, 32), _hidden(rng, 512, 7168, 32)
    while 4 * experts * hidden * inter > MAX_WEIGHT_BYTES:
        experts, topk = experts // 2, min(topk, max(1, experts // 2))
    most = min(4096, MAX_FLOPS // (4 * topk * hidden * inter),
               MAX_WORLD_BYTES // (2 * experts * (2 * hidden + inter)))
    return dict(kind="layer", world=1, experts=experts, topk=topk, hidden=hidden, tokens=_log(rng, 1, max(1, most)),
                dtype=rng.choice(["bf16", "fp16"]), routing=rng.choice(["uniform", "uniform", "zipf"]),
                layout=rng.choice(["padded", "compact"]), binding=rng.choice(["ctypes", "ext"]),
                inter=inter, bias=rng.random() < 0.5)


def _draw_job(rng):
    experts = 8 * _log(rng, 1, 32)
    topk = rng.randint(2, min(8, experts))
    hidden = _hidden(rng, 2048, 7168, 8)
    return dict(kind="job", world=8, experts=experts, topk=topk, hidden=hidden,
                tokens=_log(rng, 4, min(256, MAX_JOB_ELEMENTS // (topk * hidden))),
                dtype=rng.choice(["fp16", "bf16"]), routing=rng.choice(["uniform", "uniform", "zipf"]),
                every_rank=rng.random() < 0.5)


def _draw_linear(rng):
    n, k = _hidden(rng, 1024, 8192, 32), _hidden(rng, 256, 8192, 8)
    m = _log(rng, 1, max(1, min(8192, MAX_FLOPS // (2 * n * k))))
    return dict(kind="linear", m=m, n=n, k=k, bias=rng.random() < 0.5, dtype=rng.choice(["bf16", "bf16", "fp16"]))


def draw(rng):
    return rng.choice([_draw_rank, _draw_rank, _draw_layer, _draw_job, _draw_linear])(rng)


# ------------------------------------------------------------------------------ inputs


def _device():
    return torch.device("cuda", torch.cuda.current_device())


def _config(case):
    dt = DTYPES[case["dtype"]]
    return MoEConfig(num_experts=case["experts"], experts_per_token=case["topk"], hidden_dim=case["hidden"],
                     max_num_tokens=case["tokens"], in_dtype=dt, out_dtype=dt)


def _inputs(case, cfg, seed):
    """`(cfg, rank_data, rank, world_size)` of every rank of the job."""
    dev = _device()
    gen = torch.Generator(device=dev)
    gen.manual_seed(seed)
    T, E, K, H, W = case["tokens"], case["experts"], case["topk"], case["hidden"], case["world"]
    popularity = torch.zeros(E, device=dev)
    if case["routing"] == "zipf":  # expert popularity ~ 1 / rank^s over a permutation that all ranks share
        popularity[torch.randperm(E, generator=gen, device=dev)] = -ZIPF_S * torch.arange(1, E + 1, device=dev).log()
    world = []
    for r in range(W):
        # the K largest of popularity + Gumbel noise: K distinct experts drawn by those probabilities
        gumbel = -torch.log(-torch.log(torch.rand(T, E, device=dev, generator=gen).clamp_(1e-20, 1 - 1e-7)))
        d = object.__new__(RankTestData)
        d.num_tokens, d.rank = T, r
        d.indices = (popularity + gumbel).topk(K, dim=1).indices.int().contiguous()
        d.weights = torch.randn(T, K, device=dev, generator=gen).softmax(dim=1)
        d.x = torch.randn(T, H, device=dev, generator=gen).to(cfg.in_dtype)
        world.append((cfg, d, r, W))
    return world


def _options(case, cfg):
    """Layout and binding of the rank object. In the compact layout a rank keeps room for twice what
    balanced routing delivers, for all it can receive under skewed routing."""
    opts = dict(layout=case["layout"], binding=case["binding"])
    if case["layout"] == "compact" and case["routing"] != "zipf":
        nle = case["experts"] // case["world"]
        opts["compact_rows"] = min(2 * case["tokens"] * case["topk"] + 64,
                                   case["tokens"] * case["world"] * min(case["topk"], nle))
    return opts


def _prepare_rank(case, seed):
    cfg = _config(case)
    world = _inputs(case, cfg, seed)
    data = world[0][1]
    st = {"case": case, "data": data, "cfg": cfg, "y": torch.zeros_like(data.x)}
    if case["world"] == 1:
        a = HIPAllToAll(cfg, 0, 1, device=_device(), **_options(case, cfg))
        if case["kind"] == "layer":
            E, H, I = case["experts"], case["hidden"], case["inter"]
            gen = torch.Generator(device=_device())
            gen.manual_seed(seed + 1)

            def normal(*shape, scale):
                return torch.randn(*shape, device=_device(), dtype=cfg.in_dtype, generator=gen).mul_(scale)

            st["up"], st["down"] = normal(E, I, H, scale=H ** -0.5), normal(E, H, I, scale=I ** -0.5)
            st["up_bias"] = normal(E, I, scale=0.1) if case["bias"] else None
            st["down_bias"] = normal(E, H, scale=0.1) if case["bias"] else None
        num, ex, em = a.dispatch(data.x, data.indices)
        st["rows"] = case["tokens"] * case["topk"]
    else:
        # the whole job once: rank 0's receive buffers then hold what its peers sent
        lw = LocalWorld(cfg, case["world"], device=_device(), **_options(case, cfg))
        lw.run([w[1] for w in world])
        a, t = lw.ranks[0], lw.trace[0]
        st["arrived"] = (t["recv_counts"], t["recv_buf"], t["recv_meta"])
        st["returned"] = (t["ret_counts"], t["ret_buf"], t["ret_meta"])
        st["rows"] = int(t["recv_counts"].sum())
        ex, em = t["expert_x"], t["expert_meta"]
        for buf in a.outbound_buffers("combine"):
            buf.zero_()
    # rows of the workspace that no token fills are never written: zero ones can be compared
    ex.zero_()
    em.zero_()
    st["a"] = a
    return st


def _run_rank(st):
    """The halves of rank 0 in a job of several ranks, with the rows the fabric delivered in hand. The
    exchange tells every process how many rows arrive, so their number is known on the host."""
    a, d, rows = st["a"], st["data"], st["rows"]
    send_counts, send_buf, send_meta = a.dispatch_send(d.x, d.indices)
    num, ex, em = a.dispatch_recv(*st["arrived"], rows)
    ey = a.expert_scale(ex, num, rows)
    back_counts, back_buf, back_meta = a.combine_send(em, ey, num, rows)
    y = a.combine_recv(st["y"], d.weights, *st["returned"], accumulate=False)
    return {"send": (send_counts, send_buf, send_meta), "experts": (num, ex, em),
            "back": (back_counts, back_buf, back_meta), "y": y}


def _run_one_rank(st):
    """A job of one rank through `dispatch` and `combine`, which adds into the zeroed result as the
    reference's caller has it."""
    a, d = st["a"], st["data"]
    num, ex, em = a.dispatch(d.x, d.indices)
    if st["case"]["kind"] == "layer":
        hidden = a.expert_gemm(ex, num, st["up"], st["up_bias"])
        ey = a.expert_gemm(hidden, num, st["down"], st["down_bias"])
    else:
        ey = a.expert_scale(ex, num)
    y = st["y"].zero_()
    a.combine(y, d.weights, em, ey, num)
    return {"experts": (num, ex, em), "y": y}


def prepare(case, seed):
    if case["kind"] in ("rank", "layer"):
        return _prepare_rank(case, seed)
    if case["kind"] == "job":
        return {"case": case, "inputs": _inputs(case, _config(case), seed)}
    inp, weight, bias = gemm_rs.generate_input(0, 1, case["m"], case["n"], case["k"], case["bias"], seed, device=_device())
    dt = DTYPES[case["dtype"]]
    return {"case": case, "data": (inp.to(dt), weight.to(dt), None if bias is None else bias.to(dt))}


def run(st):
    case = st["case"]
    if case["kind"] == "linear":
        return gemm_rs.local_product(st["data"])
    if case["kind"] == "job":
        if case["every_rank"]:
            return custom_kernel_job(st["inputs"])
        set_peer_inputs(st["inputs"])
        return custom_kernel(st["inputs"][0])
    return _run_one_rank(st) if case["world"] == 1 else _run_rank(st)


# ------------------------------------------------------------------------------ costs


def work(case):
    if case["kind"] == "linear":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": 2 * (m * k + n * k + m * n + (n if case["bias"] else 0)), "flops": 2 * m * n * k}
    T, E, K, H, W = case["tokens"], case["experts"], case["topk"], case["hidden"], case["world"]
    S, row = T * K, 2 * case["hidden"]
    tokens = T * row + 8 * S  # rows in, expert ids and weights
    if case["kind"] == "job":
        ranks_out = W if case["every_rank"] else 1
        return {"bytes": W * tokens + ranks_out * T * row, "flops": 2 * S * H * ranks_out}
    if W > 1:  # each half reads its inputs and writes its outputs; the expert reads and writes every row
        halves = (S + 5 * S) * (row + META_BYTES) + 2 * S * row  # (as many rows arrive as leave)
        return {"bytes": tokens + T * row + halves, "flops": 3 * S * H}
    if case["kind"] == "rank":  # rows to the experts' buffers, through the expert, and back to their tokens
        return {"bytes": tokens + T * row + S * (row + 2 * META_BYTES) + 3 * S * row, "flops": 3 * S * H}
    inter = case["inter"]
    hit = E * (1 - (1 - K / E) ** T)  # experts that get a row, for uniform routing
    weights = hit * 2 * (2 * H * inter + ((H + inter) if case["bias"] else 0))
    rows = S * (row + 2 * META_BYTES) + S * row + 2 * S * 2 * inter + 2 * S * row
    return {"bytes": tokens + T * row + weights + rows, "flops": 4 * S * H * inter + 2 * S * H}


def tolerance(case):
    """Moving rows, the stand-in and the weighted sum are defined to the bit (every addend is rounded in
    arrival order). A product may sum in another order: one rounding to 16 bits differs, two or three in
    a row of layers."""
    if case["kind"] in ("rank", "job"):
        return "exact"
    ulp = {"bf16": 2.0 ** -8, "fp16": 2.0 ** -11}[case["dtype"]]
    if case["kind"] == "linear":
        return {"rel": ulp, "max": 4 * ulp}
    return {"rel": 2 * ulp, "max": 20 * ulp}
