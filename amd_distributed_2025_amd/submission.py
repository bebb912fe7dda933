"""`custom_kernel(data)` — the entry point the reference's harness calls
(all2all/submission.py:339-356, all2all/hipv8.py:375-394; contract in
all2all/task.py:8-9): `data = (cfg, rank_data, rank, world_size)` in, the
rank's `[num_tokens, hidden_dim]` result of `cfg.out_dtype` out.

On one GPU the other ranks of the job do not exist as processes. Their inputs
are registered once with `set_peer_inputs` (they are synthesised from the same
seeds the harness would give those ranks); `custom_kernel` then steps the whole
job through `LocalWorld` on the caller's device and returns the caller's rows.
With `world_size == 1` nothing has to be registered.

The ranks share the GPU, so a job is three launches whatever its size
(`moe_a2a_local_dispatch`, `moe_a2a_local_combine`): where every entry's row goes,
every rank's rows to their experts and through the stand-in expert, and the
weighted sums of the ranks asked for. Nothing is read back, staged or kept
between calls; buffers come from torch's allocator, so calls from several
threads and streams do not meet. A job beyond the limits of those entry points
(64 ranks, 1024 experts, 64 entries per token) steps through `LocalWorld`: the
first call of a job (a shape and the token counts of its ranks) launch by launch,
reading the exchanged counts back to size its launches, and from the second call
on as a HIP graph captured once (one per rank asked for) that reads its inputs
from buffers they are copied into. The graph's launches are sized by the counts
of the first call; sizes are a matter of speed only, every kernel moves what the
device-side counts of the call at hand say.
"""
from __future__ import annotations

from typing import Dict, List, Optional, Sequence, Tuple

import torch

from . import _binding, _lib
from .all2all import LOCAL_MAX_EXPERTS, LOCAL_MAX_K, LOCAL_MAX_RANKS, LocalWorld, _need, _raw_stream, _stream
from .task import MoEConfig, RankTestData, input_t, output_t

_peers: Optional[Sequence[input_t]] = None
_worlds: Dict[Tuple, "_World"] = {}
MAX_CAPTURED_JOBS = 18  # graphs kept per job shape (each holds only launches; the buffers are the world's)


def set_peer_inputs(inputs: Optional[Sequence[input_t]]) -> None:
    """Register the inputs of every rank of the job (index = rank). The entry of
    the calling rank is ignored: its data comes with the call."""
    global _peers
    _peers = inputs


class _World:
    """A `LocalWorld` of one job shape with the buffers its captured jobs read their inputs from."""

    def __init__(self, cfg: MoEConfig, world_size: int, device: torch.device):
        self.lw = LocalWorld(cfg, world_size, device=device)
        T, K, H = cfg.max_num_tokens, cfg.experts_per_token, cfg.hidden_dim
        self.x = [torch.empty(T, H, dtype=cfg.in_dtype, device=device) for _ in range(world_size)]
        self.indices = [torch.empty(T, K, dtype=torch.int32, device=device) for _ in range(world_size)]
        self.weights = [torch.empty(T, K, dtype=torch.float32, device=device) for _ in range(world_size)]
        self.seen: Dict[Tuple[int, ...], int] = {}
        self.graphs: Dict[Tuple, Tuple[torch.cuda.CUDAGraph, List[torch.Tensor]]] = {}

    def _staged(self, tokens: Tuple[int, ...]) -> List[RankTestData]:
        """Views of the input buffers cut to the job's token counts, as rank inputs."""
        out = []
        for r, t in enumerate(tokens):
            d = object.__new__(RankTestData)
            d.num_tokens, d.rank = t, r
            d.x, d.indices, d.weights = self.x[r][:t], self.indices[r][:t], self.weights[r][:t]
            out.append(d)
        return out

    def run(self, everyone: Sequence[RankTestData], only: Optional[int] = None) -> List[torch.Tensor]:
        """One step of the job; `only=r` leaves out what only the other ranks' results need (their
        return exchange and weighted sum) and returns None in their places."""
        tokens = tuple(int(d.num_tokens) for d in everyone)
        calls = self.seen.get(tokens, 0)
        self.seen[tokens] = calls + 1
        if calls == 0:  # launch by launch, reading the counts back: they size the later launches
            self.lw.exact_hints = True
            return self.lw.run(everyone, only=only)
        staged = self._staged(tokens)
        torch._foreach_copy_([d.x for d in staged] + [d.indices for d in staged] + [d.weights for d in staged],
                             [d.x for d in everyone] + [d.indices for d in everyone] + [d.weights for d in everyone])
        key = (tokens, only)
        if key not in self.graphs:
            while len(self.graphs) >= MAX_CAPTURED_JOBS:
                self.graphs.pop(next(iter(self.graphs)))
            # the counts sizing the launches are those the latest launch-by-launch run of this world
            # read back; a job of other token counts came in between only if it ran that way too
            self.lw.exact_hints = True
            self.lw.run(staged, only=only)  # (also leaves every workspace buffer allocated before the capture)
            self.lw.exact_hints = "last"
            torch.cuda.synchronize(self.lw.device)
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph):
                ys = self.lw.run(staged, only=only)
            self.graphs[key] = (graph, ys)
        graph, ys = self.graphs[key]
        graph.replay()
        return ys


def _world_for(cfg: MoEConfig, world_size: int, device: torch.device) -> _World:
    key = (cfg.num_experts, cfg.experts_per_token, cfg.hidden_dim, cfg.max_num_tokens,
           cfg.in_dtype, cfg.out_dtype, world_size, str(device))
    w = _worlds.get(key)
    if w is None:
        _worlds.clear()  # one job shape at a time keeps the workspaces bounded
        w = _worlds[key] = _World(cfg, world_size, device)
    return w


def _fits_direct(cfg: MoEConfig, world_size: int) -> bool:
    return (world_size <= LOCAL_MAX_RANKS and cfg.num_experts <= LOCAL_MAX_EXPERTS
            and cfg.experts_per_token <= LOCAL_MAX_K)


def _run_direct(cfg: MoEConfig, world_size: int, everyone: Sequence[RankTestData], device: torch.device,
                only: Optional[int] = None) -> List[torch.Tensor]:
    """One step of the job; `only=r` leaves out the other ranks' weighted sums (and returns rank r's alone)."""
    if cfg.num_experts % world_size:
        raise ValueError("num_experts must be a multiple of world_size")
    K, H = cfg.experts_per_token, cfg.hidden_dim
    xs, ids, weights, tokens = [], [], [], []
    for d in everyone:
        x, i, w = d.x, d.indices, d.weights
        T = i.shape[0]
        if i.shape[1] != K or x.shape != (T, H) or w.shape != (T, K):
            raise ValueError("shapes of x / indices / weights do not match the config")
        xs.append(_need(x, cfg.in_dtype, device, "x"))
        ids.append(_need(i, torch.int32, device, "indices"))
        weights.append(_need(w, torch.float32, device, "weights"))
        tokens.append(T)
    entries = sum(tokens) * K
    stream = _stream(device)
    shape = _lib.Shape(world_size, 0, cfg.num_experts, K, H, cfg.max_num_tokens)
    c = _binding.get("ctypes")
    rows = torch.empty((max(entries, 1), H), dtype=cfg.out_dtype, device=device)
    where = torch.empty((max(entries, 1),), dtype=torch.int32, device=device)
    c.local_dispatch(shape, xs, ids, True, where, None, None, rows, None, True, stream)
    if only is None:
        # (a tensor of its own for each rank: views of one would keep all results as long as any of them; empty_like
        # takes 1.2 us of the host, empty with sizes and a device 1.8)
        ys = [torch.empty_like(x, dtype=cfg.out_dtype) for x in xs]
        c.local_combine(shape, rows, where, weights, tokens, ys, -1, False, stream)
        return ys
    y = torch.empty((tokens[only], H), dtype=cfg.out_dtype, device=device)
    c.local_combine(shape, rows, where, weights, tokens, [y if r == only else None for r in range(world_size)], only,
                    False, stream)
    return [y]


def _native_job(cfg, world_size, inputs, own, rank, every_rank):
    """`_run_direct` in native code (csrc/host_calls.cpp): one rank's result or all of them; None where it refuses."""
    native = _binding.host_calls().get("job") if _raw_stream is not None else None
    return native and native(_raw_stream, cfg, world_size, inputs, own, rank, every_rank)


def _there(d: RankTestData, device: torch.device) -> RankTestData:
    index = device.index
    if d.x.get_device() == index and d.indices.get_device() == index and d.weights.get_device() == index:
        return d
    return d.to(device)


def custom_kernel_job(inputs: Sequence[input_t]) -> list:
    """Every rank's `custom_kernel` result from ONE step of the job: what W processes calling
    `custom_kernel` at the same time produce together. `inputs[r]` is rank r's tuple."""
    cfg, first, _, world_size = inputs[0]
    ys = _native_job(cfg, world_size, inputs, None, 0, True)
    if ys is not None:
        return ys
    device = first.x.device
    if device.type != "cuda":
        raise RuntimeError("custom_kernel needs its inputs on a GPU; this path has no CPU fallback")
    if len(inputs) != world_size:
        raise ValueError(f"a job of world_size={world_size} needs {world_size} inputs, got {len(inputs)}")
    everyone = [_there(d[1], device) for d in inputs]
    with torch.cuda.device(device):
        if _fits_direct(cfg, world_size):
            return _run_direct(cfg, world_size, everyone, device)
        ys = _world_for(cfg, world_size, device).run(everyone)
        return [y.clone() for y in ys]


def custom_kernel(data: input_t) -> output_t:
    cfg, rank_data, rank, world_size = data
    peers = [data] if world_size == 1 else _peers
    if peers is not None:
        y = _native_job(cfg, world_size, peers, rank_data, rank, False)
        if y is not None:
            return y
    device = rank_data.x.device
    if device.type != "cuda":
        raise RuntimeError("custom_kernel needs its inputs on a GPU; this path has no CPU fallback")
    if world_size == 1:
        everyone = [rank_data]
    else:
        if _peers is None or len(_peers) != world_size:
            raise RuntimeError(
                f"world_size={world_size}: register the job's per-rank inputs with set_peer_inputs() first"
            )
        everyone = [rank_data if r == rank else _there(_peers[r][1], device) for r in range(world_size)]
    with torch.cuda.device(device):
        if _fits_direct(cfg, world_size):
            return _run_direct(cfg, world_size, everyone, device, only=rank)[0]
        ys = _world_for(cfg, world_size, device).run(everyone, only=rank)
        return ys[rank].clone()
