"""The two ways the host layer reaches the C ABI of libmoe_a2a.so.

`CtypesBinding` calls the exported functions directly (include/moe_a2a.h);
`ExtBinding` goes through the torch extension of `csrc/moe_a2a_torch.cpp`, the
binding idiom of the reference's submissions (all2all/hipv8.py:230-252). Both
offer the same methods with the same arguments — tensors, sizes and the stream
handle — and both end in the same kernels, so results are identical. Calls in plain
forms do not get here: `host_calls()` has them done in native code, whichever
binding was asked for. Neither binding has
a fallback: a missing library, a nonzero status or a tensor that holds less than the call
addresses raises (`CtypesBinding` looks at every tensor itself, the extension in its wrappers).

Capacities (`capacity_rows` of the C ABI) are taken from the tensors: the rows a
row buffer and its meta buffer were allocated with; the kernels cut what they move to them.
"""
from __future__ import annotations

import ctypes as C
from typing import Optional

import torch

from . import _lib, build

META_DIM = 5
_DT = {torch.float16: _lib.F16, torch.bfloat16: _lib.BF16}


def _ptr(t: Optional[torch.Tensor]):
    """The address as an int (the argument types say that it is a pointer)."""
    return None if t is None else t.data_ptr()


def _pointers(tensors):
    return (C.c_void_p * len(tensors))(*[t.data_ptr() for t in tensors])


def _holds(what: str, t: Optional[torch.Tensor], elements: int) -> None:
    """The kernels address a tensor by the shape of the call: one that holds less must not get there."""
    if t is not None and t.numel() < elements:
        raise ValueError(f"{what}: holds {t.numel()} elements, the call needs {elements}")


def _padded(shape) -> int:
    """Rows of a rank's padded expert buffers."""
    return shape.num_experts // shape.world_size * shape.max_num_tokens * shape.world_size


def _holds_counts(shape, expert_num_tokens) -> None:
    _holds("expert_num_tokens", expert_num_tokens, shape.num_experts // shape.world_size)


def _holds_plan(shape, send_back_plan) -> None:
    _holds("send_back_plan", send_back_plan, 2 * shape.num_experts)


def _holds_tokens(shape, tokens: int, x, indices) -> None:
    _holds("x", x, tokens * shape.hidden_dim)
    _holds("indices", indices, tokens * shape.experts_per_token)


def _holds_layers(shape, weights, bias) -> None:
    """weights [local experts, out_dim, in_dim], bias [local experts, out_dim]"""
    local = shape.num_experts // shape.world_size
    _holds("weights", weights, local * weights.shape[1] * weights.shape[2])
    _holds("bias", bias, local * weights.shape[1])


def _rows(buf: torch.Tensor, meta: torch.Tensor, hidden_dim: int) -> int:
    return min(buf.numel() // max(hidden_dim, 1), meta.numel() // META_DIM)


class CtypesBinding:
    """(A `Shape` is passed as it is: ctypes takes its address for the call. A `byref` object kept on the shape would
    refer back to it, and such cycles are never collected.)"""

    name = "ctypes"

    def __init__(self):
        lib = _lib.load()
        self._functions = {name: getattr(lib, name) for name in _lib.SIGNATURES}

    def _call(self, name, *args):
        status = self._functions[name](*args)
        if status:
            _lib.check(status, name)

    def version(self) -> str:
        return _lib.load().moe_a2a_version().decode()

    def dispatch_send(self, shape, x, indices, num_tokens, send_buf, send_meta, send_counts, send_slot, stream):
        entries = num_tokens * shape.experts_per_token
        _holds_tokens(shape, num_tokens, x, indices)
        _holds("send_buf", send_buf, entries * shape.hidden_dim)
        _holds("send_meta", send_meta, entries * META_DIM)
        _holds("send_counts", send_counts, shape.world_size)
        _holds("send_slot", send_slot, entries)
        self._call("moe_a2a_dispatch_send", shape, _ptr(x), _ptr(indices), num_tokens, _ptr(send_buf),
                  _ptr(send_meta), _ptr(send_counts), _ptr(send_slot), stream)

    def plan_send(self, shape, indices, num_tokens, rank_counts, rank_offsets, expert_counts, dst_slot,
                  src_entry, stream):
        entries = num_tokens * shape.experts_per_token
        _holds("indices", indices, entries)
        _holds("rank_counts", rank_counts, shape.world_size)
        _holds("rank_offsets", rank_offsets, shape.world_size + 1)
        _holds("expert_counts", expert_counts, shape.num_experts)
        _holds("dst_slot", dst_slot, entries)
        _holds("src_entry", src_entry, entries)
        self._call("moe_a2a_plan_send", shape, _ptr(indices), num_tokens, _ptr(rank_counts),
                  _ptr(rank_offsets), _ptr(expert_counts), _ptr(dst_slot), _ptr(src_entry), stream)

    def dispatch_recv(self, shape, recv_buf, recv_meta, recv_counts, rows_hint, expert_num_tokens, expert_x,
                      expert_meta, send_back_plan, stream, row_position=None):
        _holds("recv_counts", recv_counts, shape.world_size)
        _holds_counts(shape, expert_num_tokens)
        _holds("expert_x", expert_x, _padded(shape) * shape.hidden_dim)
        _holds("expert_meta", expert_meta, _padded(shape) * META_DIM)
        _holds_plan(shape, send_back_plan)
        capacity = _rows(recv_buf, recv_meta, shape.hidden_dim)
        args = (shape, _ptr(recv_buf), _ptr(recv_meta), _ptr(recv_counts),
                min(rows_hint, capacity), capacity, _ptr(expert_num_tokens), _ptr(expert_x), _ptr(expert_meta),
                _ptr(send_back_plan))
        if row_position is None:
            self._call("moe_a2a_dispatch_recv", *args, stream)
        else:  # long streams: positions from a planning launch
            if row_position.numel() < capacity:
                raise ValueError("row_position must hold one int per row of the receive buffers")
            self._call("moe_a2a_dispatch_recv_long", *args, _ptr(row_position), stream)

    def combine_send(self, shape, expert_y, expert_meta, expert_num_tokens, rows_hint, send_buf, send_meta,
                     send_counts, send_back_plan, stream):
        _holds("expert_y", expert_y, _padded(shape) * shape.hidden_dim)
        _holds("expert_meta", expert_meta, _padded(shape) * META_DIM)
        _holds_counts(shape, expert_num_tokens)
        _holds("send_counts", send_counts, shape.world_size)
        _holds_plan(shape, send_back_plan)
        capacity = _rows(send_buf, send_meta, shape.hidden_dim)
        self._call("moe_a2a_combine_send", shape, _ptr(expert_y), _ptr(expert_meta),
                  _ptr(expert_num_tokens), min(rows_hint, capacity), capacity, _ptr(send_buf), _ptr(send_meta),
                  _ptr(send_counts), _ptr(send_back_plan), stream)

    def combine_recv(self, shape, recv_buf, recv_meta, recv_counts, rows_hint, weights, num_tokens, out_tokens,
                     accumulate, stream, entry_row=None):
        _holds("recv_counts", recv_counts, shape.world_size)
        _holds("weights", weights, num_tokens * shape.experts_per_token)
        _holds("out_tokens", out_tokens, num_tokens * shape.hidden_dim)
        capacity = _rows(recv_buf, recv_meta, shape.hidden_dim)
        args = (shape, _ptr(recv_buf), _ptr(recv_meta), _ptr(recv_counts),
                min(rows_hint, capacity), capacity, _ptr(weights), num_tokens, _ptr(out_tokens),
                int(bool(accumulate)), _DT[out_tokens.dtype])
        if entry_row is None:
            self._call("moe_a2a_combine_recv", *args, stream)
        else:  # long streams: rows looked up in a (token, k) -> row table
            if entry_row.numel() < num_tokens * shape.experts_per_token:
                raise ValueError("entry_row must hold num_tokens * experts_per_token ints")
            self._call("moe_a2a_combine_recv_long", *args, _ptr(entry_row), stream)

    def expert_scale(self, shape, expert_x, expert_num_tokens, rows_hint, expert_y, stream):
        _holds("expert_x", expert_x, _padded(shape) * shape.hidden_dim)
        _holds("expert_y", expert_y, _padded(shape) * shape.hidden_dim)
        _holds_counts(shape, expert_num_tokens)
        self._call("moe_a2a_expert_scale", shape, _ptr(expert_x), _ptr(expert_num_tokens), rows_hint,
                  _DT[expert_x.dtype], _DT[expert_y.dtype], _ptr(expert_y), stream)

    def expert_gemm(self, shape, expert_x, expert_num_tokens, rows_hint, weights, bias, expert_y, stream):
        _holds("expert_x", expert_x, _padded(shape) * weights.shape[2])
        _holds("expert_y", expert_y, _padded(shape) * weights.shape[1])
        _holds_counts(shape, expert_num_tokens)
        _holds_layers(shape, weights, bias)
        self._call("moe_a2a_expert_gemm", shape, _ptr(expert_x), _ptr(expert_num_tokens), rows_hint,
                  _ptr(weights), _ptr(bias), weights.shape[2], weights.shape[1], _DT[expert_x.dtype],
                  _ptr(expert_y), stream)

    def linear(self, input, weight, bias, output, stream):
        m, k = input.shape
        n = weight.shape[0]
        _holds("weight", weight, n * k)
        _holds("bias", bias, n)
        _holds("output", output, m * n)
        self._call("moe_a2a_linear", _ptr(input), _ptr(weight), _ptr(bias), m, n, k, _DT[input.dtype],
                  _ptr(output), stream)

    def exchange_local(self, world_size, hidden_dim, send_buf, send_meta, send_counts, dst_rank, recv_buf,
                       recv_meta, recv_counts, src_rank, rows_hint, stream):
        _holds("send_counts", send_counts, world_size)
        _holds("recv_counts", recv_counts, world_size)
        self._call("moe_a2a_exchange_local", world_size, hidden_dim, _ptr(send_buf), _ptr(send_meta),
                  _ptr(send_counts), dst_rank, _ptr(recv_buf), _ptr(recv_meta), _ptr(recv_counts), src_rank,
                  rows_hint, _rows(send_buf, send_meta, hidden_dim), _rows(recv_buf, recv_meta, hidden_dim),
                  stream)

    # ---- the compact expert-major layout (rows of the experts back to back)

    def dispatch_recv_compact(self, shape, recv_buf, recv_meta, recv_counts, rows_hint, expert_num_tokens,
                              expert_offsets, expert_x, expert_meta, send_back_plan, stream, row_position=None):
        _holds("recv_counts", recv_counts, shape.world_size)
        _holds_counts(shape, expert_num_tokens)
        _holds("expert_offsets", expert_offsets, shape.num_experts // shape.world_size + 1)
        _holds_plan(shape, send_back_plan)
        capacity = _rows(recv_buf, recv_meta, shape.hidden_dim)
        args = (shape, _ptr(recv_buf), _ptr(recv_meta), _ptr(recv_counts), min(rows_hint, capacity), capacity,
                _ptr(expert_num_tokens), _ptr(expert_offsets), _ptr(expert_x), _ptr(expert_meta),
                _rows(expert_x, expert_meta, shape.hidden_dim), _ptr(send_back_plan))
        if row_position is None:
            self._call("moe_a2a_dispatch_recv_compact", *args, stream)
        else:  # long streams: places from a planning launch
            if row_position.numel() < capacity:
                raise ValueError("row_position must hold one int per row of the receive buffers")
            self._call("moe_a2a_dispatch_recv_compact_long", *args, _ptr(row_position), stream)

    def expert_scale_compact(self, shape, expert_x, expert_num_tokens, rows_hint, expert_y, stream):
        capacity = min(expert_x.shape[0], expert_y.shape[0])
        _holds("expert_x", expert_x, capacity * shape.hidden_dim)
        _holds("expert_y", expert_y, capacity * shape.hidden_dim)
        _holds_counts(shape, expert_num_tokens)
        self._call("moe_a2a_expert_scale_compact", shape, _ptr(expert_x), _ptr(expert_num_tokens),
                  rows_hint, capacity, _DT[expert_x.dtype], _DT[expert_y.dtype],
                  _ptr(expert_y), stream)

    def expert_gemm_compact(self, shape, expert_x, expert_num_tokens, rows_hint, weights, bias, expert_y, stream):
        capacity = min(expert_x.shape[0], expert_y.shape[0])
        _holds("expert_x", expert_x, capacity * weights.shape[2])
        _holds("expert_y", expert_y, capacity * weights.shape[1])
        _holds_counts(shape, expert_num_tokens)
        _holds_layers(shape, weights, bias)
        self._call("moe_a2a_expert_gemm_compact", shape, _ptr(expert_x), _ptr(expert_num_tokens),
                  rows_hint, capacity, _ptr(weights), _ptr(bias),
                  weights.shape[2], weights.shape[1], _DT[expert_x.dtype], _ptr(expert_y), stream)

    def combine_send_compact(self, shape, expert_y, expert_meta, expert_num_tokens, rows_hint, send_buf,
                             send_meta, send_counts, send_back_plan, stream):
        _holds_counts(shape, expert_num_tokens)
        _holds("send_counts", send_counts, shape.world_size)
        _holds_plan(shape, send_back_plan)
        capacity = _rows(send_buf, send_meta, shape.hidden_dim)
        self._call("moe_a2a_combine_send_compact", shape, _ptr(expert_y), _ptr(expert_meta),
                  _ptr(expert_num_tokens), min(rows_hint, capacity),
                  _rows(expert_y, expert_meta, shape.hidden_dim), capacity, _ptr(send_buf), _ptr(send_meta),
                  _ptr(send_counts), _ptr(send_back_plan), stream)

    def gather_sources(self, hidden_dim, send_bufs, send_metas, send_counts):
        """The per-source pointer tables of `exchange_gather`, built once for buffers that stay where
        they are (a workspace): (tables, rows every send buffer holds, the tensors kept alive)."""
        for counts in send_counts:
            _holds("send_counts", counts, len(send_bufs))
        table = C.c_void_p * len(send_bufs)
        return ((table(*[t.data_ptr() for t in send_bufs]), table(*[t.data_ptr() for t in send_metas]),
                 table(*[t.data_ptr() for t in send_counts])),
                min(_rows(b, m, hidden_dim) for b, m in zip(send_bufs, send_metas)),
                (list(send_bufs), list(send_metas), list(send_counts)))

    def local_dispatch(self, shape, xs, indices, compact, entry_row, expert_num_tokens, expert_offsets, rows, meta,
                       standin, stream):
        of_ranks = [i.shape[0] for i in indices]
        for x, ids, n in zip(xs, indices, of_ranks):
            _holds_tokens(shape, n, x, ids)
        _holds("entry_row", entry_row, sum(of_ranks) * shape.experts_per_token)
        _holds("expert_num_tokens", expert_num_tokens, shape.num_experts)
        _holds("expert_offsets", expert_offsets, shape.num_experts + 1)
        places = rows.shape[0] if compact else shape.num_experts * shape.max_num_tokens * shape.world_size
        _holds("rows", rows, places * shape.hidden_dim)
        _holds("meta", meta, places * META_DIM)
        tokens = (C.c_int32 * len(xs))(*of_ranks)
        din, dout = (_DT[xs[0].dtype], _DT[rows.dtype]) if standin else (-1, -1)
        self._call("moe_a2a_local_dispatch", shape, _pointers(xs), _pointers(indices), tokens,
                   rows.shape[0] if compact else 0, din, dout, _ptr(entry_row), _ptr(expert_num_tokens),
                   _ptr(expert_offsets), rows.data_ptr(), _ptr(meta), stream)

    def local_combine(self, shape, rows, entry_row, weights, tokens, outs, only_rank, accumulate, stream):
        """`weights` and `outs` may hold None for ranks other than `only_rank`; `tokens` are all ranks'."""
        ranks = len(tokens)
        _holds("entry_row", entry_row, sum(tokens) * shape.experts_per_token)
        for w, out, n in zip(weights, outs, tokens):
            _holds("weights", w, n * shape.experts_per_token)
            _holds("out_tokens", out, n * shape.hidden_dim)
        self._call("moe_a2a_local_combine", shape, rows.data_ptr(), entry_row.data_ptr(),
                   (C.c_void_p * ranks)(*map(_ptr, weights)), (C.c_int32 * ranks)(*tokens),
                   (C.c_void_p * ranks)(*map(_ptr, outs)), only_rank, int(bool(accumulate)), _DT[rows.dtype], stream)

    def exchange_gather(self, world_size, hidden_dim, sources, dst_rank, recv_buf, recv_meta, recv_counts,
                        rows_hint, stream):
        (bufs, metas, counts), send_capacity, kept = sources
        if len(kept[0]) < world_size:
            raise ValueError(f"sources: of {len(kept[0])} ranks, the call needs {world_size}")
        _holds("recv_counts", recv_counts, world_size)
        self._call("moe_a2a_exchange_gather_local", world_size, hidden_dim, bufs, metas, counts, dst_rank,
                  _ptr(recv_buf), _ptr(recv_meta), _ptr(recv_counts), rows_hint, send_capacity,
                  _rows(recv_buf, recv_meta, hidden_dim), stream)


class ExtBinding:
    name = "ext"

    def __init__(self):
        from . import _ext

        self._m = _ext.load()

    @staticmethod
    def _shape(shape) -> list:
        try:
            return shape.fields
        except AttributeError:
            shape.fields = [getattr(shape, f) for f, _ in _lib.Shape._fields_]
            return shape.fields

    def version(self) -> str:
        return self._m.a2a_version()

    def dispatch_send(self, shape, x, indices, num_tokens, send_buf, send_meta, send_counts, send_slot, stream):
        self._m.a2a_dispatch_send(self._shape(shape), x, indices, num_tokens, send_buf, send_meta, send_counts,
                                  send_slot, stream)

    def plan_send(self, shape, indices, num_tokens, rank_counts, rank_offsets, expert_counts, dst_slot,
                  src_entry, stream):
        self._m.a2a_plan_send(self._shape(shape), indices, num_tokens, rank_counts, rank_offsets, expert_counts,
                              dst_slot, src_entry, stream)

    def dispatch_recv(self, shape, recv_buf, recv_meta, recv_counts, rows_hint, expert_num_tokens, expert_x,
                      expert_meta, send_back_plan, stream, row_position=None):
        self._m.a2a_dispatch_recv(self._shape(shape), recv_buf, recv_meta, recv_counts, rows_hint,
                                  expert_num_tokens, expert_x, expert_meta, send_back_plan, row_position, stream)

    def combine_send(self, shape, expert_y, expert_meta, expert_num_tokens, rows_hint, send_buf, send_meta,
                     send_counts, send_back_plan, stream):
        self._m.a2a_combine_send(self._shape(shape), expert_y, expert_meta, expert_num_tokens, rows_hint,
                                 send_buf, send_meta, send_counts, send_back_plan, stream)

    def combine_recv(self, shape, recv_buf, recv_meta, recv_counts, rows_hint, weights, num_tokens, out_tokens,
                     accumulate, stream, entry_row=None):
        self._m.a2a_combine_recv(self._shape(shape), recv_buf, recv_meta, recv_counts, rows_hint, weights,
                                 num_tokens, out_tokens, bool(accumulate), entry_row, stream)

    def expert_scale(self, shape, expert_x, expert_num_tokens, rows_hint, expert_y, stream):
        self._m.a2a_expert_scale(self._shape(shape), expert_x, expert_num_tokens, rows_hint, expert_y, stream)

    def expert_gemm(self, shape, expert_x, expert_num_tokens, rows_hint, weights, bias, expert_y, stream):
        self._m.a2a_expert_gemm(self._shape(shape), expert_x, expert_num_tokens, rows_hint, weights, bias,
                                expert_y, stream)

    def linear(self, input, weight, bias, output, stream):
        self._m.a2a_linear(input, weight, bias, output, stream)

    def exchange_local(self, world_size, hidden_dim, send_buf, send_meta, send_counts, dst_rank, recv_buf,
                       recv_meta, recv_counts, src_rank, rows_hint, stream):
        self._m.a2a_exchange_local(world_size, hidden_dim, send_buf, send_meta, send_counts, dst_rank, recv_buf,
                                   recv_meta, recv_counts, src_rank, rows_hint, stream)

    def dispatch_recv_compact(self, shape, recv_buf, recv_meta, recv_counts, rows_hint, expert_num_tokens,
                              expert_offsets, expert_x, expert_meta, send_back_plan, stream, row_position=None):
        args = (self._shape(shape), recv_buf, recv_meta, recv_counts, rows_hint, expert_num_tokens, expert_offsets,
                expert_x, expert_meta, send_back_plan)
        if row_position is None:
            self._m.a2a_dispatch_recv_compact(*args, stream)
        else:
            self._m.a2a_dispatch_recv_compact_long(*args, row_position, stream)

    def expert_scale_compact(self, shape, expert_x, expert_num_tokens, rows_hint, expert_y, stream):
        self._m.a2a_expert_scale_compact(self._shape(shape), expert_x, expert_num_tokens, rows_hint, expert_y,
                                         stream)

    def expert_gemm_compact(self, shape, expert_x, expert_num_tokens, rows_hint, weights, bias, expert_y, stream):
        self._m.a2a_expert_gemm_compact(self._shape(shape), expert_x, expert_num_tokens, rows_hint, weights, bias,
                                        expert_y, stream)

    def combine_send_compact(self, shape, expert_y, expert_meta, expert_num_tokens, rows_hint, send_buf,
                             send_meta, send_counts, send_back_plan, stream):
        self._m.a2a_combine_send_compact(self._shape(shape), expert_y, expert_meta, expert_num_tokens, rows_hint,
                                         send_buf, send_meta, send_counts, send_back_plan, stream)

    def local_dispatch(self, shape, xs, indices, compact, entry_row, expert_num_tokens, expert_offsets, rows, meta,
                       standin, stream):
        self._m.a2a_local_dispatch(self._shape(shape), xs, indices, compact, entry_row, expert_num_tokens,
                                   expert_offsets, rows, meta, standin, stream)

    def local_combine(self, shape, rows, entry_row, weights, tokens, outs, only_rank, accumulate, stream):
        if only_rank >= 0:
            raise ValueError("one rank's result of several goes through the ctypes binding")
        self._m.a2a_local_combine(self._shape(shape), rows, entry_row, weights, outs, bool(accumulate), stream)

    def gather_sources(self, hidden_dim, send_bufs, send_metas, send_counts):
        return (list(send_bufs), list(send_metas), list(send_counts))

    def exchange_gather(self, world_size, hidden_dim, sources, dst_rank, recv_buf, recv_meta, recv_counts,
                        rows_hint, stream):
        bufs, metas, counts = sources
        self._m.a2a_exchange_gather_local(world_size, hidden_dim, bufs, metas, counts, dst_rank, recv_buf,
                                          recv_meta, recv_counts, rows_hint, stream)


KINDS = (CtypesBinding, ExtBinding)
_BINDINGS = {}
_host_calls: Optional[dict] = None


def host_calls() -> dict:
    """What `csrc/host_calls.cpp` offers: `RankCalls`, `linear`, `job`. Empty where the extension has not been built
    for this library or was built from other sources than those that are here: the Python code above the bindings then
    does every call by itself."""
    global _host_calls
    if _host_calls is None:
        try:
            from . import _ext

            ext = _ext.load()
            _host_calls = ext.a2a_host_calls() if ext.a2a_extension_id() == build.extension_id() else {}
        except (_lib.MoeA2AError, ImportError, AttributeError, OSError):  # (OSError: the sources are not here)
            _host_calls = {}
    return _host_calls


def get(name: str):
    """`"ctypes"` or `"ext"`; bindings are created once."""
    b = _BINDINGS.get(name)
    if b is None:
        if name == "ctypes":
            b = CtypesBinding()
        elif name == "ext":
            b = ExtBinding()
        else:
            raise ValueError(f"unknown binding {name!r} (ctypes or ext)")
        _BINDINGS[name] = b
    return b
