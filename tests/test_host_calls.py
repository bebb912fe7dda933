"""csrc/host_calls.cpp without a GPU: whatever is not a plain tensor on the rank's GPU is refused before anything is
launched, and the class surface does without the extension."""
import copy
import functools

import pytest
import torch

from amd_distributed_2025_amd import MoEConfig, _binding, _lib, all2all

ROWS, INTS = torch.zeros(4, 16, dtype=torch.bfloat16), torch.zeros(4, 2, dtype=torch.int32)
ODD = [ROWS, INTS, None, 3, -1, 2 ** 70, "x", (1, 2), torch.zeros(0), torch.zeros(4, 16, device="meta"), torch.zeros(2, 2).to_sparse()]
CALLS = {"dispatch_send": 2, "dispatch_recv": 4, "expert_scale": 3, "expert_gemm": 5, "combine_send": 5, "combine_recv": 7,
         "direct_dispatch": 2, "direct_combine": 6}


@pytest.fixture()
def calls():
    def stream(device):
        raise AssertionError("nothing is launched")

    c = _binding.host_calls()["RankCalls"]((1, 0, 8, 2, 16, 4), torch.bfloat16, torch.bfloat16, 0, stream)
    meta = torch.zeros(8, 5, dtype=torch.int32)
    num, ex = torch.zeros(8, dtype=torch.int32), torch.zeros(8, 4, 16, dtype=torch.bfloat16)
    assert c.learn_send(num, ROWS, meta) and c.learn_recv(num, ex, meta, None, None, 100) and c.learn_scale(ex)
    assert c.learn_back(num, ROWS, meta, None) and c.learn_direct(num, ex, meta, num, None) and c.learn_gemm(ex, False)
    return c


@pytest.mark.parametrize("name", CALLS)
def test_calls_refuse_what_is_not_on_the_gpu(calls, name):
    call = getattr(calls, name)
    for shift in range(len(ODD)):
        assert call(*[ODD[(i * 3 + shift) % len(ODD)] for i in range(CALLS[name])]) is None
        assert call(*[ODD[shift]] * CALLS[name]) is None
    for n in (0, CALLS[name] - 1, CALLS[name] + 1):
        with pytest.raises(TypeError):
            call(*[ROWS] * n)
    calls.forget()
    assert call(*[ROWS] * CALLS[name]) is None


def test_functions_refuse_too():
    f = _binding.host_calls()
    for odd in ODD:
        assert f["linear"](None, odd, ROWS, None) is None and f["linear"](None, ROWS, odd, odd) is None
        assert f["job"](None, odd, 1, [odd], None, 0, True) is None
        assert f["job"](None, odd, odd, odd, odd, odd, odd) is None
    with pytest.raises(TypeError):
        _binding.host_calls()["RankCalls"]((1, 0, 8), torch.bfloat16, torch.bfloat16, 0, None)


def test_without_the_extension():
    """Every call is refused, so that the Python code does it."""
    none = all2all._PythonOnly()
    assert none.dispatch_send(ROWS, INTS) is None and none.forget() is None and none.learn_send(1, 2, 3) is None


def test_an_extension_of_other_sources_is_left_alone(monkeypatch, tmp_path):
    """The calls are those that the Python code was written with, or none."""
    from amd_distributed_2025_amd import _ext, build

    assert _ext.load().a2a_extension_id() == build.extension_id()
    other = tmp_path / "host_calls.cpp"
    other.write_bytes(build.CALLS_SOURCE.read_bytes() + b"\n")
    monkeypatch.setattr(build, "CALLS_SOURCE", other)
    monkeypatch.setattr(_binding, "_host_calls", None)
    assert _binding.host_calls() == {}
    monkeypatch.setattr(build, "CALLS_SOURCE", tmp_path / "none.cpp")
    monkeypatch.setattr(_binding, "_host_calls", None)
    assert _binding.host_calls() == {}


def test_a_copied_object_and_its_copy_use_no_learned_buffers():
    """They share a workspace: what one of them replaces the other's native calls would go on using."""
    a = object.__new__(all2all.HIPAllToAll)
    a.__dict__.update(_learned={"recv"}, _copied=False, _calls="native calls", _ws={}, _layout="padded")
    b = copy.copy(a)
    b.layout = "compact"
    assert type(a._calls) is type(b._calls) is all2all._PythonOnly and b._ws is a._ws and a.layout == "padded"
    b.binding = object()
    assert type(b._calls) is all2all._PythonOnly


def test_a_config_or_shape_of_other_sizes_gets_no_native_calls():
    """(The Python code checks by the one and launches by the other.)"""
    made = [MoEConfig(8, 2, 16, 4, torch.bfloat16, torch.bfloat16), _lib.Shape(1, 0, 8, 2, 16, 4)]
    binding = object.__new__(_binding.CtypesBinding)
    native, device = _binding.host_calls()["RankCalls"], torch.device("cuda", 0)
    assert type(all2all._rank_calls(made[1], made[0], device, binding)) is native
    assert type(all2all._rank_calls(_lib.Shape(1, 0, 8, 2, 32, 4), made[0], device, binding)) is all2all._PythonOnly
    a = object.__new__(all2all.HIPAllToAll)
    a.__dict__.update(_learned={"recv"}, _copied=False, _calls=None, _binding=binding, _cfg=made[0], _shape=made[1], device=device)
    a.cfg = MoEConfig(8, 2, 32, 4, torch.bfloat16, torch.bfloat16)
    assert type(a._calls) is all2all._PythonOnly and not a._learned
    a.shape = _lib.Shape(1, 0, 8, 2, 32, 4)
    assert type(a._calls) is native and a.cfg.hidden_dim == a.shape.hidden_dim == 32


class Recorded(_binding.CtypesBinding):
    """The binding with nothing behind it: every call is noted."""

    def __init__(self):
        self.called = []

    def _call(self, name, *args):
        self.called.append(name)


SHAPE = _lib.Shape(1, 0, 8, 2, 64, 12)  # (padded buffers of 96 rows, 24 in the compact layout)


def _bf(*shape):
    return torch.zeros(*shape, dtype=torch.bfloat16)


def _int(*shape):
    return torch.zeros(*shape, dtype=torch.int32)


# method -> its arguments (SHAPE goes ahead of them unless they begin with numbers); every tensor among them, in lists too, is
# as small as it may be, but for the row and meta buffers whose rows the binding passes on as a capacity (by place)
SIZED = {
    "dispatch_send": ([_bf(12, 64), _int(12, 2), 12, _bf(24, 64), _int(24, 5), _int(1), _int(24), 0], []),
    "plan_send": ([_int(12, 2), 12, _int(1), _int(2), _int(8), _int(24), _int(24), 0], []),
    "dispatch_recv": ([_bf(24, 64), _int(24, 5), _int(1), 24, _int(8), _bf(8, 12, 64), _int(8, 12, 5), _int(16), 0], [0, 1]),
    "dispatch_recv_compact": ([_bf(24, 64), _int(24, 5), _int(1), 24, _int(8), _int(9), _bf(24, 64), _int(24, 5), _int(16), 0],
                              [0, 1, 6, 7]),
    "expert_scale": ([_bf(8, 12, 64), _int(8), 24, _bf(8, 12, 64), 0], []),
    "expert_scale_compact": ([_bf(24, 64), _int(8), 24, _bf(24, 64), 0], [0, 3]),
    "expert_gemm": ([_bf(8, 12, 64), _int(8), 24, _bf(8, 32, 64), _bf(8, 32), _bf(8, 12, 32), 0], []),
    "expert_gemm_compact": ([_bf(24, 64), _int(8), 24, _bf(8, 32, 64), _bf(8, 32), _bf(24, 32), 0], [0, 5]),
    "combine_send": ([_bf(8, 12, 64), _int(8, 12, 5), _int(8), 24, _bf(24, 64), _int(24, 5), _int(1), _int(16), 0], [4, 5]),
    "combine_send_compact": ([_bf(24, 64), _int(24, 5), _int(8), 24, _bf(24, 64), _int(24, 5), _int(1), _int(16), 0], [0, 1, 4, 5]),
    "combine_recv": ([_bf(24, 64), _int(24, 5), _int(1), 24, torch.zeros(12, 2), 12, _bf(12, 64), True, 0], [0, 1]),
    "linear": ([_bf(12, 64), _bf(32, 64), _bf(32), _bf(12, 32), 0], [0, 1]),
    "exchange_local": ([1, 64, _bf(24, 64), _int(24, 5), _int(1), 0, _bf(24, 64), _int(24, 5), _int(1), 0, 24, 0], [2, 3, 6, 7]),
    "local_dispatch": ([[_bf(12, 64)], [_int(12, 2)], False, _int(24), _int(8), _int(9), _bf(8, 12, 64), _int(8, 12, 5), False, 0], [1]),
    "local_combine": ([_bf(24, 64), _int(24), [torch.zeros(12, 2)], [12], [_bf(12, 64)], -1, False, 0], [0]),
}


@pytest.mark.parametrize("method", SIZED)
def test_tensors_that_hold_less_than_a_call_addresses_are_refused(method):
    args, sets_a_capacity = SIZED[method]
    b = Recorded()
    call = getattr(b, method) if method in ("linear", "exchange_local") else functools.partial(getattr(b, method), SHAPE)
    call(*args)
    assert len(b.called) == 1
    looked_at = 0
    for at, arg in enumerate(args):
        tensor = arg[0] if isinstance(arg, list) else arg
        if at in sets_a_capacity or not isinstance(tensor, torch.Tensor):
            continue
        short = list(args)
        short[at] = [tensor[:-1]] if isinstance(arg, list) else tensor[:-1]
        with pytest.raises(ValueError, match="the call needs"):
            call(*short)
        looked_at += 1
    assert len(b.called) == 1 and looked_at


def test_rows_that_set_a_capacity_are_held_to_it():
    """Compact rows are as many as their buffer has of the layer's width, a weight's columns the input's, and a gather's sources as
    many as its ranks."""
    b = Recorded()
    with pytest.raises(ValueError, match="expert_x"):
        b.expert_gemm_compact(SHAPE, _bf(24, 63), _int(8), 24, _bf(8, 32, 64), None, _bf(24, 32), 0)
    with pytest.raises(ValueError, match="expert_y"):
        b.expert_gemm_compact(SHAPE, _bf(24, 64), _int(8), 24, _bf(8, 32, 64), None, _bf(24, 31), 0)
    with pytest.raises(ValueError, match="weight"):
        b.linear(_bf(12, 64), _bf(32, 63), None, _bf(12, 32), 0)
    with pytest.raises(ValueError, match="rows"):
        b.local_dispatch(SHAPE, [_bf(12, 64)], [_int(12, 2)], True, _int(24), None, None, _bf(24, 63), None, False, 0)
    with pytest.raises(ValueError, match="send_counts"):
        b.gather_sources(64, [_bf(24, 64)] * 2, [_int(24, 5)] * 2, [_int(2), _int(1)])
    sources = b.gather_sources(64, [_bf(24, 64)] * 2, [_int(24, 5)] * 2, [_int(2), _int(2)])
    with pytest.raises(ValueError, match="sources"):
        b.exchange_gather(3, 64, sources, 0, _bf(24, 64), _int(24, 5), _int(3), 24, 0)
    with pytest.raises(ValueError, match="recv_counts"):
        b.exchange_gather(2, 64, sources, 0, _bf(24, 64), _int(24, 5), _int(1), 24, 0)
    assert not b.called
    b.exchange_gather(2, 64, sources, 0, _bf(24, 64), _int(24, 5), _int(2), 24, 0)
    assert b.called == ["moe_a2a_exchange_gather_local"]


@pytest.mark.parametrize("rows, taken", [(24, False), (96, True), (95, False)])
def test_flat_expert_rows_are_held_to_the_padded_layout(rows, taken, monkeypatch):
    """Rows without their dimensions go to the padded entry point, which addresses 96 of them: flat compact ones, 24,
    had it write past the end of a buffer made for 24."""
    monkeypatch.setattr(all2all, "_stream", lambda device: 0)
    a, b = object.__new__(all2all.HIPAllToAll), Recorded()
    a.__dict__.update(_calls=all2all._PythonOnly(), _learned=set(), _ws={}, _kept={}, _send_views={}, _binding=b, _shape=SHAPE,
                      _cfg=MoEConfig(8, 2, 64, 12, torch.bfloat16, torch.bfloat16), _rows_in_hint=24, device=torch.device("cpu"))
    if taken:
        assert a.expert_scale(_bf(rows * 64), _int(8)).shape == (rows * 64,) and b.called == ["moe_a2a_expert_scale"]
    else:
        with pytest.raises(ValueError, match="the call needs"):
            a.expert_scale(_bf(rows * 64), _int(8))
        assert not b.called
