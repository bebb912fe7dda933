"""csrc/host_calls.cpp without a GPU: whatever is not a plain tensor on the rank's GPU is refused before anything is
launched, and the class surface does without the extension."""
import copy

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
