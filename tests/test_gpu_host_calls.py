"""The calls of the class surface in native code (csrc/host_calls.cpp) against the Python code that takes every form:
whatever the form of a call, both give the same result or raise the same error."""
import copy

import numpy as np
import pytest
import torch

from amd_distributed_2025_amd import HIPAllToAll, LocalWorld, MoEConfig, RankTestData, custom_kernel, custom_kernel_job, gemm_rs, set_peer_inputs
from amd_distributed_2025_amd import _binding, _lib, all2all
from amd_distributed_2025_amd._lib import MoeA2AError

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
E, K, H, T, W = 8, 2, 64, 12, 4


class Sub(torch.Tensor):
    pass


def config(out=torch.bfloat16):
    return MoEConfig(E, K, H, T, torch.bfloat16, out)


def rank(layout, native, **kw):
    a = HIPAllToAll(config(), 0, 1, device=DEV, layout=layout, **kw)
    make = a._buf

    def zeroed(name, shape, dtype):  # (rows that nobody fills are compared as well)
        new = a._kept.get(name) != (shape, dtype)
        t = make(name, shape, dtype)
        return t.zero_() if new else t

    a._buf = zeroed
    if not native:
        a._calls = all2all._PythonOnly()
    return a


def data(tokens=T, seed=0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    d = object.__new__(RankTestData)
    d.num_tokens, d.rank = tokens, 0
    d.x = torch.randn(tokens, H, generator=g, device=DEV).bfloat16()
    d.indices = torch.rand(tokens, E, generator=g, device=DEV).topk(K, dim=1).indices.int().contiguous()
    d.weights = torch.rand(tokens, K, generator=g, device=DEV)
    return d


def strided(t):
    return torch.stack([t, t], dim=-1)[..., 0]


def unreadable(t):
    """A tensor that raises where its address is asked for, as a lazily cloned one does that cannot be copied."""
    t = t.clone()
    torch._C._set_throw_on_mutable_data_ptr(t)
    return t


# how an argument may come
FORMS = {"unreadable": unreadable, "plain": lambda t: t, "strided": strided, "cpu": lambda t: t.cpu(), "double": lambda t: t.double(), "half": lambda t: t.half(),
         "long": lambda t: t.long(), "subclass": lambda t: t.as_subclass(Sub), "parameter": lambda t: torch.nn.Parameter(t, requires_grad=False),
         "flat": lambda t: t.reshape(-1), "short": lambda t: t[:-1], "wide": lambda t: torch.cat([t, t], dim=-1), "tall": lambda t: torch.cat([t, t]),
         "none": lambda t: None, "list": lambda t: t.tolist(), "empty": lambda t: t[:0], "offset": lambda t: torch.cat([t.reshape(-1)[:1], t.reshape(-1)])[1:].view(t.shape)}
HINTS = [None, 0, 5, T * K, 10 ** 6, np.int64(7), True, 3.0, -1, 2 ** 40, "7"]


def outcome(f):
    """The tensors that a call gives, or the type of what it raises."""
    try:
        got = f()
    except Exception as e:  # noqa: BLE001
        return type(e)
    torch.cuda.synchronize()
    return [t.clone() for t in (got if isinstance(got, (tuple, list)) else [got])]


def same(p, q):
    if isinstance(p, type) or isinstance(q, type):
        return p is q
    return len(p) == len(q) and all(a.dtype == b.dtype and a.shape == b.shape and torch.equal(a, b) for a, b in zip(p, q))


def cleared(a):
    for t in a._ws.values():
        t.zero_()


def halves(a, d, form=FORMS["plain"], at=None, hint=None, accumulate=True):
    """Every half of one rank of a job of one, with the argument number `at` in another form; results of all."""
    n = iter(range(100))

    def arg(t):
        return form(t) if next(n) == at else t

    out = []
    c, b, m = a.dispatch_send(arg(d.x), arg(d.indices))
    S = d.x.shape[0] * K
    out += [c, b, m]
    c, b, m = c.clone(), b.clone(), m.clone()
    num, ex, em = a.dispatch_recv(arg(c), arg(b), arg(m), hint)
    out.append(num)
    ey = a.expert_scale(arg(ex), arg(num), hint)
    bc, bb, bm = a.combine_send(arg(em), arg(ey), arg(num), hint)
    y = torch.ones(T + 1, H, dtype=torch.bfloat16, device=DEV)
    bc2, bb2, bm2 = bc.clone(), bb.clone(), bm.clone()
    got = a.combine_recv(arg(y), arg(d.weights), arg(bc2), arg(bb2), arg(bm2), accumulate=accumulate)
    return out + [ex, em, ey, bc, bb[:S], bm[:S], got, y]


@pytest.mark.parametrize("layout", ["padded", "compact"])
@pytest.mark.parametrize("form", FORMS)
def test_forms_of_the_halves(layout, form):
    print(f"halves {layout} {form}", flush=True)
    d = data()
    for at in range(15):
        pair = [rank(layout, native) for native in (True, False)]
        for a in pair:  # (the second pass in native code, the first has made the buffers known)
            halves(a, d)
            halves(a, d)
            cleared(a)
        torch.cuda.synchronize()
        got = [outcome(lambda a=a: halves(a, d, FORMS[form], at)) for a in pair]
        assert same(*got), (at, got[0] if isinstance(got[0], type) else "results", got[1] if isinstance(got[1], type) else "results")


@pytest.mark.parametrize("layout", ["padded", "compact"])
@pytest.mark.parametrize("accumulate", [True, False, 1, None])
def test_hints_and_accumulation(layout, accumulate):
    d = data(seed=3)
    for hint in HINTS:
        print(f"hints {layout} {accumulate} {hint!r}", flush=True)
        pair = [rank(layout, native) for native in (True, False)]
        for a in pair:
            halves(a, d)
            cleared(a)
        torch.cuda.synchronize()
        assert same(*[outcome(lambda a=a: halves(a, d, hint=hint, accumulate=accumulate)) for a in pair]), hint


def one_rank(a, d, form=FORMS["plain"], at=None, gemm=None):
    n = iter(range(100))

    def arg(t):
        return form(t) if next(n) == at else t

    num, ex, em = a.dispatch(arg(d.x), arg(d.indices))
    if gemm is None:
        ey = a.expert_scale(arg(ex), arg(num))
    else:
        up, down, b = gemm
        ey = a.expert_gemm(a.expert_gemm(arg(ex), arg(num), arg(up), arg(b)), num, down)
    y = torch.ones(T + 1, H, dtype=torch.bfloat16, device=DEV)
    got = a.combine(arg(y), arg(d.weights), arg(em), arg(ey), arg(num))
    return [num, ex, em, ey, got, y]


@pytest.mark.parametrize("layout", ["padded", "compact"])
@pytest.mark.parametrize("inter", [None, 96, H])  # the stand-in, two widths, one width for both layers
@pytest.mark.parametrize("form", FORMS)
def test_forms_of_a_job_of_one_rank(layout, inter, form):
    print(f"one rank {layout} {inter} {form}", flush=True)
    d = data(seed=5)
    g = torch.Generator(device=DEV).manual_seed(9)
    gemm = None if inter is None else tuple(torch.randn(*s, generator=g, device=DEV).bfloat16() for s in ((E, inter, H), (E, H, inter), (E, inter)))
    for at in range(11 if inter else 9):
        pair = [rank(layout, native) for native in (True, False)]
        for a in pair:
            one_rank(a, d, gemm=gemm)
            one_rank(a, d, gemm=gemm)
            cleared(a)
        torch.cuda.synchronize()
        assert same(*[outcome(lambda a=a: one_rank(a, d, FORMS[form], at, gemm)) for a in pair]), at


def test_results_of_many_widths():
    """Every width that the rank object has a buffer for, and both buffers where a layer reads the first of its width."""
    d, a, plain = data(seed=6), rank("padded", True), rank("padded", False)
    g = torch.Generator(device=DEV).manual_seed(2)
    num, ex, _ = plain.dispatch(d.x, d.indices)
    widths = [32 * (i + 1) for i in range(18)]
    weights = [torch.randn(E, n, H, generator=g, device=DEV).bfloat16() for n in widths]
    square = torch.randn(E, H, H, generator=g, device=DEV).bfloat16()
    for w in weights:
        a.expert_gemm(ex, num, w)
    first = a.expert_gemm(ex, num, square)
    a.expert_gemm(first, num, square)
    for w in weights:
        got = a._calls.expert_gemm(ex, num, w, None, T * K)
        assert got is not None and torch.equal(got, plain.expert_gemm(ex, num, w)), w.shape
    second = a._calls.expert_gemm(a._calls.expert_gemm(ex, num, square, None, T * K), num, square, None, T * K)
    assert second is not None and torch.equal(second, plain.expert_gemm(plain.expert_gemm(ex, num, square), num, square))


def test_workspace_that_changes_and_options_set_later():
    """Other token counts, a buffer replaced by one of another shape, options changed between calls."""
    pair = [rank("padded", native, reuse_placement=True) for native in (True, False)]
    for step, tokens in enumerate([T, 1, 7, T, 0, 5]):
        d = data(tokens, step)
        got = []
        for a in pair:
            if step == 2:
                a.reuse_placement = False
            if step == 3:
                a.long_stream_rows = 4  # every stream is a long one
            if step == 4:
                a.long_stream_rows, a.reuse_placement = None, True
            for t in a._ws.values():
                t.zero_()
            got.append([outcome(lambda a=a: halves(a, d)), outcome(lambda a=a: one_rank(a, d))])
            a._buf("expert_y", (3, 5), torch.float32)  # (the next call makes it anew)
        assert all(same(p, q) for p, q in zip(*got)), step
    assert "row_position" in pair[0]._ws and "entry_row" in pair[0]._ws


class Recorder:
    """A binding of the caller's own."""

    def __init__(self, binding):
        self._binding, self.calls = binding, []

    def __getattr__(self, name):
        call = getattr(self._binding, name)
        return lambda *a: (self.calls.append(name), call(*a))[1]


def test_layout_and_binding_set_later():
    """Both are read at every call; a binding of the caller's own is the one that is called."""
    d, pair = data(seed=8), [rank("padded", native) for native in (True, False)]
    for change in (dict(), dict(layout="compact", compact_rows=T * K + 3), dict(compact_rows=T * K), dict(layout="padded"), dict(binding=_binding.get("ext"))):
        for a in pair:
            for name, value in change.items():
                setattr(a, name, value)
            if a is pair[1]:
                a._calls = all2all._PythonOnly()
        for _ in range(2):
            got = [outcome(lambda a=a: halves(a, d)) + outcome(lambda a=a: one_rank(a, d)) for a in pair]
            assert same(*got), change
    own = pair[0].binding = Recorder(_binding.get("ctypes"))
    for _ in range(2):
        own.calls.clear()
        assert same(outcome(lambda: one_rank(pair[0], d)), got[0][-6:])
        assert own.calls == ["local_dispatch", "expert_scale", "local_combine"]


def test_config_and_bounds_set_later():
    """Both are read at every call: the types that the config names, another config, the rows that the buffers have room for."""
    d, pair = data(seed=9), [rank("padded", native) for native in (True, False)]
    bf16, f16 = torch.bfloat16, torch.float16

    def everything(a):
        x, ys = d.x.to(a.cfg.in_dtype), [torch.zeros(T, H, dtype=a.cfg.out_dtype, device=DEV) for _ in range(2)]
        sent = a.dispatch_send(x, d.indices)
        num, ex, em = a.dispatch_recv(*[t.clone() for t in sent])
        ey = a.expert_scale(ex, num)
        back = a.combine_send(em, ey, num)
        a.combine_recv(ys[0], d.weights, *[t.clone() for t in back])
        num, ex, em = a.dispatch(x, d.indices)
        a.combine(ys[1], d.weights, em, a.expert_scale(ex, num), num)
        assert torch.equal(*ys)
        return [*sent, *back, num, ex, em, ey, *ys]

    for types in ((bf16, bf16), (bf16, f16), (f16, bf16), (bf16, bf16)):
        for a in pair:
            a.cfg.in_dtype, a.cfg.out_dtype = types
        for _ in range(2):
            assert same(*[outcome(lambda a=a: everything(a)) for a in pair]), types
    for change in (dict(cfg=config(f16)), dict(max_rows_in=T * K + 8, max_rows_out=T * K + 1), dict(shape=_lib.Shape(1, 0, E, K, H, T))):
        for a in pair:
            for name, value in change.items():
                setattr(a, name, value)
        pair[1]._calls = all2all._PythonOnly()
        for _ in range(2):
            got = [outcome(lambda a=a: everything(a)) for a in pair]
            assert same(*got), change
    assert got[0][4].shape == (T * K + 8, H) and got[0][4].dtype == f16


def test_copies_share_a_workspace():
    """A copy with another layout takes turns with the object it was made of."""
    d = data()
    a = HIPAllToAll(config(), 0, 1, device=DEV)
    a.dispatch_recv(*a.dispatch_send(d.x, d.indices))
    b = copy.copy(a)
    b.layout = "compact"
    b.binding = _binding.get("ext")
    for _ in range(2):
        for of, dims in ((a, 3), (b, 2), (a, 3)):
            num, ex, em = of.dispatch_recv(*of.dispatch_send(d.x, d.indices))
            assert ex.dim() == em.dim() == dims
            fresh = HIPAllToAll(config(), 0, 1, device=DEV, layout=of.layout)
            fnum, fex, fem = fresh.dispatch_recv(*fresh.dispatch_send(d.x, d.indices))
            assert torch.equal(num, fnum)
            for e, n in enumerate(num.tolist()):
                at = slice(int(num[:e].sum()), int(num[:e].sum()) + n)
                assert torch.equal(ex[e, :n], fex[e, :n]) if dims == 3 else torch.equal(ex[at], fex[at])
            y, fy = torch.zeros(T, H, dtype=torch.bfloat16, device=DEV), torch.zeros(T, H, dtype=torch.bfloat16, device=DEV)
            of.combine_recv(y, d.weights, *of.combine_send(em, of.expert_scale(ex, num), num))
            fresh.combine_recv(fy, d.weights, *fresh.combine_send(fem, fresh.expert_scale(fex, fnum), fnum))
            assert torch.equal(y, fy)


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("which", ["x", "indices", "weights"])
def test_forms_of_a_job(form, which, monkeypatch):
    print(f"job {form} {which}", flush=True)
    for out in (torch.bfloat16, torch.float16):
        inputs = [(config(out), data(t, r), r, W) for r, t in enumerate([T, 3, 0, 7])]
        setattr(inputs[1][1], which, FORMS[form](getattr(inputs[1][1], which)))
        for mode in ("all", 0, 1, 3):
            got = []
            for native in (True, False):
                with monkeypatch.context() as m:
                    if not native:
                        m.setattr(_binding, "_host_calls", {})
                    set_peer_inputs(inputs)
                    try:
                        got.append(outcome(lambda: custom_kernel_job(inputs) if mode == "all" else custom_kernel(inputs[mode])))
                    finally:
                        set_peer_inputs(None)
            assert same(*got), (mode, got[0] if isinstance(got[0], type) else "results", got[1] if isinstance(got[1], type) else "results")


def test_jobs_that_do_not_fit_the_direct_path(monkeypatch):
    """Lists and tuples of inputs, too few of them, experts that the ranks do not divide, a world of one."""
    cases = [tuple((config(), data(4, r), r, W) for r in range(W)), [(config(), data(4, r), r, W) for r in range(W - 1)],
             [(MoEConfig(9, K, H, T, torch.bfloat16, torch.bfloat16), data(4, r), r, W) for r in range(W)], [(config(), data(5), 0, 1)]]
    for inputs in cases:
        got = []
        for native in (True, False):
            with monkeypatch.context() as m:
                if not native:
                    m.setattr(_binding, "_host_calls", {})
                got.append(outcome(lambda: custom_kernel_job(inputs)))
        assert same(*got)
    assert isinstance(custom_kernel_job(cases[0]), list)


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("at", [0, 1, 2])
def test_forms_of_the_linear_product(form, at, monkeypatch):
    g = torch.Generator(device=DEV).manual_seed(1)
    args = [torch.randn(*s, generator=g, device=DEV).bfloat16() for s in ((20, 128), (96, 128), (96,))]
    for bias in (True, False):
        call = [*args[:2], args[2] if bias else None]
        if call[at] is not None:
            call[at] = FORMS[form](call[at])
        got = []
        for native in (True, False):
            with monkeypatch.context() as m:
                if not native:
                    m.setattr(_binding, "_host_calls", {})
                got.append(outcome(lambda: gemm_rs.local_product(tuple(call))))
        assert same(*got), (form, at, bias)


def test_native_calls_are_the_ones_that_run():
    """None is what they give when they refuse: plain forms are taken once the buffers are known."""
    d = data()
    a = rank("padded", True)
    assert a._calls.dispatch_send(d.x, d.indices) is None
    halves(a, d)
    one_rank(a, d)
    assert a._calls.dispatch_send(d.x, d.indices) == T
    assert a._calls.direct_dispatch(d.x, d.indices) == T
    a._buf("expert_y", (1,), torch.float32)
    assert a._calls.dispatch_send(d.x, d.indices) is None
    side = torch.cuda.Stream()
    want = outcome(lambda: one_rank(rank("padded", False), d)[-1])
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        got = one_rank(a, d)[-1]
    side.synchronize()
    assert torch.equal(got, want[0])


class Answers:
    """The native calls of a rank object; what each of them answered."""

    def __init__(self, calls):
        self._calls, self.got = calls, {}

    def __getattr__(self, name):
        call = getattr(self._calls, name)

        def seen(*args):
            got = call(*args)
            if not name.startswith("learn_"):
                self.got.setdefault(name, []).append(got is not None)
            return got

        return seen


HALVES = {"dispatch_send", "dispatch_recv", "expert_scale", "combine_send", "combine_recv"}


@pytest.mark.parametrize("layout", ["padded", "compact"])
@pytest.mark.parametrize("reuse", [True, False])
def test_every_call_is_native_from_the_first_pass_on(layout, reuse):
    """A new object launches nothing through its binding for plain calls; from the second pass on no call is refused."""
    d, w = data(seed=4), torch.ones(E, H, H, device=DEV, dtype=torch.bfloat16)
    of_one = {"direct_dispatch", "direct_combine"} if reuse else HALVES - {"expert_scale"}
    for f, names in ((halves, HALVES), (one_rank, of_one | {"expert_scale"}), (lambda a, d: one_rank(a, d, gemm=(w, w, None)), of_one | {"expert_gemm"})):
        a, want = rank(layout, True, reuse_placement=reuse), outcome(lambda: f(rank(layout, False, reuse_placement=reuse), d))
        a._binding = own = Recorder(a._binding)  # (past the setter: the native calls stay)
        assert same(outcome(lambda: f(a, d)), want)
        a._calls = answers = Answers(a._calls)
        assert same(outcome(lambda: f(a, d)), want)
        assert set(own.calls) <= {"gather_sources", "exchange_gather"}  # (the exchange between the halves)
        taken = {name for name, got in answers.got.items() if all(got)}
        assert taken >= names and not any(any(got) for name, got in answers.got.items() if name not in names)


def test_the_linear_product_and_the_job_are_native(monkeypatch):
    answers = {}

    def seen(name, call):
        def f(*args):
            got = call(*args)
            answers.setdefault(name, []).append(got is not None)
            return got

        return f

    monkeypatch.setattr(_binding, "_host_calls", {name: seen(name, call) for name, call in _binding.host_calls().items() if name != "RankCalls"})
    x, w = torch.ones(20, 128, device=DEV).bfloat16(), torch.ones(96, 128, device=DEV).bfloat16()
    for bias in (None, w[:, 0].contiguous()):
        assert gemm_rs.local_product((x, w, bias)).shape == (20, 96)
    inputs = [(config(), data(t, r), r, W) for r, t in enumerate([T, 3, 0, 7])]
    custom_kernel_job(inputs)
    set_peer_inputs(inputs)
    try:
        custom_kernel(inputs[1])
    finally:
        set_peer_inputs(None)
    torch.cuda.synchronize()
    assert answers == {"linear": [True, True], "job": [True, True]}


@pytest.mark.parametrize("layout", ["padded", "compact"])
def test_a_call_that_fails_leaves_no_plan(layout):
    """The buffers are known from then on, and that none of them is a plan."""
    d, a = data(seed=4), rank(layout, True)
    c, b, m = [t.clone() for t in a.dispatch_send(d.x, d.indices)]
    a.dispatch_recv(c, b, m)
    a.reuse_placement = False
    with pytest.raises(MoeA2AError):
        a.dispatch_recv(c, b, m, -1)
    assert a._calls.dispatch_recv(c, b, m, T * K) == T * K
    assert same(outcome(lambda: halves(a, d)), outcome(lambda: halves(rank(layout, False, reuse_placement=False), d)))
    assert a._planned_for is None


def test_wrapped_tensors_are_refused():
    x, w = torch.zeros(3, 8, 64, device=DEV).bfloat16(), torch.zeros(32, 64, device=DEV).bfloat16()
    native = _binding.host_calls()["linear"]
    seen = []
    torch.func.vmap(lambda t: (seen.append(native(all2all._raw_stream, t, w, None)), t)[1])(x)
    neg = torch._neg_view(torch.ones(8, 64, device=DEV, dtype=torch.bfloat16))
    seen.append(native(all2all._raw_stream, neg, w, None))
    assert seen == [None, None]
