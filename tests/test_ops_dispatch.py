"""CPU checks of the operator registration (qllm2_amd/_ops.py) beside
torch.library.custom_op with the same function, fake kernel and autograd
formula: values, gradients (all, some and none needed), outputs without a
gradient, saved-tensor hooks, no-grad and inference mode, fake tensors, make_fx
and torch.compile give the same; what custom_op refuses (double backward, vmap,
batched gradients, forward mode, functorch's grad) stays refused."""

from typing import List, Optional

import pytest
import torch
from torch import Tensor

from qllm2_amd import _ops


def _fwd(a: Tensor, b: Optional[Tensor], s: float) -> List[Tensor]:
    """[a s + b, a^2]"""
    y = a * s
    return [y + b if b is not None else y, a * a]


def _bwd(a: Tensor, s: float, g0: Optional[Tensor], g1: Optional[Tensor], k: int = 1) -> List[Tensor]:
    z = torch.zeros_like(a)
    return [(g0 * s if g0 is not None else z) + (2 * a * g1 if g1 is not None else z), g0 + 0 if g0 is not None else z]


def _one(a: Tensor, s: float) -> Tensor:
    return a * s


def _single(a: Tensor) -> Tensor:
    return a * 2


def _fake(a, b, s):
    return [torch.empty_like(a), torch.empty_like(a)]


def _wire(make):
    f, bw, one = make("t_fwd", _fwd), make("t_bwd", _bwd), make("t_one", _one)
    f.register_fake(_fake)
    bw.register_fake(lambda a, s, g0, g1, k=1: [torch.empty_like(a), torch.empty_like(a)])
    one.register_fake(lambda a, s: torch.empty_like(a))

    def setup(ctx, inputs, output):
        a, b, s = inputs
        ctx.save_for_backward(a, output[1])
        ctx.s, ctx.has_b = s, b is not None
        ctx.set_materialize_grads(False)

    def back(ctx, grads):
        a, sq = ctx.saved_tensors
        assert sq.shape == a.shape
        da, db = bw(a, ctx.s, grads[0], grads[1])
        return da, (db if ctx.has_b else None), None

    f.register_autograd(back, setup_context=setup)
    single = make("t_single", _single)
    single.register_fake(lambda a: torch.empty_like(a))
    single.register_autograd(lambda ctx, g: g * 2, setup_context=lambda ctx, inputs, output: None)
    a = torch.ones(2, requires_grad=True)
    assert torch.equal(torch.autograd.grad(single(a).sum(), a)[0], torch.full((2,), 2.0))
    one.register_autograd(lambda ctx, g: (g * ctx.s, None), setup_context=lambda ctx, inputs, output: setattr(ctx, "s", inputs[1]))
    return f, bw, one


OURS = _wire(lambda n, fn: _ops.op("qpam::" + n)(fn))
THEIRS = _wire(lambda n, fn: torch.library.custom_op("qpam_ref::" + n, mutates_args=())(fn))


def _leaves():
    g = torch.Generator().manual_seed(3)
    return [torch.randn(4, 3, generator=g, requires_grad=True) for _ in range(2)]


@pytest.mark.parametrize("need_a,need_b,outs", [(1, 1, (0, 1)), (1, 0, (0,)), (0, 1, (0,)), (1, 1, (1,)), (1, 0, (1,))])
def test_values_and_gradients(need_a, need_b, outs):
    res = []
    for f, _, one in (OURS, THEIRS):
        a, b = _leaves()
        a.requires_grad_(bool(need_a)), b.requires_grad_(bool(need_b))
        y = f(a, b, 1.5)
        assert [t.requires_grad for t in y] == [True, True]
        need = [t for t in (a, b) if t.requires_grad]
        gs = torch.autograd.grad([y[i] for i in outs], need, [torch.full((4, 3), 2.0 + i) for i in outs], allow_unused=True)
        res.append([*y, *gs, one(a, 3.0)])
    for x, z in zip(*res):
        assert (x is None) == (z is None) and (x is None or torch.equal(x, z))


def test_modes_without_gradients():
    for f, _, one in (OURS, THEIRS):
        a, b = _leaves()
        with torch.no_grad():
            y = f(a, None, 2.0)
        assert not y[0].requires_grad and torch.equal(y[0], a.detach() * 2)
        with torch.inference_mode():
            assert f(a, b, 2.0)[0].is_inference() and one(a, 2.0).is_inference()
        assert not f(a.detach(), None, 2.0)[0].requires_grad


def test_saved_tensor_hooks_see_the_saved_tensors():
    seen = []
    for f, _, _ in (OURS, THEIRS):
        packed = []
        a, b = _leaves()
        with torch.autograd.graph.saved_tensors_hooks(lambda t: (packed.append(t.shape), t)[1], lambda t: t):
            y = f(a, b, 1.5)
        y[0].sum().backward()
        seen.append((packed, a.grad))
    assert seen[0][0] == seen[1][0] and torch.equal(seen[0][1], seen[1][1])


def test_tracing():
    from torch._subclasses.fake_tensor import FakeTensorMode
    from torch.fx.experimental.proxy_tensor import make_fx
    for f, _, _ in (OURS, THEIRS):
        with FakeTensorMode() as m:
            a = m.from_tensor(_leaves()[0].detach())
            assert f(a, None, 1.0)[1].shape == (4, 3)
        a, b = (t.detach() for t in _leaves())
        gm = make_fx(lambda x, z: f(x, z, 1.5)[0])(a, b)
        assert any("t_fwd" in str(n.target) for n in gm.graph.nodes)
        assert torch.equal(gm(a, b), f(a, b, 1.5)[0])
        x, z = _leaves()
        fn = torch.compile(lambda p, q: (f(p, q, 1.5)[0] * 2).sum(), backend="aot_eager", fullgraph=True)
        fn(x, z).backward()
        assert torch.equal(x.grad, torch.full((4, 3), 3.0)) and torch.equal(z.grad, torch.full((4, 3), 2.0))
    torch.library.opcheck(torch.ops.qpam.t_fwd.default, (*_leaves(), 1.5))


def _double(f, bw, one):
    a, b = _leaves()
    (g,) = torch.autograd.grad(f(a, b, 1.5)[1].sum(), [a], create_graph=True)
    g.sum().backward()


def _batched(f, bw, one):
    a, b = _leaves()
    y = f(a, b, 1.5)
    torch.autograd.grad([y[0]], [a], [torch.ones(5, 4, 3)], is_grads_batched=True)


def _forward_mode(f, bw, one):
    import torch.autograd.forward_ad as fwAD
    a, b = (t.detach() for t in _leaves())
    with fwAD.dual_level():
        y = f(fwAD.make_dual(a, torch.ones_like(a)), b, 1.5)
        assert fwAD.unpack_dual(y[0]).tangent is None      # no silent tangent either


REFUSED = {
    "double backward": _double,
    "vmap": lambda f, bw, one: torch.func.vmap(lambda x: f(x, None, 1.5)[0])(_leaves()[0].detach()),
    "batched gradients": _batched,
    "functorch grad": lambda f, bw, one: torch.func.grad(lambda x: f(x, None, 1.5)[0].sum())(_leaves()[0].detach()),
    "forward mode": _forward_mode,
}


@pytest.mark.parametrize("what", list(REFUSED))
def test_refusals_match(what):
    out = []
    for ops in (THEIRS, OURS):
        try:
            out.append(REFUSED[what](*ops))
        except Exception as e:  # noqa: BLE001  (whatever it is: both have to refuse)
            out.append(type(e))
    raised = [isinstance(x, type) for x in out]
    assert raised[0] == raised[1], out
    if not raised[0] and out[0] is not None:
        assert torch.equal(out[0], out[1])


def _scaled(a: Tensor, s: float = 2.0, k: int = 1) -> Tensor:
    return a * (s * k)


def _make(prefix, fn, name):
    if prefix == "qpam":
        return _ops.op(f"qpam::{name}")(fn)
    return torch.library.custom_op(f"{prefix}::{name}", mutates_args=())(fn)


@pytest.mark.parametrize("prefix", ["qpam", "qpam_ref"])
def test_defaults_reach_the_formula(prefix):
    """Arguments left (or equal) to their defaults, which the dispatcher drops."""
    f = _make(prefix, _scaled, "t_scaled")
    seen = []

    def setup(ctx, inputs, output):
        a, s, k = inputs
        ctx.f = s * k
        seen.append((s, k))

    def back(ctx, g):
        assert ctx.needs_input_grad[0] and not any(ctx.needs_input_grad[1:]) and len(ctx.needs_input_grad) <= 3
        return g * ctx.f, None, None

    f.register_autograd(back, setup_context=setup)
    for args, kw, want in (((), {}, 2.0), ((3.0,), {}, 3.0), ((), {"k": 5}, 10.0), ((2.0, 1), {}, 2.0)):
        a = torch.ones(2, requires_grad=True)
        y = f(a, *args, **kw)
        for _ in range(2):   # the second over the same context
            assert torch.equal(torch.autograd.grad(y.sum(), a, retain_graph=True)[0], torch.full((2,), want))
    assert seen == [(2.0, 1), (3.0, 1), (2.0, 5), (2.0, 1)]


def _same(a: Tensor) -> Tensor:
    return a


def _beside(a: Tensor) -> List[Tensor]:
    return [a * 1, a]


@pytest.mark.parametrize("prefix", ["qpam", "qpam_ref"])
@pytest.mark.parametrize("fn", [_same, _beside])
@pytest.mark.parametrize("grad", [False, True])
def test_outputs_that_are_inputs_are_refused(prefix, fn, grad):
    f = _make(prefix, fn, f"t{fn.__name__}_{grad}")
    with pytest.raises(RuntimeError):
        f(torch.ones(3, requires_grad=grad))


def _keyword(a: Tensor, *, s: float) -> Tensor:
    return a * s


def test_keyword_only_arguments_are_refused():
    with pytest.raises(ValueError, match="keyword-only"):
        _ops.op("qpam::t_keyword")(_keyword)


def test_custom_op_where_a_private_name_is_missing(monkeypatch):
    monkeypatch.setattr(_ops, "_NAMES", _ops._NAMES + ("no_such_name",))
    f, bw, one = _wire(lambda n, fn: _ops.op(f"qpam::other_{n}")(fn))
    assert not any(isinstance(x, _ops.Op) for x in (f, bw, one))
    a, b = _leaves()
    y = f(a, b, 1.5)
    want = OURS[0](a, b, 1.5)
    assert all(torch.equal(x, z) for x, z in zip(y, want))
    got = torch.autograd.grad(y, (a, b), [torch.ones_like(x) for x in y])
    assert all(torch.equal(x, z) for x, z in zip(got, torch.autograd.grad(want, (a, b), [torch.ones_like(x) for x in want])))
