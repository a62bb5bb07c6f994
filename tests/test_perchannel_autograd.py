"""CPU checks of the E1 per-channel functions' autograd formulas with the library
calls left out (their outputs are then whatever memory held): a second derivative
raises for every gradient and every input, with constant incoming gradients too,
and first derivatives come out the same way with and without create_graph."""

import contextlib

import pytest
import torch


class _Nothing:
    def __getattr__(self, name):
        return lambda *a: 0


@pytest.fixture
def stubbed(monkeypatch):
    from qllm2_amd import _lib, pam_perchannel
    monkeypatch.setattr(_lib, "lib", lambda: _Nothing())
    monkeypatch.setattr(_lib, "device", lambda dev: contextlib.nullcontext())
    monkeypatch.setattr(_lib, "stream_ptr", lambda dev=None: None)
    return pam_perchannel


def _leaves(*shapes):
    return [torch.ones(s, requires_grad=True) for s in shapes]


def _chunked(P, misaligned):
    B, H, T, d = 1, 2, 5, 3
    q, k, v, g = _leaves((B, H, T, d, 2), (B, H, T, d, 2), (B, H, T, d, 2), (B, H, T, d))
    if misaligned:  # copies of the inputs reach the function
        qc, kc, vc = (torch.cat([x.reshape(-1)[:1], x.reshape(-1)])[1:].view(x.shape) for x in (q, k, v))
    else:
        qc, kc, vc = q, k, v
    return (q, k, v, g), P._Chunked.apply(P._aligned(qc), P._aligned(kc), P._aligned(vc), g, 4, 0.5)


def _fold(P, _):
    q, k, g = _leaves((1, 2, 5, 3, 2), (1, 2, 5, 3, 2), (1, 2, 5, 3))
    return (q, k, g), P._Fold.apply(q, k, g, 4, 0.5)


def _scan(P, _):
    x, a = _leaves((2, 3, 4, 4, 2), (2, 3, 4))
    return (x, a), P._Scan.apply(x, a)


@pytest.mark.parametrize("make,misaligned", [(_chunked, False), (_chunked, True), (_fold, False), (_scan, False)])
def test_second_derivative_raises(stubbed, make, misaligned):
    leaves, outs = make(stubbed, misaligned)
    gouts = [torch.ones_like(o) for o in outs]
    first = torch.autograd.grad(outs, leaves, gouts, create_graph=True)
    assert all(a.shape == b.shape and a.dtype == b.dtype for a, b in zip(first, leaves))
    for i, g in enumerate(first):
        for x in leaves:
            # beside a term of its own, so that a constant gradient would go unnoticed
            with pytest.raises(RuntimeError, match="no second derivative"):
                torch.autograd.grad((x * x).sum() + (g * g).sum(), x, retain_graph=True)
    plain = torch.autograd.grad(outs, leaves, gouts)
    assert all(g.grad_fn is None and g.shape == x.shape for g, x in zip(plain, leaves))


def _offset(x):
    """x's values in a contiguous view one element past an aligned start."""
    buf = x.new_zeros(x.numel() + 1)
    buf[1:] = x.reshape(-1)
    return buf[1:].view(x.shape)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_incoming_gradients_reach_the_library_aligned(stubbed, monkeypatch, dtype):
    """The kernels read dy and the state's gradient as whole complex elements."""
    from qllm2_amd import _lib
    seen = {}

    class Lib:
        def qpam_pc_fwd(self, a, s):
            return 0

        def qpam_pc_bwd(self, a, s):
            seen.update(dy=a._obj.dy % (2 * dtype.itemsize), dfin=a._obj.dfin % 8)
            return 0

        def qpam_pc_scan(self, a, s):
            seen.update(init=(a._obj.init or 0) % 8, x=a._obj.x % 8)
            return 0

    monkeypatch.setattr(_lib, "lib", lambda: Lib())
    P = stubbed
    q, k, v, g = (x.to(dtype).detach().requires_grad_(True) for x in _leaves(*[(1, 2, 5, 3, 2)] * 3, (1, 2, 5, 3)))
    y, s = P._Chunked.apply(q, k, v, g, 4, 0.5)
    torch.autograd.grad((y, s), (q, k, v, g), (_offset(torch.ones_like(y)), _offset(torch.ones_like(s))))
    x, a = _leaves((2, 3, 4, 4, 2), (2, 3, 4))
    out, fin = P._Scan.apply(x, a)
    torch.autograd.grad((out, fin), (x, a), (_offset(torch.ones_like(out)), _offset(torch.ones_like(fin))))
    assert seen == {"dy": 0, "dfin": 0, "init": 0, "x": 0}


@pytest.mark.parametrize("entry,field", [("qpam_pc_fwd", f) for f in ("q", "k", "v", "x", "y", "s_fin")] +
                         [("qpam_pc_bwd", f) for f in ("x", "s_in", "dy", "dfin", "dq", "dk", "dv")])
@pytest.mark.parametrize("dtype", [0, 1])
def test_library_refuses_split_complex_elements(entry, field, dtype):
    """Refused on the host, before any launch (the addresses are never touched)."""
    from qllm2_amd import _lib
    a = _lib.PcArgs()
    a.dtype = a.v_dtype = a.g_dtype = dtype
    a.B, a.H, a.T, a.d, a.chunk, a.q_scale = 1, 2, 5, 3, 4, 0.5
    for name in ("q", "k", "v"):
        for ax, st in (("sb", 60), ("sh", 30), ("st", 6)):
            setattr(a, f"{name}_{ax}", st)
    a.g_sb, a.g_sh, a.g_st = 30, 15, 3
    names = ("q", "k", "v", "gamma", "y", "x", "atot", "s_fin", "s_in", "dy", "dfin", "dq", "dk", "dv", "dgamma")
    for i, name in enumerate(names):
        setattr(a, name, 4096 * (i + 1) + ((2 if dtype and field not in ("x", "s_fin", "s_in", "dfin") else 4) if name == field else 0))
    with pytest.raises(_lib.QpamError, match="aligned"):
        _lib.check(getattr(_lib.lib(), entry)(a, None), entry)
