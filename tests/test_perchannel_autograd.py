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
