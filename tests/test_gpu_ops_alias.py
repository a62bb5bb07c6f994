"""No output of a registered operator shares memory with an input of it, over the
training calls that reach each operator, forward and backward, with and without
padding and in both dtypes."""

import re
from pathlib import Path

import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

pytestmark = pytest.mark.gpu

SRC = Path(__file__).resolve().parent.parent / "qllm2_amd"


class _Watch(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.seen, self.bad = set(), []

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        out = func(*args, **(kwargs or {}))
        if func.namespace == "qpam":
            name = func._schema.name.split("::")[1]
            self.seen.add(name)
            ins = {a.untyped_storage().data_ptr() for a in args if isinstance(a, torch.Tensor) and a.numel()}
            outs = out if isinstance(out, (list, tuple)) else [out]
            if any(o.numel() and o.untyped_storage().data_ptr() in ins for o in outs):
                self.bad.append(name)
        return out


def _train(outs, leaves):
    outs = [o for o in outs if o is not None and o.requires_grad]
    torch.autograd.grad(outs, leaves, [torch.ones_like(o) for o in outs], allow_unused=True)


def _calls():
    from qllm2_amd import fused_ce, pam_delta, pam_prologue, pam_scan, triton_kernels
    rn = lambda *s, dtype=torch.float32: torch.randn(*s, device="cuda", dtype=dtype).requires_grad_(True)  # noqa: E731
    B, H, T = 1, 2, 70
    for d, dtype in ((64, torch.float32), (64, torch.bfloat16), (48, torch.float32)):
        q, k, v = (rn(B, H, T, d, 2, dtype=dtype) for _ in range(3))
        gamma = torch.rand(1, B, H, T, device="cuda").requires_grad_(True)
        beta = torch.rand(B, H, T, device="cuda").requires_grad_(True)
        _train(pam_scan.pam_scan_interleaved(q, k, v, gamma, d, 64), [q, k, v, gamma])
        pl = [x[..., i].detach().contiguous().requires_grad_(True) for x in (q, k, v) for i in (0, 1)]
        _train(pam_scan.pam_scan_planar(*pl, gamma, q_scale=0.1, chunk=64), [*pl, gamma])
        _train(pam_delta.forward_delta(q, k, v, gamma[0], beta, d), [q, k, v, gamma, beta])
        _train(pam_delta.delta_planar(*pl, gamma[0], beta, q_scale=0.1), [*pl, gamma, beta])
        proj = rn(B, T, pam_prologue.proj_columns(H, d), dtype=dtype) if d in pam_prologue.HEAD_DIMS else None
        if proj is not None:
            bias = rn(H)
            out = pam_prologue.pam_prologue(proj, bias, n_heads=H, head_dim=d)
            _train([x for o in out[:3] for x in o] + [out[3]], [proj, bias])
        z, up = rn(40, d, 2, dtype=dtype), rn(40, d, 2, dtype=dtype)
        p = [rn(d) for _ in range(3)]
        _train([pam_prologue.cabs(z)], [z])
        _train([triton_kernels.fused_cgu_gate(triton_kernels.fused_complex_norm(z, p[0]),
                                              triton_kernels.fused_mod_swish(up, p[1], p[2])),
                triton_kernels.fused_mod_relu(z, p[1])], [z, up, *p])
        h, w = rn(256, 128, dtype=dtype), rn(512, 128, dtype=dtype)
        _train([fused_ce.fused_linear_cross_entropy(h, w, torch.randint(0, 512, (256,), device="cuda"))], [h, w])
        g = torch.rand(4, 64, device="cuda").requires_grad_(True)
        _train([triton_kernels.fused_decay_matrix(g, 64)], [g])


def test_no_output_shares_memory_with_an_input(gpu_lib):
    with _Watch() as watch:
        _calls()
    assert not watch.bad, watch.bad
    names = {n for f in SRC.glob("*.py") for n in re.findall(r'^@op\("qpam::(\w+)"\)', f.read_text(), flags=re.M)}
    assert len(names) > 10 and names <= watch.seen, names - watch.seen
