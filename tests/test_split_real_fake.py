"""CPU check of the split-real operators' fake kernels: every output of the scan's
and the delta write's forward and backward is planned contiguous, as the kernels
allocate it, also where the gate comes in as a transposed [B,T,H] tensor."""

import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode


def _contiguous(outs):
    return all(o.numel() == 0 or o.stride() == torch.empty(o.shape, device="meta").stride() for o in outs)


@pytest.mark.parametrize("d,dtype", [(64, torch.float32), (48, torch.float32), (64, torch.bfloat16)])
@pytest.mark.parametrize("rotated", [False, True])
def test_fake_outputs_are_contiguous(d, dtype, rotated):
    from qllm2_amd import pam_delta, pam_scan
    B, H, T = 2, 4, 100
    with FakeTensorMode():
        q = torch.empty(B, H, T, d, 2, device="cuda", dtype=dtype)
        gate = torch.empty(B, T, H, device="cuda").transpose(1, 2)
        gamma = gate.unsqueeze(0)
        rot = (gamma, gamma) if rotated else (None, None)
        y, s, pl, ws = out = pam_scan.scan_il_fwd_op(q, q, q, gamma, *rot, 0.125, 64)
        assert _contiguous(out)
        g = pam_scan.scan_il_bwd_op(pl, gamma, *rot, 0.125, 64, ws, y, s, d)
        assert _contiguous(g) and g[3].shape == gamma.shape and [x.numel() for x in g[4:]] == [B * H * T * rotated] * 2
        y, s, pl, ws = out = pam_delta.delta_il_fwd_op(q, q, q, gate, gate, 0.125, 64, True)
        assert _contiguous(out)
        g = pam_delta.delta_il_bwd_op(pl, gate, gate, 0.125, 64, ws, y, s, d, dtype == torch.bfloat16)
        assert _contiguous(g) and g[3].shape == g[4].shape == gate.shape
