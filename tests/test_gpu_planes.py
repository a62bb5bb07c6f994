"""Split-real <-> plane copies (qpam_planes) and the split-real front ends built
on them.  The copies are exact (bf16 by one rounding), so they are compared bit
for bit with torch's slices and stacks; the front ends are compared bit for bit
with the planar entry points, which run the same scan / delta kernels, over head
dims with and without padding, odd lengths, both dtypes, layouts whose rows are
strided, misaligned or expanded, and missing output gradients."""

import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu

LAYOUTS = ["contiguous", "bthd", "offset", "expanded"]


def _layout(x, how):
    """x's values in another memory layout."""
    if how == "bthd":
        return x.transpose(1, 2).contiguous().transpose(1, 2)
    if how == "offset":                     # rows start 8 bytes past a 16-byte boundary
        buf = x.new_zeros(*x.shape[:3], x.shape[3] + 1, 2)
        buf[..., 1:, :] = x
        return buf[..., 1:, :]
    return x[:1, :, :, :, :].expand(x.shape) if how == "expanded" else x.contiguous()


@pytest.mark.parametrize("how", LAYOUTS)
@pytest.mark.parametrize("d", [64, 48, 33, 2])
@pytest.mark.parametrize("src,dst", [("fp32", "fp32"), ("bf16", "fp32"), ("bf16", "bf16")])
def test_split_and_merge_are_exact(gpu_lib, d, src, dst, how):
    from qllm2_amd import planes
    dt = {"fp32": torch.float32, "bf16": torch.bfloat16}
    print(f"case d={d} {src}->{dst} {how}", flush=True)
    g = torch.Generator().manual_seed(d)
    xs = [_layout(torch.randn(2, 3, 5, d, 2, generator=g).to(dt[src]).cuda(), how) for _ in range(3)]
    out = planes.split_rows(xs, dt[dst])
    for x, o in zip(xs, out):
        for i in (0, 1):
            assert torch.equal(o[i], F.pad(x[..., i], (0, 64 - d)).to(dt[dst]))
    s = torch.randn(2, 3, d, d, 2, generator=g).to(dt[src]).cuda()
    sp = planes.split_states(s)
    for i in (0, 1):
        assert torch.equal(sp[i], F.pad(s[..., i].float(), (0, 64 - d, 0, 64 - d)))
    back = planes.merge([(o[0], o[1]) for o in out], [(sp[0], sp[1])], d, dt[src])
    for x, b in zip(xs + [s], back):
        assert torch.equal(x, b)
    rounded = planes.merge([(o[0].float() * 1.001, o[1].float()) for o in out], [], d, torch.bfloat16)
    for o, b in zip(out, rounded):
        assert torch.equal(b, torch.stack([o[0].float() * 1.001, o[1].float()], -1)[..., :d, :].to(torch.bfloat16))


def _grads(y, s, leaves, dy, ds):
    outs, gs = zip(*[(o, g) for o, g in ((y, dy), (s, ds)) if g is not None])
    return torch.autograd.grad(outs, leaves, gs)


@pytest.mark.parametrize("how", LAYOUTS)
@pytest.mark.parametrize("d,M,T,chunk,dtype,given", [
    (64, 1, 70, 64, torch.float32, "both"), (48, 3, 33, 64, torch.float32, "y"), (64, 4, 65, 64, torch.bfloat16, "both"),
    (32, 2, 129, 256, torch.bfloat16, "s"), (33, 1, 16, 16, torch.float32, "both"), (64, 2, 1, 32, torch.bfloat16, "y")])
def test_scan_split_real_equals_planar(gpu_lib, d, M, T, chunk, dtype, given, how):
    from qllm2_amd.pam_scan import chunk_for, pam_scan_interleaved, pam_scan_planar
    print(f"case d={d} M={M} T={T} chunk={chunk} {dtype} {given} {how}", flush=True)
    B, H = 2, 3
    g = torch.Generator().manual_seed(T + d)
    rn = lambda *s: torch.randn(*s, generator=g).cuda()  # noqa: E731
    q, k, v = (_layout((rn(B, H, T, d, 2) * d ** -0.5).to(dtype), how).detach().requires_grad_(True) for _ in range(3))
    gamma = torch.sigmoid(rn(M, B, H, T) + 2).requires_grad_(True)
    rot = tuple(x.requires_grad_(True) for x in (rn(M, B, H, T), rn(M, B, H, T))) if M > 1 else None
    leaves = [q, k, v, gamma] + list(rot or ())
    dy = rn(B, H, T, d, 2).to(dtype) if given != "s" else None
    ds = rn(M, B, H, d, d, 2).to(dtype) if given != "y" else None
    y, s = pam_scan_interleaved(q, k, v, gamma, d, chunk, rot=rot)
    got = [y, s, *_grads(y, s, leaves, dy, ds)]
    pl = [x[..., i].contiguous() for x in (q, k, v) for i in (0, 1)]
    yr, yi, sr, si = pam_scan_planar(*pl, gamma, q_scale=d ** -0.5, chunk=chunk_for(chunk, T), rot=rot)
    y, s = torch.stack([yr, yi], -1).to(dtype), torch.stack([sr, si], -1).to(dtype)
    want = [y, s, *_grads(y, s, leaves, dy, ds)]
    for i, (a, b) in enumerate(zip(got, want)):
        assert a.dtype == b.dtype and torch.equal(a, b), i


@pytest.mark.parametrize("how", LAYOUTS)
@pytest.mark.parametrize("d,T,chunk,dtype,given", [
    (64, 70, 64, torch.float32, "both"), (32, 129, 64, torch.bfloat16, "y"), (48, 33, 16, torch.float32, "s"),
    (64, 1, 64, torch.bfloat16, "both")])
def test_delta_split_real_equals_planar(gpu_lib, d, T, chunk, dtype, given, how):
    from qllm2_amd.pam_delta import delta_planar, forward_delta
    print(f"case d={d} T={T} chunk={chunk} {dtype} {given} {how}", flush=True)
    B, H = 2, 3
    g = torch.Generator().manual_seed(T + d)
    rn = lambda *s: torch.randn(*s, generator=g).cuda()  # noqa: E731
    q, k, v = (_layout((rn(B, H, T, d, 2) * (2 * d) ** -0.5).to(dtype), how).detach().requires_grad_(True)
               for _ in range(3))
    gamma, beta = (torch.sigmoid(rn(B, H, T) + m).requires_grad_(True) for m in (2, 0))
    leaves = [q, k, v, gamma, beta]
    dy = rn(B, H, T, d, 2).to(dtype) if given != "s" else None
    ds = rn(B, H, d, d, 2).to(dtype) if given != "y" else None
    y, s = forward_delta(*leaves, d, chunk=chunk)
    got = [y, s, *_grads(y, s, leaves, dy, ds)]
    pl = [x[..., i].contiguous() for x in (q, k, v) for i in (0, 1)]
    yr, yi, sr, si = delta_planar(*pl, gamma, beta, q_scale=d ** -0.5, chunk=chunk)
    y, s = torch.stack([yr, yi], -1).to(dtype), torch.stack([sr, si], -1).to(dtype)
    want = [y, s, *_grads(y, s, leaves, dy, ds)]
    for i, (a, b) in enumerate(zip(got, want)):
        assert a.dtype == b.dtype and torch.equal(a, b), i


@pytest.mark.parametrize("kind", ["scan", "delta"])
@pytest.mark.parametrize("T,M,form", [
    (1, 1, "dense"), (63, 2, "dense"), (130, 4, "dense"),
    (70, 1, "heads_last"),   # the rows of a [B,T,H,64,2] tensor
    (70, 2, "expanded"),     # one row for all (strides 0)
    (70, 1, "padded"),       # rows of 65 complex elements: packed first
    (70, 1, "offset"),       # 8-byte aligned storage: packed first
    (70, 1, "none"),         # the state's gradient only
])
def test_split_real_rows_equal_planes(gpu_lib, T, M, form, kind):
    """fp32, head dim 64 (64-step chunks for the scan): y leaves and the gradients arrive and leave as
    split-real rows.  The arithmetic is that of the planes, so every result is the
    planar call's bit for bit, whatever the strides of dy."""
    from qllm2_amd.pam_delta import delta_planar, forward_delta
    from qllm2_amd.pam_scan import pam_scan_interleaved, pam_scan_planar
    B, H, d = 2, 3, 64
    g = torch.Generator().manual_seed(17 * T + M)
    qkv = [(0.3 * torch.randn(B, H, T, d, 2, generator=g)).cuda() for _ in range(3)]
    lead = (M, B, H) if kind == "scan" else (B, H)
    gates = [(0.85 + 0.15 * torch.rand(*lead, T, generator=g)).cuda()]
    if kind == "delta":
        gates.append(torch.rand(*lead, T, generator=g).cuda())
    ds = torch.randn(*lead, d, d, 2, generator=g).cuda()
    dy = torch.randn(B, H, T, d, 2, generator=g).cuda()
    if form == "heads_last":
        dy = dy.transpose(1, 2).contiguous().transpose(1, 2)
    elif form == "expanded":
        dy = dy[:1, :1, :1].expand(B, H, T, d, 2)
    elif form == "padded":
        dy = torch.nn.functional.pad(dy, (0, 0, 0, 1))[..., :d, :]
    elif form == "offset":
        buf = torch.empty(dy.numel() + 2, device="cuda")
        buf[2:] = dy.reshape(-1)
        dy = buf[2:].view(B, H, T, d, 2)

    xs = [x.clone().requires_grad_(True) for x in (*qkv, *gates)]
    y, s = pam_scan_interleaved(*xs, d, 64) if kind == "scan" else forward_delta(*xs, d)
    ps = [x[..., i].contiguous().requires_grad_(True) for x in qkv for i in (0, 1)]
    gs = [x.clone().requires_grad_(True) for x in gates]
    y_re, y_im, s_re, s_im = (pam_scan_planar(*ps, *gs, q_scale=d ** -0.5, chunk=64) if kind == "scan"
                              else delta_planar(*ps, *gs, q_scale=d ** -0.5))
    assert torch.equal(y, torch.stack([y_re, y_im], -1)) and torch.equal(s, torch.stack([s_re, s_im], -1))
    if form == "none":
        got = torch.autograd.grad([s], xs, [ds])
        ref = torch.autograd.grad([s_re, s_im], [*ps, *gs], [ds[..., 0], ds[..., 1]])
    else:
        got = torch.autograd.grad([y, s], xs, [dy, ds])
        ref = torch.autograd.grad([y_re, y_im, s_re, s_im], [*ps, *gs],
                                  [dy[..., 0].contiguous(), dy[..., 1].contiguous(), ds[..., 0], ds[..., 1]])
    for i in range(3):
        assert torch.equal(got[i], torch.stack([ref[2 * i], ref[2 * i + 1]], -1)), i
    for a, b in zip(got[3:], ref[6:]):
        assert torch.equal(a, b)


@pytest.mark.parametrize("d,M,T,dtype", [(64, 1, 70, torch.float32), (48, 2, 33, torch.float32), (64, 2, 65, torch.bfloat16)])
def test_fake_kernels_match_the_real_ones(gpu_lib, d, M, T, dtype):
    """Shape, strides and dtype of every output, with a gate (and rotations) transposed from [B,T,H]."""
    from torch._subclasses.fake_tensor import FakeTensorMode
    from qllm2_amd import pam_delta, pam_scan
    print(f"case d={d} M={M} T={T} {dtype}", flush=True)
    B, H = 2, 4

    def calls(make):
        q = make(B, H, T, d, 2).to(dtype)
        gate = make(B, T, H).transpose(1, 2)
        gamma = make(M, B, T, H).transpose(2, 3)
        rot = (gamma, gamma) if M > 1 else (None, None)
        y, s, pl, ws = out = pam_scan.scan_il_fwd_op(q, q, q, gamma, *rot, 0.125, 64)
        outs = out + pam_scan.scan_il_bwd_op(pl, gamma, *rot, 0.125, 64, ws, y, s, d)
        y, s, pl, ws = out = pam_delta.delta_il_fwd_op(q, q, q, gate, gate, 0.125, 64, True)
        return outs + out + pam_delta.delta_il_bwd_op(pl, gate, gate, 0.125, 64, ws, y, s, d, dtype == torch.bfloat16)

    real = calls(lambda *s: torch.full(s, 0.5, device="cuda"))
    with FakeTensorMode():
        fake = calls(lambda *s: torch.empty(s, device="cuda"))
    for i, (r, f) in enumerate(zip(real, fake)):
        assert r.shape == f.shape and r.stride() == f.stride() and r.dtype == f.dtype, i
