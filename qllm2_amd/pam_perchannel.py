"""E1 per-channel decay on the GPU: V11PAMLayer._forward_chunked_perchannel
(v11/model.py:421-489) with the reference's signature and return tuple.

Per chunk of `chunk` steps the reference folds the decay into the operands
(L = max(cumsum(log max(gamma, 1e-6)), -30) per key channel): queries carry
e^{L} q_scale, keys e^{-L}, the state-write keys e^{L_last - L}, and the state
decays column j by e^{L_last[j]}.  Head dims up to 64 run whole on the HIP
library (qpam_pc_fwd / qpam_pc_bwd): the operands are folded on their way into
LDS, the chunk products run on fp32 MFMA, and only the chunk states pass through
HBM.  Larger head dims (two or more 64-wide tiles per operand) run as

  * the fold in one HIP kernel over all chunks at once (qpam_pc_fold_fwd;
    its backward, qpam_pc_fold_bwd, forms dq, dk and dgamma through both
    clamps);
  * the chunk-parallel products -- the masked score Q K^H, its read of V, the
    chunk's state increment V^T conj(W) and the carried read Q S^T -- as
    batched complex GEMMs over every (b, h, chunk) at once (the library GEMM,
    fp32 complex);
  * the state entering each chunk from the per-column decayed scan over the
    chunks (qpam_pc_scan; backward: the same kernel in reverse).

Both have gradients for q, k, v and gamma.  The whole computation is fp32 (the
reference computes in the input dtype); outputs are cast back to the input
dtype.  A second derivative raises, as it does for the registered operators.
"""

import ctypes
import functools

import torch

from . import _lib

_MASKS = {}


def _mask(c, device):
    key = (c, device)
    m = _MASKS.get(key)
    if m is None:
        m = torch.tril(torch.ones(c, c, device=device, dtype=torch.float32))
        _MASKS[key] = m
    return m


def _dt(t):
    if t.dtype == torch.float32:
        return _lib.QPAM_F32
    if t.dtype == torch.bfloat16:
        return _lib.QPAM_BF16
    raise ValueError(f"qpam per-channel scan: dtype {t.dtype} is not supported (fp32 or bf16)")


def _pairs(x):
    """x [..., d, 2] with the last two dims contiguous (a copy otherwise)."""
    return x if (x.stride(-1) == 1 and x.stride(-2) == 2) else x.contiguous()


def _whole(x):
    """x contiguous, its complex elements on their own alignment (a gradient may
    be a contiguous view at an odd offset)."""
    x = x.contiguous()
    return x if x.data_ptr() % (2 * x.element_size()) == 0 else x.clone()


def _ptr(t):
    return t.data_ptr() if t is not None else None


class _FirstOrder(torch.autograd.Function):
    """The first n arguments (a backward's results, formed outside autograd), tied
    to the others, the tensors they were formed from."""

    @staticmethod
    def forward(ctx, n, *tensors):
        return tuple(t.view_as(t) if t is not None else None for t in tensors[:n])

    @staticmethod
    def backward(ctx, *grads):
        raise RuntimeError("qpam per-channel scan: the gradients come from the HIP library and have no second "
                           "derivative")


def _first_order(backward):
    """A backward whose results a second derivative must not take for constants:
    under create_graph they raise when they are differentiated.  (torch's
    once_differentiable ties them to the incoming gradients only: with a constant
    one, their dependence on the saved tensors would be lost without an error.)
    The saved tensors are inputs or outputs of the function, not copies of them."""

    @functools.wraps(backward)
    def wrapped(ctx, *grads):
        with torch.no_grad():
            out = backward(ctx, *grads)
        if not torch.is_grad_enabled():
            return out
        return _FirstOrder.apply(len(out), *out, *ctx.saved_tensors, *grads)

    return wrapped


class _Fold(torch.autograd.Function):
    """(q, k [B,H,T,d,2] of one dtype, complex rows contiguous, gamma [B,H,T,d],
    channels contiguous) -> qf, kf, wf [B*H, n, C, d, 2] fp32 and atot [B*H, n, d]:
    the folded operands of every chunk."""

    @staticmethod
    def forward(ctx, q, k, gamma, chunk, q_scale):
        if q.dim() != 5 or q.shape[-1] != 2 or k.shape != q.shape or gamma.shape != q.shape[:4]:
            raise ValueError(f"qpam per-channel fold: q, k [B,H,T,d,2] and gamma [B,H,T,d] expected, got "
                             f"{tuple(q.shape)}, {tuple(k.shape)}, {tuple(gamma.shape)}")
        B, H, T, d = q.shape[:4]
        n = -(-T // chunk)
        dev = q.device
        qf, kf, wf = (torch.empty(B * H, n, chunk, d, 2, device=dev, dtype=torch.float32) for _ in range(3))
        atot = torch.empty(B * H, n, d, device=dev, dtype=torch.float32)
        a = _Fold._args(q, k, gamma, chunk, q_scale)
        a.qf, a.kf, a.wf, a.atot = qf.data_ptr(), kf.data_ptr(), wf.data_ptr(), atot.data_ptr()
        with _lib.device(dev):
            _lib.check(_lib.lib().qpam_pc_fold_fwd(ctypes.byref(a), _lib.stream_ptr(dev)), "qpam_pc_fold_fwd")
        ctx.save_for_backward(q, k, gamma)
        ctx.chunk, ctx.q_scale = chunk, q_scale
        return qf, kf, wf, atot

    @staticmethod
    def _args(q, k, gamma, chunk, q_scale):
        B, H, T, d = q.shape[:4]
        a = _lib.PcFoldArgs()
        a.dtype, a.g_dtype = _dt(q), _dt(gamma)
        a.B, a.H, a.T, a.d = B, H, T, d
        a.chunk, a.q_scale = int(chunk), float(q_scale)
        a.q, a.k, a.gamma = q.data_ptr(), k.data_ptr(), gamma.data_ptr()
        a.q_sb, a.q_sh, a.q_st = q.stride(0), q.stride(1), q.stride(2)
        a.k_sb, a.k_sh, a.k_st = k.stride(0), k.stride(1), k.stride(2)
        a.g_sb, a.g_sh, a.g_st = gamma.stride(0), gamma.stride(1), gamma.stride(2)
        return a

    @staticmethod
    @_first_order
    def backward(ctx, dqf, dkf, dwf, datot):
        q, k, gamma = ctx.saved_tensors
        dq, dk = torch.empty(q.shape, device=q.device, dtype=q.dtype), torch.empty(k.shape, device=k.device,
                                                                                     dtype=q.dtype)
        dgamma = torch.empty(gamma.shape, device=gamma.device, dtype=gamma.dtype)
        grads = [_whole(g) if g is not None else None for g in (dqf, dkf, dwf, datot)]
        a = _Fold._args(q, k, gamma, ctx.chunk, ctx.q_scale)
        a.dqf, a.dkf, a.dwf, a.datot = (_ptr(g) for g in grads)
        a.dq, a.dk, a.dgamma = dq.data_ptr(), dk.data_ptr(), dgamma.data_ptr()
        with _lib.device(q.device):
            _lib.check(_lib.lib().qpam_pc_fold_bwd(ctypes.byref(a), _lib.stream_ptr(q.device)), "qpam_pc_fold_bwd")
        return dq, dk, dgamma, None, None


def _scan(x, a, out, init, fin, reverse):
    N, n, d = a.shape
    s = _lib.PcScanArgs()
    s.N, s.n, s.d = N, n, d
    s.x, s.a, s.out, s.init, s.fin = x.data_ptr(), a.data_ptr(), out.data_ptr(), _ptr(init), _ptr(fin)
    s.reverse = 1 if reverse else 0
    with _lib.device(x.device):
        _lib.check(_lib.lib().qpam_pc_scan(ctypes.byref(s), _lib.stream_ptr(x.device)), "qpam_pc_scan")


class _Scan(torch.autograd.Function):
    """(x [N,n,d,d,2] chunk increments, a [N,n,d] column decays, contiguous) ->
    (state entering each chunk [N,n,d,d,2], final state [N,d,d,2])."""

    @staticmethod
    def forward(ctx, x, a):
        if a.dim() != 3 or x.shape != (*a.shape, a.shape[2], 2):
            raise ValueError(f"qpam per-channel scan: x [N,n,d,d,2] and a [N,n,d] expected, got "
                             f"{tuple(x.shape)}, {tuple(a.shape)}")
        N, n, d = a.shape
        out = torch.empty_like(x)
        fin = torch.empty(N, d, d, 2, device=x.device, dtype=torch.float32)
        _scan(x, a, out, None, fin, False)
        ctx.save_for_backward(a, out)
        return out, fin

    @staticmethod
    @_first_order
    def backward(ctx, dout, dfin):
        a, out = ctx.saved_tensors
        dout = _whole(dout) if dout is not None else torch.zeros_like(out)
        dfin = _whole(dfin) if dfin is not None else None
        dx = torch.empty_like(out)
        _scan(dout, a, dx, dfin, None, True)
        # d a[c][j] = sum_i Re(conj(S_in[c][i][j]) dx[c][i][j])
        da = (out * dx).sum(-1).sum(-2)
        return dx, da


KERNEL_D = 64  # head dims up to this run on the chunk kernels


def _aligned(x):
    """x [..., d, 2] whose complex elements start on their own alignment."""
    x = _pairs(x)
    ok = all(s % 2 == 0 for s in x.stride()[:3]) and x.data_ptr() % (2 * x.element_size()) == 0
    return x if ok else x.clone(memory_format=torch.contiguous_format)


class _Chunked(torch.autograd.Function):
    """(q, k, v [B,H,T,d,2], _aligned, gamma [B,H,T,d], channels contiguous,
    d <= 64) -> y [B,H,T,d,2] in q's dtype and the final state [B,H,d,d,2] fp32."""

    @staticmethod
    def forward(ctx, q, k, v, gamma, chunk, q_scale):
        B, H, T, d = q.shape[:4]
        n = -(-T // chunk)
        f32 = dict(device=q.device, dtype=torch.float32)
        y = torch.empty(B, H, T, d, 2, device=q.device, dtype=q.dtype)
        x, atot = torch.empty(B * H, n, d, d, 2, **f32), torch.empty(B * H, n, d, **f32)
        s_fin = torch.empty(B, H, d, d, 2, **f32)
        a = _Chunked._args(q, k, v, gamma, chunk, q_scale, x, atot)
        a.y, a.s_fin = y.data_ptr(), s_fin.data_ptr()
        with _lib.device(q.device):
            _lib.check(_lib.lib().qpam_pc_fwd(ctypes.byref(a), _lib.stream_ptr(q.device)), "qpam_pc_fwd")
        ctx.save_for_backward(q, k, v, gamma, x, atot)
        ctx.chunk, ctx.q_scale = chunk, q_scale
        ctx.set_materialize_grads(False)
        return y, s_fin

    @staticmethod
    def _args(q, k, v, gamma, chunk, q_scale, x, atot):
        a = _lib.PcArgs()
        a.dtype, a.v_dtype, a.g_dtype, a.chunk = _dt(q), _dt(v), _dt(gamma), chunk
        a.B, a.H, a.T, a.d = q.shape[:4]
        a.q_scale = q_scale
        a.q, a.k, a.v, a.gamma = q.data_ptr(), k.data_ptr(), v.data_ptr(), gamma.data_ptr()
        a.q_sb, a.q_sh, a.q_st = q.stride()[:3]
        a.k_sb, a.k_sh, a.k_st = k.stride()[:3]
        a.v_sb, a.v_sh, a.v_st = v.stride()[:3]
        a.g_sb, a.g_sh, a.g_st = gamma.stride()[:3]
        a.x, a.atot = x.data_ptr(), atot.data_ptr()
        return a

    @staticmethod
    @_first_order
    def backward(ctx, dy, dfin):
        q, k, v, gamma, s_in, atot = ctx.saved_tensors
        dy = _whole(dy) if dy is not None else torch.zeros(q.shape, device=q.device, dtype=q.dtype)
        dfin = _whole(dfin) if dfin is not None else None
        dq, dk, dv, dgamma = (torch.empty(t.shape, device=t.device, dtype=t.dtype) for t in (q, k, v, gamma))
        ws = torch.empty_like(s_in)
        a = _Chunked._args(q, k, v, gamma, ctx.chunk, ctx.q_scale, ws, atot)
        a.s_in, a.dy, a.dfin = s_in.data_ptr(), dy.data_ptr(), _ptr(dfin)
        a.dq, a.dk, a.dv, a.dgamma = dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), dgamma.data_ptr()
        with _lib.device(q.device):
            _lib.check(_lib.lib().qpam_pc_bwd(ctypes.byref(a), _lib.stream_ptr(q.device)), "qpam_pc_bwd")
        return dq, dk, dv, dgamma, None, None


def perchannel_chunked(queries, keys, protected_values, decay_gamma, head_dim, chunk_size):
    """V11PAMLayer._forward_chunked_perchannel (v11/model.py:421-489):
    queries, keys, protected_values [B,H,T,d,2], decay_gamma [B,H,T,d] (CUDA,
    fp32 or bf16) -> (y [B,H,T,d,2], final state [B,H,d,d,2]) in the input
    dtype; differentiable in all four inputs."""
    if not queries.is_cuda:
        raise ValueError("qpam per-channel scan: tensors must be on the GPU (no CPU path in this library)")
    B, H, T, d = queries.shape[:4]
    C = int(chunk_size)
    if not 1 <= C <= 64:
        raise ValueError(f"qpam per-channel scan: chunk_size {C} outside 1..64")
    gamma = decay_gamma if decay_gamma.stride(-1) == 1 else decay_gamma.contiguous()
    if d <= KERNEL_D:
        if queries.dim() != 5 or keys.shape != queries.shape or protected_values.shape != queries.shape \
                or queries.shape[-1] != 2 or decay_gamma.shape != queries.shape[:4]:
            raise ValueError(f"qpam per-channel scan: q, k, v [B,H,T,d,2] and gamma [B,H,T,d] expected, got "
                             f"{tuple(queries.shape)}, {tuple(keys.shape)}, {tuple(protected_values.shape)}, "
                             f"{tuple(decay_gamma.shape)}")
        v = protected_values
        y, s_fin = _Chunked.apply(_aligned(queries), _aligned(keys.to(queries.dtype)),
                                  _aligned(v if v.dtype in (torch.float32, torch.bfloat16) else v.float()), gamma, C,
                                  head_dim ** -0.5)
        return y, s_fin.to(queries.dtype)
    n = -(-T // C)
    qf, kf, wf, atot = _Fold.apply(_pairs(queries), _pairs(keys.to(queries.dtype)), gamma, C, head_dim ** -0.5)
    Q, K, W = (torch.view_as_complex(t) for t in (qf, kf, wf))   # [N, n, C, d]
    v = protected_values.float()
    if n * C != T:
        v = torch.nn.functional.pad(v, (0, 0, 0, 0, 0, n * C - T))
    V = torch.view_as_complex(v.reshape(B * H, n, C, d, 2).contiguous())
    # the right operands of the products as contiguous tensors
    P = (Q @ K.conj().transpose(-1, -2).contiguous()) * _mask(C, queries.device)   # masked score [N,n,C,C]
    Y = P @ V
    dS = V.transpose(-1, -2).contiguous() @ W.conj().resolve_conj()                # sum_s v_s[i] conj(w_s[j])
    s_in, s_fin = _Scan.apply(torch.view_as_real(dS).contiguous(), atot)
    Y = Y + Q @ torch.view_as_complex(s_in).transpose(-1, -2).contiguous()      # carried read q' S^T
    y = torch.view_as_real(Y).reshape(B, H, n * C, d, 2)[:, :, :T]
    return y.to(queries.dtype), s_fin.reshape(B, H, d, d, 2).to(queries.dtype)
