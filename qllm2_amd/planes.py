"""Split-real [..., d, 2] tensors to and from pairs of planes (qpam_planes):
every tensor of a call in one launch, dtype conversion and zero padding to the
kernels' head dim included.  Replaces the per-plane slices, casts, pads and
stacks around the reference's split-real entry points (v11/model.py:378-417,
491-576, v11/flash_pam.py:56-152).  No autograd here: the custom ops that call
these functions carry their own backward.
"""

import torch

from . import _lib

KD = 64  # head dim of the scan and delta kernels (plane width)

_CODE = {torch.float32: _lib.QPAM_F32, torch.bfloat16: _lib.QPAM_BF16}


def covers(*ts):
    """True when every tensor is on the GPU in one dtype the kernel converts."""
    return all(t.is_cuda and t.dtype == ts[0].dtype for t in ts) and ts[0].dtype in _CODE


def fits(q, n_states):
    """True when the element groups of q [B,H,T,d,2] and of n_states states per
    head stay inside the kernel's 31-bit index."""
    heads = q.shape[0] * q.shape[1]
    return heads * max(q.shape[2], n_states * KD) * (KD // 4) < 2 ** 31


def _pairs(x):
    return x if x.stride(-1) == 1 and x.stride(-2) == 2 else x.contiguous()


def _launch(items, merge, device):
    a = _lib.PlanesArgs(len(items), merge)
    for i, (il, re, im, n0, n1, n2, n2_il, d, dp, ls, ps) in enumerate(items):
        a.item[i] = _lib.PlanesItem(il.data_ptr(), *ls, re.data_ptr(), im.data_ptr(), *ps, n0, n1, n2, n2_il, d, dp,
                                    _CODE[il.dtype], _CODE[re.dtype])
    with _lib.device(device):
        _lib.check(_lib.lib().qpam_planes(a, _lib.stream_ptr(device)), "qpam_planes")


def split_rows(xs, dtype):
    """xs: up to four [B,H,T,d,2] tensors of one shape -> one [len(xs), 2, B, H, T, 64]
    tensor in `dtype` (re plane, im plane of each; columns d.. zero)."""
    B, H, T, d = xs[0].shape[:4]
    out = torch.empty(len(xs), 2, B, H, T, KD, device=xs[0].device, dtype=dtype)
    xs = [_pairs(x) for x in xs]
    ps = (H * T * KD, T * KD, KD)
    _launch([(x, o[0], o[1], B, H, T, T, d, KD, x.stride()[:3], ps) for x, o in zip(xs, out)], 0, out.device)
    return out


def split_states(s):
    """s [..., d, d, 2] -> fp32 [2, ..., 64, 64] (padded rows and columns zero)."""
    lead, d = s.shape[:-3], s.shape[-2]
    s = s.contiguous()
    n = s.numel() // (d * d * 2)
    out = torch.empty(2, *lead, KD, KD, device=s.device, dtype=torch.float32)
    _launch([(s, out[0], out[1], 1, n, KD, d, d, KD, (0, 2 * d * d, 2 * d), (0, KD * KD, KD))], 0, s.device)
    return out


def _rows_item(re, im, d, dtype):
    B, H, T = re.shape[:3]
    il = torch.empty(B, H, T, d, 2, device=re.device, dtype=dtype)
    return il, (il, re, im, B, H, T, T, d, re.shape[-1], il.stride()[:3], re.stride()[:3])


def _states_item(re, im, d, dtype):
    """Planes [..., 64, 64] -> [..., d, d, 2]."""
    lead = re.shape[:-2]
    il = torch.empty(*lead, d, d, 2, device=re.device, dtype=dtype)
    n = re.numel() // (KD * KD)
    return il, (il, re, im, 1, n, KD, d, d, KD, (0, 2 * d * d, 2 * d), (0, KD * KD, KD))


def merge(rows, states, d, dtype):
    """Planes back to split-real tensors in `dtype`, one launch: rows is a list of
    (re, im) [B,H,T,64] plane pairs -> [B,H,T,d,2] each, states a list of (re, im)
    [..., 64, 64] pairs -> [..., d, d, 2] each (up to four in all)."""
    made = [_rows_item(re, im, d, dtype) for re, im in rows]
    made += [_states_item(re, im, d, dtype) for re, im in states]
    _launch([m[1] for m in made], 1, made[0][0].device)
    return [m[0] for m in made]
