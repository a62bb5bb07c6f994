"""The per-channel chunk kernels (head dims up to 64, qpam_pc_fwd / qpam_pc_bwd)
against the general path (fold kernels and batched library products), which is
itself checked against the oracle: same calls over head dims and chunk lengths at
the edges of the 16-wide tiles, ragged last chunks, one step, mixed dtypes,
strided / misaligned / expanded layouts, prefixes past the -30 clamp and missing
output gradients.  Both sum the same fp32 products in other orders: a 64-term
sum of both sits within 64 * 2^-24 = 4e-6 of the exact one relative to the sum of
magnitudes, and the two chained products and e^{+-L} factors (2^-22 each) add
about as much: 2e-5 of the tensor's largest value.  bf16 inputs are widened
exactly; bf16 results differ by one rounding on each side, of at most 2^-8 of the
value each (8 bits of significand): 2^-7 more.
dgamma is held element by element (_dgamma_terms)."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _layout(x, how):
    if how == "bthd":
        return x.transpose(1, 2).contiguous().transpose(1, 2)
    if how == "offset":          # complex elements start between their alignments
        buf = x.new_zeros(x.numel() + 1)
        buf[1:] = x.reshape(-1)
        return buf[1:].view(x.shape)
    return x[:1].expand(x.shape) if how == "expanded" else x.contiguous()


def _dgamma_terms(q, k, dq, dk, C):
    """Sum of the magnitudes that gamma's gradient at a step and channel is made of
    (times gamma): q dq and k dk of the chunk's steps from this one on, and behind
    the chunk's last prefix k dk of the whole chunk and, through the entering state,
    of every earlier step."""
    def size(x, dx):
        if dx is None:
            return torch.zeros(x.shape[:-1], device=x.device)
        return (x.float() * dx.float()).abs().sum(-1)

    tq, tk = size(q, dq), size(k, dk)
    T = tq.shape[2]
    chunks = lambda x: torch.nn.functional.pad(x, (0, 0, 0, -T % C)).unflatten(2, (-1, C))  # noqa: E731
    own, keys = chunks(tq + tk), chunks(tk)
    after = own.flip(3).cumsum(3).flip(3)
    return (after + keys.sum(3).cumsum(2).unsqueeze(3)).flatten(2, 3)[:, :, :T]


@pytest.mark.parametrize("d,C,T,dtypes,how,given,strong", [
    (64, 64, 130, "fff", "contiguous", "both", False), (64, 64, 64, "fff", "bthd", "y", False),
    (33, 33, 70, "fff", "offset", "both", False), (32, 64, 129, "bbb", "contiguous", "both", False),
    (31, 17, 50, "bff", "bthd", "s", False), (16, 16, 33, "fbf", "offset", "both", True),
    (17, 64, 63, "ffb", "expanded", "both", False), (48, 48, 1, "fff", "contiguous", "both", False),
    (1, 1, 5, "fff", "contiguous", "both", False), (2, 64, 65, "bfb", "contiguous", "y", True),
    (64, 32, 100, "bbb", "offset", "both", True), (64, 15, 46, "fff", "bthd", "both", False),
    (64, 64, 130, "fff", "contiguous", "both", True), (48, 32, 100, "fff", "bthd", "both", True),
    (64, 32, 65, "bff", "contiguous", "both", True),
])
def test_chunk_kernels_equal_general_path(gpu_lib, monkeypatch, d, C, T, dtypes, how, given, strong):
    from qllm2_amd import pam_perchannel as P
    print(f"case d={d} C={C} T={T} {dtypes} {how} {given} strong={strong}", flush=True)
    B, H = 2, 3
    dt = [{"f": torch.float32, "b": torch.bfloat16}[x] for x in dtypes]      # q and k, v, gamma
    g = torch.Generator().manual_seed(T + d)
    rn = lambda *s: torch.randn(*s, generator=g).cuda()  # noqa: E731
    q, k, v = (_layout((rn(B, H, T, d, 2) * (2 * d) ** -0.5).to(t), how) for t in (dt[0], dt[0], dt[1]))
    gamma = torch.sigmoid(rn(B, H, T, d) + (-1.0 if strong else 3.0)).to(dt[2])
    leaves = [x.detach().requires_grad_(True) for x in (q, k, v, gamma)]
    dy = rn(B, H, T, d, 2).to(dt[0]) if given != "s" else None
    ds = rn(B, H, d, d, 2).to(dt[0]) if given != "y" else None
    res = []
    for limit in (64, 0):
        monkeypatch.setattr(P, "KERNEL_D", limit)
        y, s = P.perchannel_chunked(*leaves, d, C)
        outs, gs = zip(*[(o, x) for o, x in ((y, dy), (s, ds)) if x is not None])
        res.append([y, s, *torch.autograd.grad(outs, leaves, gs, allow_unused=True)])
    for name, a, b in zip(("y", "s", "dq", "dk", "dv", "dgamma"), *res):
        if b is None:            # the general path has no gradient here (dq from the state alone)
            assert a is None or not a.any(), name
            continue
        assert a.dtype == b.dtype and a.shape == b.shape, name
        err, ref = (a.float() - b.float()).abs(), b.float().abs()
        rounding = 2.0 ** -7 if a.dtype == torch.bfloat16 else 0.0
        if name == "dgamma":
            _, _, dq, dk, _, _ = res[1]
            bound = 2e-5 * _dgamma_terms(q, k, dq, dk, C) / gamma.float() + rounding * ref
            assert (err <= bound + 1e-30).all(), f"{name}: {(err / (bound + 1e-30)).max().item():.2f} of its bound"
            continue
        top = max(ref.max().item(), 1e-30)
        assert err.max().item() <= (2e-5 + rounding) * top, f"{name}: {err.max().item():.2e} of {top:.2e}"


@pytest.mark.parametrize("d,C,T,shift", [(64, 64, 300, 3.0), (64, 64, 300, 0.0), (64, 16, 200, 3.0), (33, 33, 100, 5.0),
                                         (16, 64, 200, 3.0)])
def test_chunk_kernels_are_as_exact_as_the_general_path(gpu_lib, monkeypatch, d, C, T, shift):
    """Each plane's distance from 64 bits, the chunk kernels' against the general
    path's: no larger, but for chance.  With E the squared errors of the groups that
    are independent of one another (an element, whose two parts share its factors;
    for dgamma a channel's chunk, which is one running sum), a squared norm sum(E)
    has a variance of at most sum(E^2), so two norms differ by a deviation of
    (sum(E^2) / 2)^(1/2) / sum(E); three of them.  shift 0: prefixes past -30, where
    the factors e^{L}, e^{-L} and e^{L_last - L} are far apart."""
    from oracle import pam as O
    from qllm2_amd import pam_perchannel as P
    B, H = 2, 4
    g = torch.Generator().manual_seed(10 * T + d)
    q, k, v = (torch.randn(B, H, T, d, 2, generator=g) * (2 * d) ** -0.5 for _ in range(3))
    gamma = torch.sigmoid(torch.randn(B, H, T, d, generator=g) + shift)
    dy, ds = torch.randn(B, H, T, d, 2, generator=g), torch.randn(B, H, d, d, 2, generator=g)
    ref = [x.double().requires_grad_(True) for x in (q, k, v, gamma)]
    y, s = O.chunked_perchannel(*ref, d, C)
    want = [y, s, *torch.autograd.grad((y, s), ref, (dy.double(), ds.double()))]
    res = []
    for limit in (64, 0):
        monkeypatch.setattr(P, "KERNEL_D", limit)
        leaves = [x.cuda().requires_grad_(True) for x in (q, k, v, gamma)]
        y, s = P.perchannel_chunked(*leaves, d, C)
        res.append([y, s, *torch.autograd.grad((y, s), leaves, (dy.cuda(), ds.cuda()))])
    worse = []
    for name, r, a, b in zip(("y", "s", "dq", "dk", "dv", "dgamma"), want, *res):
        ea, eb = ((x.detach().double().cpu() - r.detach()) ** 2 for x in (a, b))
        if name == "dgamma":
            eb = torch.nn.functional.pad(eb, (0, 0, 0, -T % C)).unflatten(2, (-1, C))
            E, parts = eb.sum(3), [(ea.sum(), eb.sum())]
        else:
            E, parts = eb.sum(-1), [(ea[..., i].sum(), eb[..., i].sum()) for i in (0, 1)]
        slack = 3 * (((E ** 2).sum() / 2) ** 0.5 / E.sum()).item()
        for i, (x, z) in enumerate(parts):
            ratio = (x / z).sqrt().item()
            print(f"d={d} C={C} T={T} {name}[{i}]: chunk kernels / general path {ratio:.3f}, slack {slack:.3f}", flush=True)
            if ratio > 1 + slack:
                worse.append((name, i, ratio, slack))
    assert not worse, worse


@pytest.mark.parametrize("d,dtype", [(64, torch.float32), (33, torch.bfloat16), (80, torch.float32)])
def test_incoming_gradients_at_any_offset(gpu_lib, d, dtype):
    """Contiguous gradients whose complex elements start between their alignments
    give what aligned ones give, on the chunk kernels and on the general path."""
    from qllm2_amd import pam_perchannel as P
    print(f"case d={d} {dtype}", flush=True)
    B, H, T, C = 1, 2, 70, 64
    g = torch.Generator().manual_seed(d)
    rn = lambda *s: torch.randn(*s, generator=g).cuda()  # noqa: E731
    q, k, v = ((rn(B, H, T, d, 2) * (2 * d) ** -0.5).to(dtype).requires_grad_(True) for _ in range(3))
    gamma = torch.sigmoid(rn(B, H, T, d) + 3).to(dtype).requires_grad_(True)
    dy, ds = rn(B, H, T, d, 2).to(dtype), rn(B, H, d, d, 2).to(dtype)
    got = []
    for how in ("contiguous", "offset"):
        y, s = P.perchannel_chunked(q, k, v, gamma, d, C)
        got.append(torch.autograd.grad((y, s), (q, k, v, gamma), (_layout(dy, how), _layout(ds, how))))
    for a, b in zip(*got):
        assert torch.equal(a, b)


def test_more_chunks_than_one_grid_row_of_threads(gpu_lib):
    """8.64 million chunks of one step: 2^32 threads and more in one row of 512-thread
    blocks.  The result does not depend on the chunk length (prefixes stay far above
    -30), so chunks of 64 steps are the reference; both sum at most 100 decayed terms
    of weight (a sum of gamma^n below 1 / (1 - 0.9)) in fp32: 2e-5 of the largest."""
    from qllm2_amd import pam_perchannel as P
    B, H, T, d = 1, 96, 90000, 1
    g = torch.Generator(device="cuda").manual_seed(0)
    q, k, v = (torch.randn(B, H, T, d, 2, device="cuda", generator=g).requires_grad_(True) for _ in range(3))
    gamma = (0.7 + 0.2 * torch.rand(B, H, T, d, device="cuda", generator=g)).requires_grad_(True)
    dy = torch.randn(B, H, T, d, 2, device="cuda", generator=g)
    res = []
    for C in (1, 64):
        print(f"chunk {C}: {B * H * -(-T // C)} chunks", flush=True)
        y, s = P.perchannel_chunked(q, k, v, gamma, d, C)
        res.append([y, s, *torch.autograd.grad(y, (q, k, v, gamma), dy)])
    for name, a, b in zip(("y", "s", "dq", "dk", "dv", "dgamma"), *res):
        assert (a - b).abs().max().item() <= 2e-5 * b.abs().max().item(), name


@pytest.mark.parametrize("where", ["q", "k", "v", "dy", "ds"])
def test_an_infinity_stays_in_its_part(gpu_lib, monkeypatch, where):
    """No NaN where the general path has a number or an infinity."""
    from qllm2_amd import pam_perchannel as P
    print(f"case {where}", flush=True)
    B, H, T, d, C = 1, 2, 150, 64, 64
    g = torch.Generator().manual_seed(5)
    x = {n: torch.randn(B, H, T, d, 2, generator=g) * (2 * d) ** -0.5 for n in ("q", "k", "v", "dy")}
    x["ds"] = torch.randn(B, H, d, d, 2, generator=g)
    x[where][(0, 1, 3, 4, 0) if where == "ds" else (0, 1, 70, 5, 0)] = float("inf")
    gamma = torch.sigmoid(torch.randn(B, H, T, d, generator=g) + 2)
    res = []
    for limit in (64, 0):
        monkeypatch.setattr(P, "KERNEL_D", limit)
        leaves = [t.cuda().requires_grad_(True) for t in (x["q"], x["k"], x["v"], gamma)]
        y, s = P.perchannel_chunked(*leaves, d, C)
        res.append([y, s, *torch.autograd.grad((y, s), leaves, (x["dy"].cuda(), x["ds"].cuda()))])
    assert any(not b.isfinite().all() for b in res[1])
    for name, a, b in zip(("y", "s", "dq", "dk", "dv", "dgamma"), *res):
        assert not (a.isnan() & ~b.isnan()).any(), name
