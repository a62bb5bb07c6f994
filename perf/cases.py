"""Workloads that stand for this framework's use, one pass each, for timing and
for comparing outputs: prefill and training of the PAM scan (one state and E3,
fp32 and bf16, planar and split-real entry points), the whole PAM layer, the
E1 per-channel and E2 delta variants, ragged decode over a slot pool, token
decode of a whole model, the LM-head cross-entropy and the complex elementwise
layers.

`listed()` names twelve of them, `draw(rng)` gives others of the same ranges.
Inputs are made on the GPU from the seed alone; `exact` computes a case's
outputs in float64 with plain torch.
"""

import copy
import math

import torch
import torch.nn.functional as F

DEV = "cuda"
DTYPES = {"fp32": torch.float32, "bf16": torch.bfloat16}


def listed():
    return [
        # one short prompt of a serving process through the split-real drop-in: launches and host work
        dict(name="scan_prompt_fp32", kind="scan", api="flash", B=1, H=12, T=100, d=64, M=1, chunk=64, dtype="fp32",
             grad=False),
        # the headline prefill: a batch of full-length sequences, fp32, planar operands
        dict(name="scan_prefill_fp32", kind="scan", api="planar", B=8, H=12, T=2048, d=64, M=1, chunk=64, dtype="fp32",
             grad=False),
        # fp32 training of a one-state layer at a ragged length through the split-real drop-in
        dict(name="scan_train_fp32", kind="scan", api="flash", B=4, H=12, T=1000, d=64, M=1, chunk=256, dtype="fp32",
             grad=True),
        # E3 training in bf16: three states per head with read rotations
        dict(name="scan_train_e3_bf16", kind="scan", api="planar", B=8, H=12, T=2048, d=64, M=3, chunk=64, dtype="bf16",
             grad=True),
        # prefill of one ragged prompt through the whole PAM layer (projections, prologue, scan, o_proj)
        dict(name="layer_prompt_bf16", kind="layer", B=1, T=1000, dim=768, H=12, d=64, M=3, dtype="bf16", grad=False),
        # a training step of the production E3 layer
        dict(name="layer_train_bf16", kind="layer", B=8, T=2048, dim=768, H=12, d=64, M=3, dtype="bf16", grad=True),
        # one token for three quarters of 256 slots, every layer's heads in one launch
        dict(name="decode_slots", kind="decode", slots=256, live=192, groups=192, d=64, M=1, rope=False),
        # one token of a 16-block model for 192 live sequences, graph replay, logits of every row
        dict(name="model_decode_bf16", kind="model", blocks=16, slots=256, live=192, dim=768, H=12, d=64, M=3,
             vocab=50261, dtype="bf16"),
        # the tied LM head's loss and gradients over the full vocabulary
        dict(name="ce_train_bf16", kind="ce", N=16384, D=1024, V=50261, dtype="bf16", master=False, grad=True),
        # the elementwise layers of a block, forward and backward: norm, then gate of two halves
        dict(name="norm_cgu_train_bf16", kind="elementwise", rows=16384, dim=1024, dtype="bf16", grad=True),
        # E2 delta-write training
        dict(name="delta_train_fp32", kind="delta", B=8, H=12, T=2048, d=64, chunk=64, dtype="fp32", grad=True),
        # E1 per-channel-decay training
        dict(name="perchannel_train_fp32", kind="perchannel", B=8, H=12, T=2048, d=64, chunk=64, dtype="fp32", grad=True),
    ]


def _span(rng, lo, hi):
    """An integer of [lo, hi], uniform over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["scan"] * 4 + ["layer"] * 2 + ["decode", "model", "ce", "elementwise", "delta", "perchannel"])
    if kind in ("scan", "delta", "perchannel"):
        B, H, T = _span(rng, 1, 8), rng.choice([4, 6, 8, 12, 16]), _span(rng, 33, 2048)
        while B * H * T > 8 * 12 * 2048:
            B -= 1
        grad = rng.random() < 0.6
        if kind == "scan":
            M, dtype = rng.choice([1, 1, 2, 3, 4]), rng.choice(["fp32", "bf16"])
            d, chunk = rng.choice([64, 64, 64, 64, 32, 48]), rng.choice([64, 64, 256, 32])
            if M == 4 and B * H * T > 6 * 12 * 2048:
                T = T * 3 // 4
            return dict(kind="scan", api="flash" if M == 1 and rng.random() < 0.5 else "planar", B=B, H=H, T=T, d=d, M=M,
                        chunk=chunk, dtype=dtype, grad=grad)
        return dict(kind=kind, B=B, H=H, T=T, d=rng.choice([64, 64, 64, 32]), chunk=rng.choice([64, 64, 32]),
                    dtype=rng.choice(["fp32", "fp32", "bf16"]), grad=grad)
    if kind == "layer":
        H, d = rng.choice([(4, 64), (8, 64), (12, 64), (12, 64), (16, 64), (12, 32), (6, 128)])
        B, T = _span(rng, 1, 8), _span(rng, 33, 2048)
        while B * T * H * d > 8 * 2048 * 768:
            B -= 1
        return dict(kind="layer", B=B, T=T, dim=H * d, H=H, d=d, M=rng.choice([1, 2, 3, 4] if d == 64 else [1, 2]),
                    dtype=rng.choice(["bf16", "bf16", "fp32"]), grad=rng.random() < 0.5)
    if kind == "decode":
        slots, M = _span(rng, 2, 256), rng.choice([1, 1, 2, 3, 4])
        d = rng.choice([64, 64, 64, 32, 128]) if M == 1 else rng.choice([64, 64, 32])
        groups = 12 * _span(rng, 1, 16)
        while slots * groups * M * d * d > 256 * 192 * 4096:
            groups = max(1, groups // 2)
        return dict(kind="decode", slots=slots, live=max(1, int(slots * rng.uniform(0.5, 1.0))), groups=groups, d=d, M=M,
                    rope=rng.random() < 0.5)
    if kind == "model":
        H, slots = rng.choice([4, 8, 12]), _span(rng, 4, 256)
        return dict(kind="model", blocks=rng.choice([2, 3, 4, 6]), slots=slots,
                    live=max(1, int(slots * rng.uniform(0.5, 1.0))), dim=64 * H, H=H, d=64, M=rng.choice([1, 2, 3]),
                    vocab=rng.choice([8192, 32000, 50261]), dtype="bf16")
    if kind == "ce":
        N, D, V = _span(rng, 64, 16384), rng.choice([512, 768, 1024, 1536]), rng.choice([8192, 32000, 50261])
        while N * D * V > 16384 * 1024 * 50261:
            N -= N // 4
        return dict(kind="ce", N=N, D=D, V=V, dtype="bf16", master=rng.random() < 0.3, grad=rng.random() < 0.7)
    return dict(kind="elementwise", rows=_span(rng, 200, 32768), dim=rng.choice([256, 384, 512, 768, 1024]),
                dtype=rng.choice(["bf16", "bf16", "fp32"]), grad=rng.random() < 0.7)


# ---------------------------------------------------------------- inputs

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _randn(g, *shape, std=1.0, mean=0.0, dtype=torch.float32):
    x = torch.empty(*shape, device=DEV, dtype=torch.float32).normal_(mean, std, generator=g)
    return x.to(dtype)


def _unit(x):
    """Complex rows [..., d, 2] scaled to unit norm (the keys and queries of a normalised layer)."""
    return x / x.square().sum((-1, -2), keepdim=True).sqrt()


def _gammas(g, M, *shape):
    """Decays of M states, slower from state to state, as a layer's softplus gates give them."""
    return torch.stack([torch.sigmoid(_randn(g, *shape, mean=(3.0 if M == 1 else 2.0 + m))) for m in range(M)])


def _prepare_scan(c, g):
    B, H, T, d, M, dt = c["B"], c["H"], c["T"], c["d"], c["M"], DTYPES[c["dtype"]]
    q, k = (_unit(_randn(g, B, H, T, d, 2)).to(dt) * math.sqrt(d) ** (i == 0) for i in (0, 1))
    v = _randn(g, B, H, T, d, 2, dtype=dt)
    gamma = _gammas(g, M, B, H, T)
    phase = _randn(g, M, B, H, T) if M > 1 else None
    dy = _randn(g, B, H, T, d, 2)
    if c["api"] == "flash":
        leaves = [q, k, v, gamma[0]]
        s = dict(dy=dy.to(dt))
    else:
        leaves = [x[..., i].contiguous() for x in (q, k, v) for i in (0, 1)] + [gamma]
        if M > 1:
            leaves += [torch.cos(phase), torch.sin(phase)]
        s = dict(dy=(dy[..., 0].contiguous(), dy[..., 1].contiguous()))
    s["leaves"] = [x.requires_grad_(c["grad"]) for x in leaves]
    return s


def _module(**attrs):
    m = torch.nn.Module()
    for k, v in attrs.items():
        setattr(m, k, v)
    return m


def _pam_module(g, dim, H, d, M, T, dtype):
    """A PAM layer of the production setting with the reference's attribute
    names: fused QKV, RoPE, GSP gate and phase routing on |x|, head decay,
    additive write."""
    from qllm2_amd.decode import build_rope_cache

    def prm(*shape, std, mean=0.0):
        return torch.nn.Parameter(_randn(g, *shape, std=std, mean=mean, dtype=dtype))

    def clin(o, i):
        return _module(weight_real=prm(o, i, std=(2 * i) ** -0.5), weight_imag=prm(o, i, std=(2 * i) ** -0.5),
                       bias_real=None, bias_imag=None)

    def lin(o, i, std, mean=0.0):
        m = torch.nn.Linear(i, o, device=DEV, dtype=dtype)
        m.weight, m.bias = prm(o, i, std=std), prm(o, std=0.1, mean=mean)
        return m

    mod = _module(num_heads=H, head_dim=d, n_states=M, inner_dim=H * d, chunk_size=256, use_rope=True, use_gsp=True,
                  qk_norm=False, fused_qkv=True, gamma_floor=0.0, gate_content_aware=False,
                  routing_content_aware=False, state_compete=False, decay_mode="head", write_mode="additive",
                  fused_e3=True, gate_surprisal_lambda=0.0, dt_bias=prm(H, std=0.5, mean=-2.0),
                  qkv_proj=clin(3 * H * d, dim), o_proj=clin(dim, H * d), dt_proj=lin(H, 2 * dim, 0.3 * (2 * dim) ** -0.5),
                  protect_gate=lin(H, dim, dim ** -0.5, -1.0), dropout=torch.nn.Dropout(0.0))
    if M > 1:
        mod.state_dt_offset = torch.nn.Parameter(torch.linspace(-1.0, 1.0, M, device=DEV).to(dtype))
        mod.phase_proj = lin(H * M, dim, dim ** -0.5)
    mod.register_buffer("rope_cache", build_rope_cache(2 * T, d, device=DEV), persistent=False)
    mod._route_balance_loss = lambda w: None
    mod.eval()
    return mod


def _model(g, c):
    """A V11LM-shaped module with random weights: ComplexNorm, a ModSwish CGU of
    three times the width, a PAM layer, per block; tied embedding and LM head."""
    dim, hid = c["dim"], 3 * c["dim"]

    def prm(*shape, std, mean=0.0):
        return torch.nn.Parameter(_randn(g, *shape, std=std, mean=mean), requires_grad=False)

    def clin(o, i, bias=False):
        return _module(weight_real=prm(o, i, std=(2 * i) ** -0.5), weight_imag=prm(o, i, std=(2 * i) ** -0.5),
                       bias_real=prm(o, std=0.02) if bias else None, bias_imag=prm(o, std=0.02) if bias else None)

    def norm(n):
        return _module(scale=prm(n, std=0.05, mean=1.0), eps=1e-6)

    blocks = []
    for _ in range(c["blocks"]):
        cgu = _module(gate_proj=clin(hid, dim), up_proj=clin(hid, dim), down_proj=clin(dim, hid),
                      act=_module(bias=prm(hid, std=0.1), beta=prm(hid, std=0.1, mean=1.0)))
        blocks.append(_module(norm1=norm(dim), norm2=norm(dim), cgu=cgu, cgu_scale=prm(1, std=0.0, mean=1.0)[0],
                              pam_scale=prm(1, std=0.0, mean=0.1)[0],
                              pam=_pam_module(g, dim, c["H"], c["d"], c["M"], 16, torch.float32)))
    V = c["vocab"]
    return _module(embed=_module(embed_real=_module(weight=prm(V, dim, std=0.02)),
                                 embed_imag=_module(weight=prm(V, dim, std=0.02))),
                   pos_embed=None, embed_norm=norm(dim), output_norm=norm(dim), lm_head_norm=norm(dim),
                   lm_head_proj=clin(dim, dim, bias=True), blocks=blocks)


def _prepare_model(c, g):
    from qllm2_amd.model_decode import ModelDecoder
    model = _model(g, c)
    dec = ModelDecoder(model, n_slots=c["slots"], max_len=8192, dtype=DTYPES[c["dtype"]], graphs=True, graph_bucket=16)
    pos = torch.randint(1, 4096, (c["slots"],), device=DEV, generator=g).tolist()
    slots = [dec.engine.admit(p) for p in pos]
    dec.pool.state.normal_(0.0, 0.01, generator=g)
    live = torch.randperm(c["slots"], device=DEV, generator=g)[:c["live"]].sort().values.tolist()
    host = [slots[i] for i in live]
    return dict(model=model, dec=dec, host=host, slots=torch.tensor(host, dtype=torch.int32, device=DEV),
                ids=torch.randint(0, c["vocab"], (c["live"],), device=DEV, generator=g))


def _prepare_decode(c, g):
    S, G, M, d = c["slots"], c["groups"], c["M"], c["d"]
    state = _randn(g, S, G, M, d, d, 2, std=0.1)
    q, k, v = (_randn(g, S, G, d, 2) for _ in range(3))
    k = _unit(k)
    gamma = torch.sigmoid(_randn(g, S, G, M, mean=3.0))
    rot = None
    if M > 1:
        phase = _randn(g, S, G, M)
        rot = torch.stack([torch.cos(phase), torch.sin(phase)], -1)
    active = torch.randperm(S, device=DEV, generator=g)[:c["live"]].sort().values.to(torch.int32)
    s = dict(state=state, q=q, k=k, v=v, gamma=gamma, rot=rot, active=active, y=torch.zeros_like(q), rope=None, pos=None)
    if c["rope"]:
        from qllm2_amd.decode import build_rope_cache
        s["rope"] = build_rope_cache(4096, d, device=DEV)
        s["pos"] = torch.randint(0, 4096, (S,), device=DEV, generator=g, dtype=torch.int32)
    return s


def prepare(case, seed):
    c, g = case, _gen(seed)
    kind = c["kind"]
    if kind == "scan":
        s = _prepare_scan(c, g)
    elif kind == "layer":
        dt = DTYPES[c["dtype"]]
        mod = _pam_module(g, c["dim"], c["H"], c["d"], c["M"], c["T"], dt)
        x = _randn(g, c["B"], c["T"], c["dim"], 2, dtype=dt)
        s = dict(mod=mod, x=x.requires_grad_(c["grad"]), params=[p for p in mod.parameters()],
                 dy=_randn(g, *x.shape, dtype=dt))
    elif kind == "decode":
        s = _prepare_decode(c, g)
    elif kind == "model":
        s = _prepare_model(c, g)
    elif kind == "ce":
        N, D, V, dt = c["N"], c["D"], c["V"], DTYPES[c["dtype"]]
        w = _randn(g, V, D, std=D ** -0.5, dtype=torch.float32 if c["master"] else dt)
        t = torch.randint(0, V, (N,), device=DEV, generator=g)
        t[torch.rand(N, device=DEV, generator=g) < 0.02] = -100    # padding rows
        s = dict(h=_randn(g, N, D, dtype=dt).requires_grad_(c["grad"]), w=w.requires_grad_(c["grad"]), t=t)
    elif kind == "elementwise":
        dt = DTYPES[c["dtype"]]
        z, up = (_randn(g, c["rows"], c["dim"], 2, dtype=dt) for _ in range(2))
        scale = _randn(g, c["dim"], std=0.05, mean=1.0)
        bias, beta = _randn(g, c["dim"], std=0.1), _randn(g, c["dim"], std=0.1, mean=1.0)
        s = dict(leaves=[x.requires_grad_(c["grad"]) for x in (z, up, scale, bias, beta)],
                 dy=_randn(g, c["rows"], c["dim"], 2, dtype=dt))
    else:
        B, H, T, d, dt = c["B"], c["H"], c["T"], c["d"], DTYPES[c["dtype"]]
        q, k, v = (_randn(g, B, H, T, d, 2) for _ in range(3))
        dy = _randn(g, B, H, T, d, 2, dtype=dt)
        q, k, v = (_unit(q) * math.sqrt(d)).to(dt), _unit(k).to(dt), v.to(dt)
        if kind == "delta":
            gamma = 0.5 + 0.5 * torch.sigmoid(_randn(g, B, H, T, mean=2.0))
            leaves = [q, k, v, gamma, torch.sigmoid(_randn(g, B, H, T))]
        else:
            leaves = [q, k, v, torch.sigmoid(_randn(g, B, H, T, d, mean=3.0))]
        s = dict(leaves=[x.requires_grad_(c["grad"]) for x in leaves], dy=dy)
    s["case"] = c
    return s


# ---------------------------------------------------------------- one pass

def run(state):
    c = state["case"]
    with torch.set_grad_enabled(bool(c.get("grad"))):
        return _RUN[c["kind"]](c, state)


def _with_grads(outs, y, leaves, dy, on):
    if on:
        outs["grads"] = list(torch.autograd.grad(y, leaves, dy))
    return outs


def _run_scan(c, s):
    if c["api"] == "flash":
        from qllm2_amd.flash_pam import flash_pam_chunked_head
        y, st = flash_pam_chunked_head(*s["leaves"], c["d"], c["chunk"])
        return _with_grads({"y": y, "state": st}, [y], s["leaves"], [s["dy"]], c["grad"])
    from qllm2_amd.pam_scan import chunk_for, pam_scan_planar
    L = s["leaves"]
    rot = (L[7], L[8]) if c["M"] > 1 else None
    y_re, y_im, s_re, s_im = pam_scan_planar(*L[:7], q_scale=c["d"] ** -0.5, chunk=chunk_for(c["chunk"], c["T"]), rot=rot)
    return _with_grads({"y": [y_re, y_im], "state": [s_re, s_im]}, [y_re, y_im], L, list(s["dy"]), c["grad"])


def _run_layer(c, s):
    from qllm2_amd import pam_layer
    out, st = pam_layer.forward(s["mod"], s["x"], None, 0)
    return _with_grads({"out": out, "state": st}, [out], [s["x"]] + s["params"], [s["dy"]], c["grad"])


def _run_decode(c, s):
    from qllm2_amd.decode import decode_step
    y = decode_step(s["state"], s["q"], s["k"], s["v"], s["gamma"], active=s["active"], rot=s["rot"],
                    q_scale=c["d"] ** -0.5, out=s["y"], rope=s["rope"], pos=s["pos"])
    return {"y": y, "state": s["state"]}


def _run_model(c, s):
    logits = s["dec"].step(s["ids"], s["slots"], host_slots=s["host"])
    return {"logits": logits, "state": s["dec"].pool.state}


def _run_ce(c, s):
    from qllm2_amd import fused_ce
    if not c["grad"]:
        return {"loss": fused_ce.linear_ce_per_token(s["h"], s["w"], s["t"])}
    loss = fused_ce.fused_linear_cross_entropy(s["h"], s["w"], s["t"])
    return _with_grads({"loss": loss}, [loss], [s["h"], s["w"]], None, True)


def _run_elementwise(c, s):
    from qllm2_amd import triton_kernels as tk
    z, up, scale, bias, beta = s["leaves"]
    y = tk.fused_cgu_gate(tk.fused_complex_norm(z, scale), tk.fused_mod_swish(up, bias, beta))
    return _with_grads({"y": y}, [y], s["leaves"], [s["dy"]], c["grad"])


def _run_delta(c, s):
    from qllm2_amd.pam_delta import forward_delta
    y, st = forward_delta(*s["leaves"], c["d"], chunk=c["chunk"])
    return _with_grads({"y": y, "state": st}, [y], s["leaves"], [s["dy"]], c["grad"])


def _run_perchannel(c, s):
    from qllm2_amd.pam_perchannel import perchannel_chunked
    y, st = perchannel_chunked(*s["leaves"], c["d"], c["chunk"])
    return _with_grads({"y": y, "state": st}, [y], s["leaves"], [s["dy"]], c["grad"])


_RUN = {"scan": _run_scan, "layer": _run_layer, "decode": _run_decode, "model": _run_model, "ce": _run_ce,
        "elementwise": _run_elementwise, "delta": _run_delta, "perchannel": _run_perchannel}


# ---------------------------------------------------------------- work and tolerance

def _scan_flops(B, H, T, d, M):
    """Score and intra read over the causal half of 64-step chunks, carried read
    and state write per state: 8 flops per complex multiply-add."""
    C = min(64, T)
    return B * H * T * (8 * 2 * d * (C + 1) / 2 + M * 8 * 2 * d * d)


def work(case):
    """Bytes: each input read once and each output written once.  Flops: the
    path's products (a backward counts twice its forward)."""
    c = case
    e = {"fp32": 4, "bf16": 2}[c.get("dtype", "fp32")]
    both = 3 if c.get("grad") else 1
    kind = c["kind"]
    if kind in ("scan", "delta", "perchannel"):
        B, H, T, d, M = c["B"], c["H"], c["T"], c["d"], c.get("M", 1)
        plane = B * H * T * d * 2
        ye = 4 if c.get("api") == "planar" else e
        small = {"scan": M * (1 if M == 1 else 3), "delta": 2, "perchannel": d}[kind] * B * H * T * 4
        state = M * B * H * d * d * 2 * (4 if c.get("api") == "planar" else e)
        fwd = 3 * plane * e + small + plane * ye + state
        bwd = 3 * plane * e + small + plane * ye + 3 * plane * e + small
        flops = _scan_flops(B, H, T, d, M)
        if kind == "delta":     # the Gram and query scores, the solve, U's read, the carried terms and the write
            flops = B * H * T * (8 * 4 * d * 65 / 2 + 8 * 3 * d * d)
        return {"bytes": fwd + (bwd if c["grad"] else 0), "flops": flops * both}
    if kind == "layer":
        n, dim, inner, M, H = c["B"] * c["T"], c["dim"], c["H"] * c["d"], c["M"], c["H"]
        w = 2 * dim * inner * 4 + dim * H * (3 + (M if M > 1 else 0))
        gemm = 2 * n * (2 * dim) * (8 * inner) + 2 * n * dim * H * (3 + (M if M > 1 else 0))
        flops = gemm + _scan_flops(c["B"], H, c["T"], c["d"], M)
        fwd = (2 * 2 * n * dim + w) * e + M * c["B"] * H * c["d"] ** 2 * 2 * e
        return {"bytes": fwd + (2 * fwd if c["grad"] else 0), "flops": flops * both}
    if kind == "decode":
        rows = c["live"] * c["groups"]
        return {"bytes": rows * (c["M"] * (16 * c["d"] ** 2 + 4 + (8 if c["M"] > 1 else 0)) + 4 * 8 * c["d"]),
                "flops": rows * c["M"] * 18 * c["d"] ** 2}
    if kind == "model":
        n, dim, hid, L, M, H, V = c["live"], c["dim"], 3 * c["dim"], c["blocks"], c["M"], c["H"], c["vocab"]
        w = L * 2 * (3 * 2 * dim * hid + 4 * 2 * dim * dim) + 2 * 2 * dim * V + 8 * dim * dim
        state = L * n * H * M * 16 * 64 * 64
        flops = n * (w * 2 + L * H * M * 18 * 64 * 64)
        return {"bytes": w * e + state + n * V * 4, "flops": flops}
    if kind == "ce":
        N, D, V = c["N"], c["D"], c["V"]
        we = 4 if c["master"] else e
        return {"bytes": (N * D * e + V * D * we) * (2 if c["grad"] else 1) + 12 * N, "flops": 2 * N * D * V * both}
    n = c["rows"] * c["dim"] * 2
    return {"bytes": n * e * (3 + (3 if c["grad"] else 0)), "flops": n * 20 * both}


def tolerance(case):
    """About four times the distance of these paths from float64 (fp32 5e-7,
    decay gradients 1.3e-6; bf16 3e-3 to 5e-3; a bf16 layer's bias gradients
    8.5e-3; a 16-block bf16 model's logits, where each block's roundings travel
    through those after it, 3.5e-2: the most that can be told apart)."""
    kind = case["kind"]
    if kind == "decode":
        return {"rel": 2e-6}
    if kind == "model":
        return {"rel": 0.03}
    if case["dtype"] == "bf16":
        return {"rel": 0.025 if kind == "layer" else 0.015}
    return {"rel": 1e-5}


# ---------------------------------------------------------------- float64

def _c(x):
    return torch.complex(x[..., 0].double(), x[..., 1].double())


def _r(z):
    return torch.view_as_real(z)


def _pad_chunks(x, C, n, value=0.0):
    """[..., T, d] -> [..., n, C, d] (d kept), padded."""
    T = x.shape[-2]
    x = F.pad(x, (0, 0, 0, n * C - T), value=value)
    return x.reshape(*x.shape[:-2], n, C, x.shape[-1])


def _scan_exact(q, k, v, gamma, rot, scale, C=64):
    """q, k, v complex128 [B,H,T,d], gamma [M,B,H,T], rot complex [M,B,H,T] or
    None -> y [B,H,T,d], final states [M,B,H,d,d]."""
    M, B, H, T = gamma.shape
    n = -(-T // C)
    Q, K, V = (_pad_chunks(torch.view_as_real(x).reshape(B, H, T, -1), C, n).reshape(B, H, n, C, -1, 2) for x in (q, k, v))
    Q, K, V = (torch.view_as_complex(x.contiguous()) for x in (Q, K, V))
    Q = Q * scale
    lg = F.pad(torch.log(gamma + 1e-6), (0, n * C - T)).reshape(M, B, H, n, C)
    L = lg.cumsum(-1)
    D = torch.exp((L.unsqueeze(-1) - L.unsqueeze(-2)).clamp(max=0.0)).tril()
    if rot is None:
        R = torch.ones(M, B, H, n, C, device=q.device, dtype=torch.complex128)
    else:
        R = torch.nn.functional.pad(torch.view_as_real(rot), (0, 0, 0, n * C - T))
        R = torch.view_as_complex(R.reshape(M, B, H, n, C, 2).contiguous())
    A = (Q @ K.conj().transpose(-1, -2)) * (R.unsqueeze(-1) * D).sum(0)
    y = A @ V
    tail = torch.exp((L[..., -1:] - L).clamp(max=0.0))
    dS = (V.unsqueeze(0) * tail.unsqueeze(-1)).transpose(-1, -2) @ K.conj()
    tot, cum = torch.exp(L[..., -1]), torch.exp(L)
    S = torch.zeros(M, B, H, v.shape[-1], q.shape[-1], device=q.device, dtype=torch.complex128)
    ins = []
    for i in range(n):
        ins.append(S)
        S = tot[..., i, None, None] * S + dS[..., i, :, :]
    S_in = torch.stack(ins, 3)
    y = y + ((R * cum).unsqueeze(-1) * (Q @ S_in.transpose(-1, -2))).sum(0)
    return y.reshape(B, H, n * C, -1)[:, :, :T], S


def _delta_exact(q, k, v, gamma, beta, scale, C):
    """The chunked delta write (unit-triangular solve per chunk), complex128."""
    B, H, T, d = q.shape
    n = -(-T // C)

    def cut(z):
        return torch.view_as_complex(_pad_chunks(_r(z).reshape(B, H, T, -1), C, n).reshape(B, H, n, C, -1, 2).contiguous())

    Q, K, V = cut(q) * scale, cut(k), cut(v)
    L = F.pad(torch.log(gamma + 1e-6), (0, n * C - T)).reshape(B, H, n, C).cumsum(-1)
    b = F.pad(beta, (0, n * C - T)).reshape(B, H, n, C, 1)
    D = torch.exp((L.unsqueeze(-1) - L.unsqueeze(-2)).clamp(max=0.0)).tril()
    al = torch.exp(L)
    N = (K @ K.conj().transpose(-1, -2)) * (b * D).tril(-1)
    eye = torch.eye(C, device=q.device, dtype=torch.complex128)
    Ti, P = eye - N, N @ N          # (I + N)^-1 = (I - N)(I + N^2)(I + N^4)...: N is nilpotent
    m = 2
    while m < C:
        Ti, P, m = Ti + Ti @ P, P @ P, 2 * m
    A = (Q @ K.conj().transpose(-1, -2)) * D
    w = (al[..., -1:] / (al + 1e-12)).unsqueeze(-1)
    S = torch.zeros(B, H, d, d, device=q.device, dtype=torch.complex128)
    ys = []
    for i in range(n):
        a_i = al[:, :, i].unsqueeze(-1)
        U = Ti[:, :, i] @ (b[:, :, i] * (V[:, :, i] - a_i * (K[:, :, i] @ S.transpose(-1, -2))))
        ys.append(A[:, :, i] @ U + a_i * (Q[:, :, i] @ S.transpose(-1, -2)))
        S = al[:, :, i, -1, None, None] * S + (w[:, :, i] * U).transpose(-1, -2) @ K[:, :, i].conj()
    return torch.cat(ys, 2)[:, :, :T], S


def _perchannel_exact(q, k, v, gamma, scale, C):
    B, H, T, d = q.shape
    n = -(-T // C)

    def cut(z):
        return torch.view_as_complex(_pad_chunks(_r(z).reshape(B, H, T, -1), C, n).reshape(B, H, n, C, -1, 2).contiguous())

    Q, K, V = cut(q) * scale, cut(k), cut(v)
    L = _pad_chunks(torch.log(gamma.clamp_min(1e-6)), C, n).cumsum(-2).clamp(min=-30.0)
    last = L[..., -1:, :]
    Q, Kf, W = Q * torch.exp(L), K * torch.exp(-L), K * torch.exp(last - L)
    y = ((Q @ Kf.conj().transpose(-1, -2)).tril()) @ V
    dS = V.transpose(-1, -2) @ W.conj()
    S = torch.zeros(B, H, d, d, device=q.device, dtype=torch.complex128)
    ins, tot = [], torch.exp(last)
    for i in range(n):
        ins.append(S)
        S = tot[:, :, i] * S + dS[:, :, i]
    y = y + Q @ torch.stack(ins, 2).transpose(-1, -2)
    return y.reshape(B, H, n * C, d)[:, :, :T], S


def _cabs(z):
    return torch.sqrt(z[..., 0].square() + z[..., 1].square() + 1e-8)


def _clin(m, z):
    """ComplexLinear on [..., dim, 2] in float64."""
    w = torch.complex(m.weight_real.double(), m.weight_imag.double())
    y = torch.complex(z[..., 0], z[..., 1]) @ w.T
    if m.bias_real is not None:
        y = y + torch.complex(m.bias_real.double(), m.bias_imag.double())
    return _r(y)


def _lin(m, x, w=None):
    return x @ m.weight.double().T + m.bias.double()


def _pam_inputs(mod, x, rope):
    """q, k, v complex [B,T,H,d], gamma [M,B,T,H], rot [M,B,T,H] or None, from x
    [B,T,dim,2] float64 and the rotary rows [B or 1,T,d] (complex)."""
    B, T, H, d, M = x.shape[0], x.shape[1], mod.num_heads, mod.head_dim, mod.n_states
    qkv = _clin(mod.qkv_proj, x).reshape(B, T, 3, H, d, 2)
    q, k, v = (torch.complex(qkv[:, :, i, ..., 0], qkv[:, :, i, ..., 1]) for i in range(3))
    q, k = q * rope.unsqueeze(2), k * rope.unsqueeze(2)
    mag = _cabs(x)
    dt = _lin(mod.dt_proj, torch.cat([x[..., 0], x[..., 1]], -1)) + mod.dt_bias.double()
    off = mod.state_dt_offset.double().view(M, 1, 1, 1) if M > 1 else torch.zeros(1, 1, 1, 1, device=x.device)
    p = torch.sigmoid(_lin(mod.protect_gate, mag))
    gamma = torch.exp(-F.softplus(dt + off)) * (1 - p) + p
    rot = None
    if M > 1:
        ph = _lin(mod.phase_proj, mag).reshape(B, T, H, M).permute(3, 0, 1, 2)
        rot = torch.complex(torch.cos(ph), torch.sin(ph))
    return q, k, v * (1 - p).unsqueeze(-1), gamma, rot


def _exact_layer(c, s):
    mod, x = copy.deepcopy(s["mod"]).double(), s["x"].detach().double().requires_grad_(c["grad"])
    B, T, H, d = c["B"], c["T"], c["H"], c["d"]
    q, k, v, gamma, rot = _pam_inputs(mod, x, _c(mod.rope_cache[:T]).unsqueeze(0))
    heads = lambda z: z.transpose(1, 2)  # noqa: E731
    y, S = _scan_exact(heads(q), heads(k), heads(v), gamma.transpose(2, 3), None if rot is None else rot.transpose(2, 3),
                       d ** -0.5)
    out = _clin(mod.o_proj, _r(y.transpose(1, 2).reshape(B, T, H * d)))
    outs = {"out": out, "state": _r(S) if c["M"] > 1 else _r(S[0])}
    return _with_grads(outs, [out], [x] + list(mod.parameters()), [s["dy"].double()], c["grad"])


def _decode_exact(S, q, k, v, gamma, rot, scale):
    """S complex [n,G,M,d,d]; q, k, v [n,G,d]; gamma, rot [n,G,M] -> y, S."""
    S = gamma[..., None, None] * S + (v.unsqueeze(-1) * k.conj().unsqueeze(-2)).unsqueeze(2)
    y = (S @ (q * scale)[:, :, None, :, None])[..., 0]
    return (y if rot is None else y * rot.unsqueeze(-1)).sum(2), S


def _exact_decode(c, s):
    y, state = _c(s["y"]), s["state"].clone()
    act = s["active"].long()
    for part in act.split(32):
        q, k, v = (_c(s[n][part]) for n in "qkv")
        if c["rope"]:
            r = _c(s["rope"][s["pos"][part].long()]).unsqueeze(1)
            q, k = q * r, k * r
        rot = _c(s["rot"][part]) if s["rot"] is not None else None
        yp, Sp = _decode_exact(_c(s["state"][part]), q, k, v, s["gamma"][part].double(), rot, c["d"] ** -0.5)
        y[part], state[part] = yp, _r(Sp).float()
    return {"y": _r(y), "state": state}


def _exact_norm(z, m_scale, eps=1e-6):
    mag = _cabs(z)
    rms = torch.sqrt(mag.square().mean(-1, keepdim=True) + eps)
    return (z / (mag.unsqueeze(-1) + 1e-8)) * ((mag / rms) * m_scale.double()).unsqueeze(-1)


def _exact_act(z, bias, beta):
    mag = _cabs(z)
    return (z / (mag.unsqueeze(-1) + 1e-8)) * (mag * torch.sigmoid(beta.double() * mag + bias.double())).unsqueeze(-1)


def _exact_gate(gate, up):
    mag = _cabs(gate)
    z = torch.complex(gate[..., 0], gate[..., 1]) / (mag + 1e-8) * torch.sigmoid(mag) * torch.complex(up[..., 0], up[..., 1])
    return _r(z)


def _exact_model(c, s):
    m, dec, slots = s["model"], s["dec"], s["slots"].long()
    pool, M = dec.pool, c["M"]
    rope = _c(pool.rope[pool.pos[slots].long()]).unsqueeze(1)               # [n, 1, d]
    x = torch.stack([m.embed.embed_real.weight[s["ids"]], m.embed.embed_imag.weight[s["ids"]]], -1).double()
    x = _exact_norm(x, m.embed_norm.scale)
    for li, b in enumerate(m.blocks):
        h = _exact_norm(x, b.norm1.scale)
        g = _exact_gate(_clin(b.cgu.gate_proj, h), _exact_act(_clin(b.cgu.up_proj, h), b.cgu.act.bias, b.cgu.act.beta))
        x = x + b.cgu_scale.double() * _clin(b.cgu.down_proj, g)
        q, k, v, gamma, rot = _pam_inputs(b.pam, _exact_norm(x, b.norm2.scale).unsqueeze(1), rope)
        at = lambda z: z[:, :, 0].permute(1, 2, 0)  # noqa: E731  [M,n,1,H] -> [n,H,M]
        y, _ = _decode_exact(_c(pool.state[slots, li]), q[:, 0], k[:, 0], v[:, 0], at(gamma),
                             at(rot) if rot is not None else None, c["d"] ** -0.5)
        x = x + b.pam_scale.double() * _clin(b.pam.o_proj, _r(y.reshape(y.shape[0], -1)))
    lm = _exact_norm(_clin(m.lm_head_proj, _exact_norm(x, m.output_norm.scale)), m.lm_head_norm.scale)
    logits = lm[..., 0] @ m.embed.embed_real.weight.double().T + lm[..., 1] @ m.embed.embed_imag.weight.double().T
    return {"logits": logits, "state": None}


def _exact_ce(c, s):
    h, w, t = s["h"].detach().double(), s["w"].detach().double(), s["t"]
    if c["master"]:     # the products run on the weight's bf16 copy
        w = s["w"].detach().to(torch.bfloat16).double()
    dh, dw, loss, ok = torch.zeros_like(h), torch.zeros_like(w), [], t != -100
    denom = ok.sum().double().clamp_min(1)
    for i in range(0, h.shape[0], 2048):
        z, ti, oki = h[i:i + 2048] @ w.T, t[i:i + 2048].clamp_min(0), ok[i:i + 2048].double()
        lse = z.logsumexp(-1)
        loss.append((lse - z.gather(1, ti[:, None])[:, 0]) * oki)
        if c["grad"]:
            z = torch.exp(z - lse[:, None])
            z.scatter_add_(1, ti[:, None], -torch.ones_like(lse)[:, None])
            z *= (oki / denom)[:, None]
            dh[i:i + 2048] = z @ w
            dw += z.T @ h[i:i + 2048]
    loss = torch.cat(loss)
    return {"loss": loss.sum() / denom, "grads": [dh, dw]} if c["grad"] else {"loss": loss}


def exact(case, seed):
    c, s = case, prepare(case, seed)
    kind = c["kind"]
    with torch.set_grad_enabled(bool(c.get("grad"))):
        if kind == "layer":
            return _exact_layer(c, s)
        if kind in ("decode", "model"):
            return {"decode": _exact_decode, "model": _exact_model}[kind](c, s)
        if kind == "ce":
            with torch.no_grad():
                return _exact_ce(c, s)
        L = [x.detach().double().requires_grad_(c["grad"]) for x in s["leaves"]]
        if kind == "elementwise":
            y = _exact_gate(_exact_norm(L[0], L[2]), _exact_act(L[1], L[3], L[4]))
            return _with_grads({"y": y}, [y], L, [s["dy"].double()], c["grad"])
        if kind == "scan" and c["api"] == "planar":
            q, k, v = (torch.complex(L[2 * i], L[2 * i + 1]) for i in range(3))
            rot = torch.complex(L[7], L[8]) if c["M"] > 1 else None
            y, S = _scan_exact(q, k, v, L[6], rot, c["d"] ** -0.5)
            y = [y.real, y.imag]
            return _with_grads({"y": y, "state": [S.real, S.imag]}, y, L, [x.double() for x in s["dy"]], c["grad"])
        q, k, v = (torch.complex(x[..., 0], x[..., 1]) for x in L[:3])
        scale = c["d"] ** -0.5
        if kind == "scan":
            y, S = _scan_exact(q, k, v, L[3].unsqueeze(0), None, scale)
            S = S[0]
        elif kind == "delta":
            y, S = _delta_exact(q, k, v, L[3], L[4], scale, c["chunk"])
        else:
            y, S = _perchannel_exact(q, k, v, L[3], scale, c["chunk"])
        y, S = _r(y), _r(S)
        return _with_grads({"y": y, "state": S}, [y], L, [s["dy"].double()], c["grad"])
