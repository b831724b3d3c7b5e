"""Workloads of the Continuum Attention framework, through its public entry points.

Each case is one call (or one forward and backward) that a program using this
framework makes: the operator over its range of sizes, head dims and element
types, the materialised-weight API, the decoder's attention layer, its
residual-add RMSNorm and the whole CA-S decoder.  ``run`` makes the call,
``exact`` computes the same results in float64 with plain torch.
"""
import importlib
import math

import torch

ca = importlib.import_module("continuum-attention_amd")

_DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
_ESIZE = {"f32": 4, "bf16": 2, "f16": 2}

# [B, H, T, D] operator sizes beyond which a drawn case would cost more than
# the largest listed one: causal pairs x head dim
_MAX_PAIR_DIMS = 16 * 8192 * 8192 // 2 * 64


def listed():
    return [
        # the smallest operator call, forward and backward: a unit-test-sized
        # model's layer, where launches and host work count
        {"name": "op_f32_tiny", "kind": "op", "B": 1, "H": 2, "T": 64, "D": 16, "dtype": "f32",
         "backward": True, "keys": "normal"},
        # one attention layer of the CA-P TinyLM decoder at its training batch
        {"name": "op_f32_short", "kind": "op", "B": 16, "H": 4, "T": 512, "D": 64, "dtype": "f32",
         "backward": True, "keys": "normal"},
        # the headline operator size: forward and backward of two sequences
        {"name": "op_f32", "kind": "op", "B": 2, "H": 16, "T": 2048, "D": 64, "dtype": "f32",
         "backward": True, "keys": "normal"},
        # the long-context size: half the heads have near-duplicate neighbouring
        # keys, half have large score differences
        {"name": "op_f32_long", "kind": "op", "B": 1, "H": 16, "T": 8192, "D": 64, "dtype": "f32",
         "backward": True, "keys": "mixed"},
        # a training batch in bf16 of ragged length
        {"name": "op_bf16_ragged", "kind": "op", "B": 4, "H": 16, "T": 1001, "D": 64, "dtype": "bf16",
         "backward": True, "keys": "normal"},
        # forward only (inference, prompt scoring) in fp16, the reference
        # decoder's default half type
        {"name": "op_f16_forward", "kind": "op", "B": 1, "H": 16, "T": 2048, "D": 64, "dtype": "f16",
         "backward": False, "keys": "normal"},
        # the largest fused head dim, odd length
        {"name": "op_f32_d128", "kind": "op", "B": 1, "H": 8, "T": 1537, "D": 128, "dtype": "f32",
         "backward": True, "keys": "normal"},
        # a head dim that is no power of two (width 640 over 8 heads)
        {"name": "op_f32_d80", "kind": "op", "B": 2, "H": 8, "T": 768, "D": 80, "dtype": "f32",
         "backward": True, "keys": "normal"},
        # the CA-S decoder's attention between its projections, as bf16
        # autocast calls it: RoPE, operator, token-major gradients
        {"name": "layer_bf16", "kind": "layer", "B": 1, "H": 16, "T": 2048, "D": 64, "dtype": "bf16"},
        # materialised weights of a batch of heads and their score gradient
        # (weight diagnostics, the 'hip_weights' backend)
        {"name": "weights_f32", "kind": "weights", "N": 64, "T": 512},
        # a decoder block's residual add + RMSNorm at a training batch
        {"name": "add_norm_bf16", "kind": "norm", "rows": 8192, "C": 1024, "dtype": "bf16"},
        # the whole CA-S decoder (101M parameters) at its training length:
        # bf16 autocast forward, loss and backward
        {"name": "decoder_bf16", "kind": "decoder", "B": 1, "T": 2048},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["op", "op", "op", "op", "op", "layer", "weights", "norm"])
    if kind == "norm":
        return {"kind": "norm", "rows": _log_int(rng, 64, 16384), "C": 4 * _log_int(rng, 16, 1024),
                "dtype": rng.choice(["f32", "bf16", "f16"])}
    if kind == "weights":
        T = _log_int(rng, 16, 1536)
        return {"kind": "weights", "N": max(1, min(_log_int(rng, 1, 128), (1 << 25) // (T * T))), "T": T}
    D = rng.choice([64, 64, 64, 128, 32, 16, 8, 80, 96, 48, 24])
    if kind == "layer" and D not in (16, 32, 64, 128):
        D = 64
    # head dims without a power of two stay at moderate lengths
    T = _log_int(rng, 16, 4096 if D in (8, 16, 32, 64, 128) else 1024)
    slices = max(1, min(_log_int(rng, 1, 64), _MAX_PAIR_DIMS // (2 * T * T * max(D, 64))))
    B = rng.choice([b for b in (1, 2, 3, 4) if b <= slices])
    case = {"kind": kind, "B": B, "H": slices // B, "T": T, "D": D,
            "dtype": rng.choice(["f32", "bf16", "f16"])}
    if kind == "op":
        case.update(backward=rng.random() < 0.7, keys=rng.choice(["normal", "normal", "mixed"]))
    return case


# ---- inputs -------------------------------------------------------------------


def _keys(case, gen):
    B, H, T, D = case["B"], case["H"], case["T"], case["D"]
    k = torch.randn(B, H, T, D, generator=gen, device="cuda")
    if case.get("keys") == "mixed":
        # slowly varying keys in the first half of the heads, large ones in the rest
        n = H // 2
        if n:
            step = 1e-4 * k[:, :n, 1:]
            k[:, :n, 1:] = k[:, :n, :1] + torch.cumsum(step, 2)
        k[:, n:] *= 4.0
    return k


def _op_inputs(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    B, H, T, D = case["B"], case["H"], case["T"], case["D"]
    dt = _DTYPES[case["dtype"]]
    k = _keys(case, gen).to(dt)
    q, v, dy = (torch.randn(B, H, T, D, generator=gen, device="cuda").to(dt) for _ in range(3))
    log_gain = 0.1 * torch.randn(H, generator=gen, device="cuda")
    return q, k, v, log_gain, dy


def _layer_inputs(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    B, H, T, D = case["B"], case["H"], case["T"], case["D"]
    dt = _DTYPES[case["dtype"]]
    qkv = torch.randn(B, T, 3 * H * D, generator=gen, device="cuda").to(dt)
    log_gain = 0.1 * torch.randn(H, generator=gen, device="cuda")
    dy = torch.randn(B, T, H * D, generator=gen, device="cuda").to(dt)
    return qkv, log_gain, dy


def _weights_inputs(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    logits = 1.5 * torch.randn(case["N"], case["T"], case["T"], generator=gen, device="cuda")
    return logits, torch.randn(logits.shape, generator=gen, device="cuda")


def _norm_inputs(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    N, C = case["rows"], case["C"]
    dt = _DTYPES[case["dtype"]]
    x = torch.randn(N, C, generator=gen, device="cuda")
    res = (0.5 * torch.randn(N, C, generator=gen, device="cuda")).to(dt)
    w = 1.0 + 0.1 * torch.randn(C, generator=gen, device="cuda")
    dsum = torch.randn(N, C, generator=gen, device="cuda")
    dy = torch.randn(N, C, generator=gen, device="cuda").to(dt)
    return x, res, w, dsum, dy


def _decoder(case, seed):
    cfg = ca.decoder.ContinuumDecoderConfig()
    torch.manual_seed(seed)
    with torch.device("cuda"):
        model = ca.decoder.ContinuumDecoderLM(cfg)
    gen = torch.Generator(device="cuda").manual_seed(seed)
    ids = torch.randint(0, cfg.vocab_size, (case["B"], case["T"]), generator=gen, device="cuda")
    return model, ids


def prepare(case, seed):
    kind = case["kind"]
    state = {"case": case}
    if kind == "op":
        *leaves, dy = _op_inputs(case, seed)
        state["leaves"] = [t.requires_grad_(case["backward"]) for t in leaves]
        state["dy"] = dy
    elif kind == "layer":
        qkv, log_gain, dy = _layer_inputs(case, seed)
        state["leaves"] = [qkv.requires_grad_(), log_gain.requires_grad_()]
        state["dy"] = dy
    elif kind == "weights":
        logits, gw = _weights_inputs(case, seed)
        state["logits"], state["gw"] = logits.requires_grad_(), gw
    elif kind == "norm":
        x, res, w, dsum, dy = _norm_inputs(case, seed)
        norm = ca.decoder.RMSNorm(case["C"]).to("cuda")
        with torch.no_grad():
            norm.weight.copy_(w)
        state.update(norm=norm, x=x.requires_grad_(), res=res.requires_grad_(), dsum=dsum, dy=dy)
    else:
        model, ids = _decoder(case, seed)
        state.update(model=model, ids=ids, opt=ca.decoder.build_fused_adamw(model))
    return state


# ---- one pass -----------------------------------------------------------------


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "op":
        if not case["backward"]:
            with torch.no_grad():
                return ca.continuum_attention(*state["leaves"])
        y = ca.continuum_attention(*state["leaves"])
        return [y.detach(), *torch.autograd.grad(y, state["leaves"], state["dy"])]
    if kind == "layer":
        qkv, log_gain = state["leaves"]
        y = ca.decoder.rope_continuum_attention(qkv, log_gain, 10000.0, case["H"])
        return [y.detach(), *torch.autograd.grad(y, state["leaves"], state["dy"])]
    if kind == "weights":
        w = ca.continuous_attention_weights(state["logits"])
        return [w.detach(), *torch.autograd.grad(w, state["logits"], state["gw"])]
    if kind == "norm":
        norm, x, res = state["norm"], state["x"], state["res"]
        dt = _DTYPES[case["dtype"]]
        with torch.autocast("cuda", dtype=dt, enabled=dt != torch.float32):
            s, y = norm.add_and_norm(x, res)
        grads = torch.autograd.grad([s, y], [x, res, norm.weight], [state["dsum"], state["dy"]])
        return [s.detach(), y.detach(), *grads]
    model, ids, opt = state["model"], state["ids"], state["opt"]
    opt.zero_grad()
    with torch.autocast("cuda", dtype=torch.bfloat16):
        out = model(ids, targets=ids)
    out["loss"].backward()
    return [out["logits"].detach(), out["loss"].detach(), *opt.grads()]


# ---- what a pass cannot do without ----------------------------------------------


def _pairs(case):
    return case["B"] * case["H"] * case["T"] * (case["T"] + 1) // 2


def work(case):
    kind = case["kind"]
    if kind == "op":
        n = case["B"] * case["H"] * case["T"] * case["D"] * _ESIZE[case["dtype"]]
        if not case["backward"]:
            return {"bytes": 4 * n, "flops": 4 * case["D"] * _pairs(case)}
        return {"bytes": 8 * n, "flops": 14 * case["D"] * _pairs(case)}
    if kind == "layer":
        n = case["B"] * case["H"] * case["T"] * case["D"] * _ESIZE[case["dtype"]]
        return {"bytes": 8 * n, "flops": 14 * case["D"] * _pairs(case)}
    if kind == "weights":
        n = case["N"] * case["T"] * case["T"]
        # scores and weight gradient read (visible half), weights and score
        # gradient written whole
        return {"bytes": 4 * n + 4 * 2 * n, "flops": 40 * n // 2}
    if kind == "norm":
        n, e = case["rows"] * case["C"], _ESIZE[case["dtype"]]
        # x, res, dsum, dy read; s, y, dx, dres written
        return {"bytes": n * (4 + e + 4 + e) + n * (4 + e + 4 + e), "flops": 16 * n}
    cfg = ca.decoder.ContinuumDecoderConfig()
    C, T, L = cfg.d_model, case["T"], cfg.n_layers
    params = 12 * C * C * L + 2 * C * cfg.vocab_size
    pairs = case["B"] * cfg.n_heads * T * (T + 1) // 2
    return {"bytes": 2 * 2 * params + 2 * params + 4 * case["B"] * T * cfg.vocab_size,
            "flops": 6 * case["B"] * T * (params - C * cfg.vocab_size) + L * 14 * (C // cfg.n_heads) * pairs}


def tolerance(case):
    kind = case["kind"]
    if kind in ("op", "layer"):
        # f32: outputs and gradients 1e-7 to 3e-6 from float64; the gain
        # gradient, a sum of cancelling terms, 4e-6 (3.5e-5 with mixed keys)
        f32 = 2e-4 if case.get("keys") == "mixed" else 5e-5
        return {"rel": {"f32": f32, "bf16": 1e-2, "f16": 2e-3}[case["dtype"]]}
    if kind == "weights":
        return {"rel": 5e-6}
    if kind == "norm":
        return {"rel": {"f32": 2e-6, "bf16": 1e-2, "f16": 2e-3}[case["dtype"]]}
    return {"rel": 8e-2}


# ---- the same in float64 --------------------------------------------------------


def _weights64(s, start):
    """Exact CA weights [n, R, K] of rows ``start ..`` from float64 scores: the
    integral of exp over piecewise-linear scores against each key's hat
    function, half-token caps at key 0 and at the query, rows normalised."""
    R, K = s.shape[-2:]
    i = start + torch.arange(R, device=s.device)[:, None]
    j = torch.arange(K, device=s.device)[None, :]
    vis = j <= i
    m = torch.where(vis, s, -torch.inf).amax(-1, keepdim=True).detach()
    p = torch.where(vis, torch.exp(torch.where(vis, s - m, 0.0)), 0.0)
    w = 0.5 * p * (j == 0) + 0.5 * p * (j == i)
    if K == 1:
        return w / w.sum(-1, keepdim=True)
    seg = vis[:, 1:]  # segment (j, j + 1) is visible when its right key is
    pl, pr = p[..., :-1], p[..., 1:]
    x = torch.where(seg, s[..., 1:] - s[..., :-1], 0.0)
    small = x.abs() < 0.5
    xs = torch.where(small, x, 0.0)
    xc = torch.where(small, 1.0, x)

    def j1(t):  # int_0^1 u exp(t u) du
        acc = torch.full_like(t, 1.0 / (math.factorial(15) * 17))
        for n in range(14, -1, -1):
            acc = acc * t + 1.0 / (math.factorial(n) * (n + 2))
        return acc

    mean = (pr - pl) / xc
    right_c = (pr - mean) / xc
    right = torch.where(small, pl * j1(xs), right_c) * seg
    left = torch.where(small, pr * j1(-xs), mean - right_c) * seg
    zero = torch.zeros_like(w[..., :1])
    w = w + torch.cat([left, zero], -1) + torch.cat([zero, right], -1)
    return w / w.sum(-1, keepdim=True)


def _attention64(q, k, v, gain, dy=None):
    """Operator on float64 [N, T, D] slices with per-slice score scale
    ``gain`` [N] (dL/dscale is returned for it); gradients when dy is given."""
    N, T, D = q.shape
    y = torch.empty_like(q)
    grads = None if dy is None else [torch.zeros_like(t) for t in (q, k, v, gain)]
    rows = max(1, min(T, 512 if T > 4096 else 1024))
    for n0 in range(0, N, max(1, (1 << 22) // (rows * T))):
        sl = slice(n0, n0 + max(1, (1 << 22) // (rows * T)))
        for a in range(0, T, rows):
            b = min(T, a + rows)
            with torch.set_grad_enabled(dy is not None):
                leaves = [t.detach().requires_grad_(dy is not None)
                          for t in (q[sl, a:b], k[sl, :b], v[sl, :b], gain[sl])]
                s = torch.bmm(leaves[0], leaves[1].transpose(1, 2)) * leaves[3][:, None, None]
                o = torch.bmm(_weights64(s, a), leaves[2])
            y[sl, a:b] = o.detach()
            if dy is not None:
                g = torch.autograd.grad(o, leaves, dy[sl, a:b])
                grads[0][sl, a:b] = g[0]
                grads[1][sl, :b] += g[1]
                grads[2][sl, :b] += g[2]
                grads[3][sl] += g[3]
    return y, grads


def _operator64(q, k, v, log_gain, dy=None):
    """[B, H, T, D] float64 operator: y and, with dy, (dq, dk, dv, dlog_gain)."""
    B, H, T, D = q.shape
    c = (log_gain.double().exp() * D ** -0.5).repeat(B)
    flat = [t.reshape(B * H, T, D) for t in (q, k, v)]
    y, g = _attention64(*flat, c, None if dy is None else dy.reshape(B * H, T, D))
    if dy is None:
        return y.view(B, H, T, D), None
    dg = (g[3] * c).view(B, H).sum(0)
    return y.view(B, H, T, D), [t.view(B, H, T, D) for t in g[:3]] + [dg]


def _rope_table(T, D, theta, dtype):
    freq = 1.0 / (theta ** (torch.arange(0, D, 2, device="cuda", dtype=torch.float32) / D))
    phase = torch.outer(torch.arange(T, device="cuda", dtype=torch.float32), freq)
    return (phase.cos().repeat_interleave(2, -1).to(dtype),
            phase.sin().repeat_interleave(2, -1).to(dtype))


def _pairs_rotated(t):
    p = t.unflatten(-1, (-1, 2))
    return torch.stack((-p[..., 1], p[..., 0]), -1).flatten(-2)


class _Attention64(torch.autograd.Function):
    @staticmethod
    def forward(ctx, q, k, v, log_gain):
        ctx.save_for_backward(q, k, v, log_gain)
        return _operator64(q, k, v, log_gain)[0]

    @staticmethod
    def backward(ctx, dy):
        return tuple(_operator64(*ctx.saved_tensors, dy)[1])


def _decoder64(model, ids):
    """Logits, loss and parameter gradients of the decoder in float64."""
    cfg = model.cfg
    P = {n: p.detach().double().requires_grad_() for n, p in model.named_parameters()}
    B, T = ids.shape
    H, D = cfg.n_heads, cfg.d_model // cfg.n_heads
    cos, sin = _rope_table(T, D, cfg.rope_theta, torch.float64)

    def norm(x, name):
        return P[name] * x * torch.rsqrt(x.square().mean(-1, keepdim=True) + cfg.eps)

    x = torch.nn.functional.embedding(ids, P["byte_emb.weight"])
    for n in range(cfg.n_layers):
        b = "blocks.%d." % n
        qkv = norm(x, b + "norm1.weight") @ P[b + "attn.qkv.weight"].t()
        q, k, v = qkv.view(B, T, 3, H, D).permute(2, 0, 3, 1, 4).unbind(0)
        q = q * cos + _pairs_rotated(q) * sin
        k = k * cos + _pairs_rotated(k) * sin
        a = _Attention64.apply(q, k, v, P[b + "attn.log_qk_gain"])
        x = x + a.transpose(1, 2).reshape(B, T, -1) @ P[b + "attn.out.weight"].t()
        h = norm(x, b + "norm2.weight") @ P[b + "mlp.fc1.weight"].t()
        h = torch.nn.functional.gelu(h, approximate="tanh")
        x = x + h @ P[b + "mlp.fc2.weight"].t()
    logits = norm(x, "norm_f.weight") @ P["lm_head.weight"].t()
    loss = torch.nn.functional.cross_entropy(logits[:, :-1].reshape(-1, cfg.vocab_size),
                                             ids[:, 1:].reshape(-1))
    grads = torch.autograd.grad(loss, list(P.values()))
    return [logits.detach(), loss.detach(), *grads]


def exact(case, seed):
    kind = case["kind"]
    if kind == "op":
        q, k, v, log_gain, dy = _op_inputs(case, seed)
        y, g = _operator64(q.double(), k.double(), v.double(), log_gain.double(),
                           dy.double() if case["backward"] else None)
        return [y, *g] if case["backward"] else y
    if kind == "layer":
        B, H, T, D = case["B"], case["H"], case["T"], case["D"]
        dt = _DTYPES[case["dtype"]]
        qkv, log_gain, dy = _layer_inputs(case, seed)
        cos, sin = _rope_table(T, D, 10000.0, dt)
        q, k, v = qkv.view(B, T, 3, H, D).permute(2, 0, 3, 1, 4).unbind(0)
        # the rotation is defined in the operands' type
        q = q * cos + _pairs_rotated(q) * sin
        k = k * cos + _pairs_rotated(k) * sin
        y, (dq, dk, dv, dg) = _operator64(q.double(), k.double(), v.double(), log_gain.double(),
                                          dy.view(B, T, H, D).transpose(1, 2).double())
        cos, sin = cos.double(), sin.double()
        dq, dk = (t * cos - _pairs_rotated(t * sin) for t in (dq, dk))
        dqkv = torch.stack((dq, dk, dv)).permute(1, 3, 0, 2, 4).reshape(B, T, 3 * H * D)
        return [y.transpose(1, 2).reshape(B, T, H * D), dqkv, dg]
    if kind == "weights":
        logits, gw = _weights_inputs(case, seed)
        T = case["T"]
        w, ds = [], []
        n = max(1, (1 << 22) // (T * T))
        for a in range(0, case["N"], n):
            s = logits[a:a + n].double().requires_grad_()
            o = _weights64(s, 0)
            w.append(o.detach())
            ds.append(torch.autograd.grad(o, s, gw[a:a + n].double())[0])
        return [torch.cat(w), torch.cat(ds)]
    if kind == "norm":
        x, res, w, dsum, dy = (t.double() for t in _norm_inputs(case, seed))
        x.requires_grad_()
        w.requires_grad_()
        s = x + res
        y = w * s * torch.rsqrt(s.square().mean(-1, keepdim=True) + 1e-6)
        dx, dw = torch.autograd.grad([s, y], [x, w], [dsum, dy])
        return [s.detach(), y.detach(), dx, dx, dw]
    model, ids = _decoder(case, seed)
    return _decoder64(model, ids)
