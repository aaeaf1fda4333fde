"""The cases by which this framework's speed is followed: its public entry points at the sizes a
user's program calls them with.

One case is one call (or one call and its backward pass) of

  attention   ``pallas_afa_forward`` (inference) and ``algebraic_flash_attention`` (inference and
              training: forward, then dq, dk, dv), with and without the Cayley rotary tables;
  softmax     ``algebraic_softmax`` over materialised scores, forward and VJP;
  rotate      ``apply_ago_rotations`` of q and k, forward and VJP;
  head        ``fused_linear_oace``: the vocabulary projection with the OACE loss, and its gradients;
  logits      ``fused_oace_softmax_loss``: the OACE loss of given logits, and their gradient.

Everything that a training or serving program keeps between steps (weights, rotary tables, input
buffers) is made by ``prepare``; ``run`` is the step.
"""
import math

import torch

import algebraic_intelligence_amd as A

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
_DEV = torch.device("cuda")


def _named(name, case):
    return {"name": name, **case} if name else case


def _attn(name, mode, B, H, L, D, dtype, causal, rotary, entry="flash"):
    return _named(name, {"kind": "attention", "mode": mode, "batch": B, "heads": H, "seq": L, "head_dim": D,
                         "dtype": dtype, "causal": causal, "rotary": rotary, "entry": entry})


def _softmax(name, rows, cols, dtype):
    return _named(name, {"kind": "softmax", "rows": rows, "cols": cols, "dtype": dtype})


def _head(name, rows, d_model, vocab, dtype, tied):
    return _named(name, {"kind": "head", "rows": rows, "d_model": d_model, "vocab": vocab, "dtype": dtype,
                         "tied": tied})


def listed():
    return [
        # One short fp32 prompt of a few heads: the launch- and latency-bound end, and the shape of
        # the reference's own parity check.
        _attn("attn_prompt_f32", "forward", 1, 4, 256, 64, "fp32", False, False, "pallas"),
        # The headline configuration: one attention layer over a batch of 4096-token sequences,
        # rotary inside the call.
        _attn("attn_forward_4k", "forward", 8, 12, 4096, 64, "bf16", True, True, "pallas"),
        # Serving a batch of prompts whose length is no multiple of any tile, wide heads,
        # bidirectional.
        _attn("attn_forward_ragged", "forward", 3, 8, 1531, 128, "bf16", False, False),
        # The attention layer of the small pilot model (6 heads of 48, 512 tokens) in training.
        _attn("attn_train_pilot", "train", 16, 6, 512, 48, "bf16", True, True),
        # Full precision training of a small model: forward and backward in fp32.
        _attn("attn_train_f32", "train", 32, 4, 1024, 64, "fp32", True, True),
        # Long-context training: 8192 tokens, heads of 128, forward and backward.
        _attn("attn_train_8k", "train", 2, 16, 8192, 128, "bf16", True, False),
        # A-Softmax over the score rows of 2048 keys (the materialised-scores path), training.
        _softmax("softmax_train", 24576, 2048, "bf16"),
        # The same over the scores of a ragged batch, in fp32.
        _softmax("softmax_train_ragged", 12 * 1531, 1531, "fp32"),
        # Rotating q and k of the 125M model's layer (12 heads of 64, 2048 tokens), training.
        {"name": "rotate_train", "kind": "rotate", "batch": 8, "heads": 12, "seq": 2048, "head_dim": 64,
         "dtype": "bf16"},
        # The loss head of a 50257-token vocabulary on 512 rows of a 768-wide model, with gradients.
        _head("head_train", 512, 768, 50257, "bf16", False),
        # The pilot model's head in full precision (288 wide, embedding tied to the head).
        _head("head_train_f32", 512, 288, 50257, "fp32", True),
        # The loss of logits that the program computed itself.
        {"name": "logits_train", "kind": "logits", "rows": 2048, "vocab": 50257, "dtype": "bf16"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _ragged(rng, n, step):
    """n itself (any size) half of the time, otherwise the next multiple of step."""
    return n if rng.random() < 0.5 else max(step, (n + step - 1) // step * step)


def draw(rng):
    kind = rng.choice(["attention", "attention", "attention", "softmax", "rotate", "head", "logits"])
    if kind == "attention":
        dtype = rng.choice(["bf16", "bf16", "fp16", "fp32"])
        mode = rng.choice(["forward", "train"])
        D = rng.choice([32, 48, 64, 64, 96, 128, 128])
        L = _ragged(rng, _log_int(rng, 64, 4096 if dtype == "fp32" else 8192), 128)
        H = rng.choice([4, 6, 8, 12, 16])
        # between one sequence and a batch of 32k tokens
        B = max(1, min(32, _log_int(rng, 256, 32768) // L))
        # no more work than the long-context training step
        while B > 1 and B * H * D * L * L > 2 * 16 * 128 * 8192 * 8192 // 2:
            B //= 2
        return _attn(None, mode, B, H, L, D, dtype, rng.random() < 0.7, rng.random() < 0.5)
    if kind == "softmax":
        cols = _ragged(rng, _log_int(rng, 64, 8192), 64)
        rows = max(16, _log_int(rng, 1 << 16, 1 << 26) // cols)
        return _softmax(None, rows, cols, rng.choice(["bf16", "fp16", "fp32"]))
    if kind == "rotate":
        D = rng.choice([32, 48, 64, 96, 128])
        L = _ragged(rng, _log_int(rng, 64, 8192), 64)
        H = rng.choice([4, 6, 8, 12, 16])
        B = max(1, _log_int(rng, 256, 32768) // L)
        return {"kind": "rotate", "batch": B, "heads": H, "seq": L, "head_dim": D,
                "dtype": rng.choice(["bf16", "fp16", "fp32"])}
    if kind == "head":
        dtype = rng.choice(["bf16", "bf16", "fp32"])
        d = 32 * rng.randint(3, 32)
        V = _ragged(rng, _log_int(rng, 1000, 50257), 64)
        N = _ragged(rng, _log_int(rng, 64, 1024 if dtype == "fp32" else 8192), 64)
        return _head(None, N, d, V, dtype, rng.random() < 0.5)
    V = _ragged(rng, _log_int(rng, 1000, 50257), 64)
    N = max(16, _log_int(rng, 1 << 18, 1 << 27) // V)
    # no fp16: without loss scaling the gradient of a mean over this many rows is below its range
    return {"kind": "logits", "rows": N, "vocab": V, "dtype": rng.choice(["bf16", "fp32"])}


# ------------------------------------------------------------------------------------- inputs
def _gen(seed):
    return torch.Generator(device=_DEV).manual_seed(int(seed))


def _randn(shape, g, dtype, scale=1.0):
    return (torch.randn(shape, generator=g, device=_DEV) * scale).to(dtype)


def _tables(case):
    """Cayley rotary tables in fp32: position m turns pair k by 2 m atan(w_k), w_k = 1/(1 + alpha k)^2."""
    pairs = case["head_dim"] // 2
    alpha = (math.sqrt(10000.0) - 1.0) / max(pairs - 1, 1)
    k = torch.arange(pairs, dtype=torch.float64, device=_DEV)
    m = torch.arange(case["seq"], dtype=torch.float64, device=_DEV)
    ang = 2.0 * m[:, None] * torch.atan(1.0 / (1.0 + alpha * k) ** 2)[None, :]
    return torch.cos(ang).float(), torch.sin(ang).float()


def _inputs(case, seed):
    """The tensors of a case, from the seed alone."""
    g = _gen(seed)
    dt = _DTYPES[case["dtype"]]
    kind = case["kind"]
    if kind == "attention":
        shape = (case["batch"], case["heads"], case["seq"], case["head_dim"])
        # fp16 programs keep their scores small: the weight rho(s)^8 itself is held in fp16, which
        # ends at s = 1.8
        scale = 0.4 if case["dtype"] == "fp16" else 1.0
        x = {"q": _randn(shape, g, dt, scale), "k": _randn(shape, g, dt, scale), "v": _randn(shape, g, dt)}
        if case["mode"] == "train":
            x["g"] = _randn(shape, g, dt)
        return x
    if kind == "softmax":
        shape = (case["rows"], case["cols"])
        return {"x": _randn(shape, g, dt), "g": _randn(shape, g, dt)}
    if kind == "rotate":
        shape = (case["batch"], case["heads"], case["seq"], case["head_dim"])
        return {n: _randn(shape, g, dt) for n in ("q", "k", "gq", "gk")}
    N, V = case["rows"], case["vocab"]
    targets = torch.randint(0, V, (N,), generator=g, device=_DEV)
    if kind == "head":
        d = case["d_model"]
        w_shape = (V, d) if case["tied"] else (d, V)
        # normalised hidden rows, weights of the usual initialisation
        return {"h": _randn((N, d), g, dt), "w": _randn(w_shape, g, dt, 1.0 / math.sqrt(d)), "t": targets}
    return {"z": _randn((N, V), g, dt), "t": targets}


def prepare(case, seed):
    s = {"case": dict(case), **_inputs(case, seed)}
    kind = case["kind"]
    if kind == "attention":
        s["rot"] = A.CayleyRotary(*_tables(case)) if case["rotary"] else None
        if case["mode"] == "train":
            for n in ("q", "k", "v"):
                s[n].requires_grad_(True)
    elif kind == "softmax":
        s["x"].requires_grad_(True)
    elif kind == "rotate":
        s["rot"] = A.CayleyRotary(*_tables(case))
        s["q"].requires_grad_(True)
        s["k"].requires_grad_(True)
    elif kind == "head":
        s["h"].requires_grad_(True)
        s["w"].requires_grad_(True)
    else:
        s["z"].requires_grad_(True)
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "attention":
        if case["entry"] == "pallas":
            return A.pallas_afa_forward(s["q"], s["k"], s["v"], causal=case["causal"], rotary_params=s["rot"])
        out = A.algebraic_flash_attention(s["q"], s["k"], s["v"], causal=case["causal"], rotary_params=s["rot"])
        if case["mode"] != "train":
            return out
        return (out.detach(), *torch.autograd.grad(out, (s["q"], s["k"], s["v"]), s["g"]))
    if kind == "softmax":
        y = A.algebraic_softmax(s["x"])
        return (y.detach(), *torch.autograd.grad(y, s["x"], s["g"]))
    if kind == "rotate":
        qr, kr = A.apply_ago_rotations(s["q"], s["k"], s["rot"])
        return (qr.detach(), kr.detach(), *torch.autograd.grad((qr, kr), (s["q"], s["k"]), (s["gq"], s["gk"])))
    if kind == "head":
        w = s["w"].t() if case["tied"] else s["w"]
        loss = A.fused_linear_oace(s["h"], w, s["t"])
        return (loss.detach(), *torch.autograd.grad(loss, (s["h"], s["w"])))
    loss = A.fused_oace_softmax_loss(s["z"], s["t"])
    return (loss.detach(), *torch.autograd.grad(loss, s["z"]))


def work(case):
    es = 4 if case["dtype"] == "fp32" else 2
    kind = case["kind"]
    if kind == "attention":
        L, D = case["seq"], case["head_dim"]
        bh = case["batch"] * case["heads"]
        pairs = L * (L + 1) // 2 if case["causal"] else L * L
        tables = 4 * L * D if case["rotary"] else 0
        n = bh * L * D * es
        if case["mode"] == "train":
            return {"bytes": 8 * n + tables, "flops": 14 * bh * D * pairs}
        return {"bytes": 4 * n + tables, "flops": 4 * bh * D * pairs}
    if kind == "softmax":
        n = case["rows"] * case["cols"]
        return {"bytes": 4 * n * es, "flops": 30 * n}
    if kind == "rotate":
        n = case["batch"] * case["heads"] * case["seq"] * case["head_dim"]
        return {"bytes": 8 * n * es + 4 * case["seq"] * case["head_dim"], "flops": 12 * n}
    N, V = case["rows"], case["vocab"]
    if kind == "head":
        d = case["d_model"]
        return {"bytes": 2 * (N * d + d * V) * es + 8 * N, "flops": 6 * N * d * V}
    return {"bytes": 2 * N * V * es + 8 * N, "flops": 40 * N * V}


def tolerance(case):
    """About four times the largest error against 64 bits that was measured over the ranges."""
    kind, dtype = case["kind"], case["dtype"]
    if dtype == "bf16":
        # with rotary tables q and k are rounded once more after the rotation, before rho^8
        return {"rel": (3e-2 if case["rotary"] else 1.3e-2) if kind == "attention" else 1e-2}
    if dtype == "fp16":
        return {"rel": 3e-3 if kind == "attention" else 1.2e-3}
    return {"rel": {"attention": 5e-6, "softmax": 2e-6, "rotate": 2e-7, "head": 1.6e-5, "logits": 1e-6}[kind]}


# -------------------------------------------------------------------------- 64-bit restatement
def _rho8(s):
    """rho(s)^8 and r = 1/sqrt(1 + s^2), rho = s + sqrt(1 + s^2), without cancellation."""
    t = torch.sqrt(1.0 + s * s)
    rho = torch.where(s < 0, 1.0 / (t + s.abs()), t + s)
    return rho ** 8, 1.0 / t


def _rot(x, c, s):
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack((c * a - s * b, s * a + c * b), dim=-1).reshape(x.shape)


def _exact_attention(case, x):
    B, H, L, D = (case[n] for n in ("batch", "heads", "seq", "head_dim"))
    scale, sink = 1.0 / math.sqrt(D), 0.5
    train = case["mode"] == "train"
    c, s = (t.double() for t in _tables(case)) if case["rotary"] else (None, None)
    outs = [torch.empty((B, H, L, D), dtype=torch.float64, device=_DEV) for _ in range(4 if train else 1)]
    mask = torch.ones((L, L), dtype=torch.bool, device=_DEV).tril() if case["causal"] else None
    for b in range(B):
        for h in range(H):
            q, k, v = (x[n][b, h].detach().double() for n in ("q", "k", "v"))
            if c is not None:
                q, k = _rot(q, c, s), _rot(k, c, s)
            S = q @ k.t() * scale
            w, r = _rho8(S)
            if mask is not None:
                w = w * mask
            d = w.sum(-1, keepdim=True) + sink
            p = w / d
            out = p @ v
            outs[0][b, h] = out
            if train:
                g = x["g"][b, h].double()
                dp = g @ v.t()
                ds = 8.0 * r * p * (dp - (g * out).sum(-1, keepdim=True)) * scale
                dq, dk = ds @ k, ds.t() @ q
                if c is not None:
                    dq, dk = _rot(dq, c, -s), _rot(dk, c, -s)
                outs[1][b, h], outs[2][b, h], outs[3][b, h] = dq, dk, p.t() @ g
    return tuple(outs) if train else outs[0]


def _octic_xent(z, t, eps, gamma):
    """Mean loss and dz of the OACE of logits z (rows, vocab) in 64 bits."""
    N, V = z.shape
    tau = torch.rsqrt((z * z).mean(-1, keepdim=True) + eps)
    x = z * tau
    k8, r = _rho8(x)
    S = k8.sum(-1, keepdim=True)
    p = k8 / S
    pt = p.gather(1, t[:, None])
    p78 = p ** 0.875
    loss = gamma * (8.0 * pt ** -0.125 + 8.0 / 7.0 * p78.sum(-1, keepdim=True) - 64.0 / 7.0)
    # d loss / d p, through p = k8 / S with d k8 / d x = 8 r k8, then x = tau z
    dp = gamma * p ** -0.125
    dp.scatter_add_(1, t[:, None], -gamma * pt ** -1.125)
    dx = 8.0 * r * p * (dp - (dp * p).sum(-1, keepdim=True)) / N
    dz = tau * (dx - x * (dx * x).mean(-1, keepdim=True))
    return loss.mean(), dz


def exact(case, seed):
    x = _inputs(case, seed)
    kind = case["kind"]
    if kind == "attention":
        return _exact_attention(case, x)
    if kind == "softmax":
        ys, dxs = [], []
        for xs, gs in zip(x["x"].split(4096), x["g"].split(4096)):
            z, g = xs.double(), gs.double()
            tau = torch.rsqrt((z * z).mean(-1, keepdim=True) + 1e-5)
            y = z * tau
            w, r = _rho8(y)
            p = w / (w.sum(-1, keepdim=True) + 0.5)
            ng = 8.0 * r * p * (g - (p * g).sum(-1, keepdim=True))
            ys.append(p)
            dxs.append(tau * (ng - (ng * y).mean(-1, keepdim=True) * y))
        return torch.cat(ys), torch.cat(dxs)
    if kind == "rotate":
        # the entry point takes the tables in x's type
        c, s = (t.to(_DTYPES[case["dtype"]]).double() for t in _tables(case))
        return tuple(_rot(x[n].double(), c, t) for n, t in (("q", s), ("k", s), ("gq", -s), ("gk", -s)))
    t = x["t"]
    if kind == "head":
        h, w = x["h"].double(), x["w"].double()
        if case["tied"]:
            w = w.t()
        loss, dh, dw = 0.0, [], torch.zeros_like(w)
        N = h.shape[0]
        for hs, ts in zip(h.split(512), t.split(512)):
            part, dz = _octic_xent(hs @ w, ts, 100.0, 2.0)
            share = hs.shape[0] / N
            loss = loss + part * share
            dz = dz * share
            dh.append(dz @ w.t())
            dw += hs.t() @ dz
        return loss, torch.cat(dh), dw.t() if case["tied"] else dw
    N = x["z"].shape[0]
    loss, dzs = 0.0, []
    for zs, ts in zip(x["z"].split(512), t.split(512)):
        part, dz = _octic_xent(zs.double(), ts, 100.0, 2.0)
        loss = loss + part * (zs.shape[0] / N)
        dzs.append(dz * (zs.shape[0] / N))
    return loss, torch.cat(dzs)
