"""Performance cases of the Born attention entry points on one GPU.

A case is one call of a public entry point as a program makes it: the
attention alone (``flash_born_attention``, ``flash_purified_born_attention``)
on contiguous ``(B, H, T, D)`` heads, or the layer's data flow
(``flash_born_attention_qk_prologue`` on the ``(B, T, H, D)`` projection
outputs viewed as heads, with the heads merged again behind it).  ``train``
cases run the forward and the backward and return the output and every
gradient; the others run the forward alone, as generation and evaluation do.

Keys of a case: ``op`` ("born", "purified" or "layer"), ``B``, ``H``, ``T``,
``D``, ``dtype``, ``train``, ``causal``, ``window`` (keys, 0 for none), ``docs``
(mean document length in tokens, 0 for none) and ``scale`` ("float", as a
layer with a fixed temperature passes it, or "heads", one learnable value per
head).
"""

from __future__ import annotations

import math

import torch

import quantumdlblocks_amd as qdl

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
SCALE = 8.0        # sqrt(64), and the purified layers' default gamma
TAU = 0.0625       # the purified layers' defaults
EPS_BASE = 0.05
SHARED = 0.6       # length of the rows' shared part over that of their own
EOT = 50256
CHUNK = 1 << 26    # elements of one T x T float64 temporary in exact()


def _case(op, B, H, T, D, dtype="bf16", train=False, causal=True, window=0, docs=0, scale="float", name=None):
    c = dict(op=op, B=B, H=H, T=T, D=D, dtype=dtype, train=train, causal=causal, window=window, docs=docs, scale=scale)
    return dict(c, name=name) if name else c


def listed():
    return [
        # The shortest useful call: one prompt of a small model.  Latency and launches.
        _case("born", 1, 4, 256, 64, name="prompt_1x4x256"),
        # Prompts of a 16-head model for generation: two sequences of a length
        # that is a multiple of nothing.
        _case("born", 2, 16, 1531, 64, name="prompts_2x16x1531"),
        # The forward benchmark: evaluation batches of a 16-head, 1024-token model.
        _case("born", 16, 16, 1024, 64, name="eval_16x16x1024"),
        # The training benchmark: one attention layer's step at 2048 tokens.
        _case("born", 16, 16, 2048, 64, train=True, name="train_16x16x2048"),
        # Pre-training on packed documents (mean 512 tokens in 8192), a
        # learnable temperature per head.
        _case("born", 4, 16, 8192, 64, train=True, docs=512, scale="heads", name="packed_train_4x16x8192"),
        # The wavelet models' layers: purified attention with a 384-key window
        # over packed documents.
        _case("purified", 4, 16, 8192, 64, train=True, window=384, docs=512, scale="heads",
              name="purified_packed_4x16x8192"),
        # The layer's data flow (RoPE, normalisation, attention, head merge) on
        # projection outputs, at the layer benchmark's batch and heads.
        _case("layer", 8, 16, 1024, 64, train=True, name="layer_train_8x16x1024"),
        # A unit-test-sized model in fp32: four heads of 32, 64 tokens.
        _case("born", 2, 4, 64, 32, dtype="fp32", train=True, scale="heads", name="small_train_fp32_2x4x64"),
        # Training without autocast: fp32 at an odd length.
        _case("born", 2, 8, 1000, 64, dtype="fp32", train=True, name="train_fp32_2x8x1000"),
        # Long-context fine-tuning of one sequence at head dim 128.
        _case("born", 1, 8, 4096, 128, train=True, name="long_train_1x8x4096_d128"),
        # fp16 purified attention at a padded head dim and a ragged length.
        _case("purified", 3, 6, 1100, 96, dtype="fp16", train=True, name="purified_fp16_3x6x1100_d96"),
        # Few wide heads: head dim 256, a batch of 1024-token prompts.
        _case("born", 4, 4, 1024, 256, name="wide_4x4x1024_d256"),
    ]


def _pairs(case):
    """Visible (query, key) pairs of one head (expected, with documents)."""
    T, w = case["T"], case["window"]
    keep = 1.0 - 1.0 / case["docs"] if case["docs"] else 1.0

    def side(n):  # sum of keep^l over l < n, the visible keys at lags 0 .. n - 1
        return n if keep == 1.0 else (1.0 - keep ** n) / (1.0 - keep)

    total = 0.0
    for i in range(T):
        total += side(min(i + 1, w) if w else i + 1)
        if not case["causal"]:
            total += side(T - i) - 1.0
    return total


def _cost(case):
    """Rough cost in bf16 Born flops, to keep drawn cases below the largest listed one."""
    pairs = case["T"] * (case["T"] + 1) / 2 * (1 if case["causal"] else 2)
    if case["window"]:
        pairs = min(pairs, case["T"] * case["window"] * (1 if case["causal"] else 2))
    f = 4.0 * max(case["D"], 64) * pairs * case["B"] * case["H"] * (3.5 if case["train"] else 1.0)
    return f * (16 if case["dtype"] == "fp32" else 1) * (2 if case["op"] == "purified" else 1)


def draw(rng):
    most = _cost(_case("born", 16, 16, 2048, 64, train=True))
    while True:
        op = rng.choice(["born", "born", "born", "purified", "layer"])
        dtype = rng.choice(["bf16", "bf16", "bf16", "fp16", "fp32"])
        D = rng.choice([64, 64, 64, 128, 128, 32, 48, 80, 96, 256])
        T = int(round(2.0 ** rng.uniform(6.0, 13.0)))
        if rng.random() < 0.5:
            T = max(64, T // 64 * 64)
        c = _case(op, rng.choice([1, 1, 2, 3, 4, 8, 16]), rng.choice([2, 4, 6, 8, 12, 16]), T, D, dtype=dtype,
                  train=rng.random() < 0.6)
        if op == "layer" and dtype == "fp32":
            continue  # the layers run under bf16 or fp16 autocast
        kind = rng.choice(["causal", "causal", "causal", "window", "docs", "both", "full"])
        if kind in ("window", "both"):
            c["window"] = rng.choice([128, 256, 384, 512])
        if kind in ("docs", "both"):
            c["docs"] = rng.choice([128, 512])
        c["causal"] = kind != "full"
        # Born weights are invariant to the scale but for eps, so behind the
        # layer's 16-bit prologue its gradient is all rounding: floats there.
        c["scale"] = "float" if op == "layer" else rng.choice(["float", "heads"])
        if c["B"] * c["H"] * T * D <= 16 * 16 * 2048 * 64 and _cost(c) <= most:
            return c


def _normal(shape, gen):
    return torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32)


def _heads_with_overlap(shape, gen, dim):
    """Queries and keys that share a direction per head (``dim`` is the heads'
    dimension), so that most overlaps are positive, as in a trained head."""
    D = shape[-1]
    one = [1] * (len(shape) - 1) + [D]
    one[dim] = shape[dim]
    shared = _normal(one, gen)
    shared = shared * (SHARED * math.sqrt(D) / shared.norm(dim=-1, keepdim=True))
    return [_normal(shape, gen) + shared for _ in range(2)]


def _rope_tables(T, D):
    half = D // 2
    freqs = 1.0 / (10000.0 ** (torch.arange(half, dtype=torch.float32) / half))
    ang = torch.outer(torch.arange(T, dtype=torch.float32), freqs)
    return torch.cos(ang).view(1, 1, T, half).cuda(), torch.sin(ang).view(1, 1, T, half).cuda()


def prepare(case, seed):
    """Heads with unit-length query and key rows (the layers normalise them),
    or the raw projection outputs for the layer; values and upstream gradients
    are standard normal."""
    gen = torch.Generator("cuda").manual_seed(seed)
    B, H, T, D = case["B"], case["H"], case["T"], case["D"]
    dt = DTYPES[case["dtype"]]
    st = {"case": case}
    layer = case["op"] == "layer"
    shape = (B, T, H, D) if layer else (B, H, T, D)
    q, k = _heads_with_overlap(shape, gen, 2 if layer else 1)
    if not layer:
        q, k = (x / x.norm(dim=-1, keepdim=True) for x in (q, k))
    q, k, v, g = (x.to(dt) for x in (q, k, _normal(shape, gen), _normal(shape, gen)))
    st["grad"] = g
    if layer:
        st["grad"] = g.view(B, T, H * D)
        st["cos"], st["sin"] = _rope_tables(T, D)
    train = case["train"]
    st["q"], st["k"], st["v"] = (x.requires_grad_(train) for x in (q, k, v))
    st["scale"], st["tau"] = SCALE, TAU
    if case["scale"] == "heads":
        jitter = torch.rand(2, H, generator=gen, device="cuda")
        st["scale"] = (SCALE * (0.8 + 0.4 * jitter[0])).view(1, H, 1, 1).requires_grad_(train)
        if case["op"] == "purified":
            st["tau"] = (TAU * (0.8 + 0.4 * jitter[1])).view(1, H, 1, 1).requires_grad_(train)
    st["doc"] = None
    if case["docs"]:
        ends = torch.rand(B, T, generator=gen, device="cuda") < 1.0 / case["docs"]
        st["doc"] = qdl.compute_document_ids(torch.where(ends, EOT, 0))
    return st


def _forward(st):
    case = st["case"]
    kw = dict(is_causal=case["causal"], window_size=case["window"], doc_ids=st["doc"])
    if case["op"] == "born":
        return qdl.flash_born_attention(st["q"], st["k"], st["v"], st["scale"], **kw)
    if case["op"] == "purified":
        return qdl.flash_purified_born_attention(st["q"], st["k"], st["v"], st["scale"], st["tau"], EPS_BASE, **kw)
    q, k, v = (x.transpose(1, 2) for x in (st["q"], st["k"], st["v"]))
    heads = qdl.flash_born_attention_qk_prologue(q, k, v, st["scale"], st["cos"], st["sin"], **kw)
    return heads.transpose(1, 2).reshape(st["grad"].shape)


def _learnt(st):
    """The tensors whose gradients a training step needs, by name."""
    return {n: st[n] for n in ("q", "k", "v", "scale", "tau") if isinstance(st[n], torch.Tensor)}


def run(state):
    if not state["case"]["train"]:
        with torch.no_grad():
            return {"out": _forward(state)}
    out = _forward(state)
    wrt = _learnt(state)
    grads = torch.autograd.grad(out, list(wrt.values()), state["grad"])
    return {"out": out.detach(), **{"d" + n: g for n, g in zip(wrt, grads)}}


def work(case):
    rows = case["B"] * case["H"] * case["T"] * case["D"]
    item = 4 if case["dtype"] == "fp32" else 2
    flops = 4.0 * case["D"] * _pairs(case) * case["B"] * case["H"]
    if case["train"]:  # q, k, v, dout in; out, dq, dk, dv out
        return {"bytes": 8.0 * rows * item, "flops": 3.5 * flops}
    return {"bytes": 4.0 * rows * item, "flops": flops}


def tolerance(case):
    """About four times the error against float64 (worst output: bf16 3.3e-3,
    fp16 3.9e-4, fp32 7.9e-7); the layer's 16-bit prologue doubles it (bf16
    6.4e-3), and the gradient of a purified head's temperature is a cancelling
    sum (bf16 up to 1.7e-2)."""
    rel = {"bf16": 1.2e-2, "fp16": 1.6e-3, "fp32": 4e-6}[case["dtype"]]
    cancels = case["op"] == "purified" and case["train"] and case["scale"] == "heads"
    return {"rel": rel * (2 if case["op"] == "layer" or cancels else 1)}


def _rope_backward(g, c, s):
    half = g.shape[-1] // 2
    g1, g2 = g[..., :half], g[..., half:]
    return torch.cat([g1 * c + g2 * s, g2 * c - g1 * s], dim=-1)


def exact(case, seed):
    """The entry points' mathematics in float64, some heads at a time."""
    st = prepare(case, seed)
    B, H, T, D = case["B"], case["H"], case["T"], case["D"]
    layer, train, purified = case["op"] == "layer", case["train"], case["op"] == "purified"
    if 3e-13 * B * H * T * T * D > 15.0:
        return None
    eps = 1e-8 if purified else 1e-12

    def heads(x):
        x = x.detach().double()
        return (x.transpose(1, 2) if layer else x).reshape(B * H, T, D)

    q, k, v, g = (heads(x) for x in (st["q"], st["k"], st["v"], st["grad"].view(st["q"].shape)))
    if layer:
        c, s = st["cos"].double()[0], st["sin"].double()[0]
        half = D // 2

        def prologue(x):
            y = torch.cat([x[..., :half] * c - x[..., half:] * s, x[..., :half] * s + x[..., half:] * c], dim=-1)
            r = (y.square().sum(-1, keepdim=True) + 1e-12).rsqrt()
            return y * r, r

        (q, rq), (k, rk) = prologue(q), prologue(k)

    def per_head(x):
        x = torch.as_tensor(x, device="cuda").detach().double().reshape(-1)
        return x.expand(H).repeat(B) if x.numel() == 1 else x.repeat(B)

    scale, tau = per_head(st["scale"]), per_head(st["tau"])
    lag = torch.arange(T, device="cuda")[:, None] - torch.arange(T, device="cuda")[None, :]
    keep = torch.ones((T, T), dtype=torch.bool, device="cuda")
    if case["causal"]:
        keep &= lag >= 0
    if case["window"]:
        keep &= lag < case["window"]
    out = torch.empty_like(q)
    dq, dk, dv = (torch.empty_like(q) for _ in range(3)) if train else (None, None, None)
    dscale, dtau = torch.zeros_like(scale), torch.zeros_like(scale)
    step = max(1, min(B * H, CHUNK // (T * T)))
    for b in range(0, B * H, step):
        at = slice(b, b + step)
        sc, ta = scale[at].view(-1, 1, 1), tau[at].view(-1, 1, 1)
        mask = keep[None]
        if st["doc"] is not None:
            doc = st["doc"][torch.arange(B * H, device="cuda")[at] // H]
            mask = mask & (doc[:, :, None] == doc[:, None, :])
        qk = torch.bmm(q[at], k[at].transpose(1, 2).contiguous())
        if purified:
            u = torch.relu(qk - ta)
            w = (sc * u) ** 4 + EPS_BASE * torch.relu(qk) ** 2
        else:
            w = torch.relu(sc * qk) ** 2
        w *= mask
        z = w.sum(-1, keepdim=True) + eps
        out[at] = torch.bmm(w, v[at]) / z
        if not train:
            continue
        delta = (g[at] * out[at]).sum(-1, keepdim=True)
        dv[at] = torch.bmm((w / z).transpose(1, 2).contiguous(), g[at])
        dw = (torch.bmm(g[at], v[at].transpose(1, 2).contiguous()) - delta) / z * mask
        if purified:
            du = dw * 4.0 * sc ** 4 * u ** 3
            dtau[at] = -du.sum((1, 2))
            dscale[at] = (dw * 4.0 * sc ** 3 * u ** 4).sum((1, 2))
            ds = du + dw * 2.0 * EPS_BASE * torch.relu(qk)
        else:
            ds = dw * 2.0 * sc ** 2 * torch.relu(qk)
            # sum of dw * dw/dscale: the weights' common factor cancels against
            # z but for eps.
            dscale[at] = (2.0 / sc * delta * eps / z).sum((1, 2))
        dq[at] = torch.bmm(ds, k[at])
        dk[at] = torch.bmm(ds.transpose(1, 2).contiguous(), q[at])

    def laid(x):
        x = x.view(B, H, T, D)
        return x.transpose(1, 2).contiguous() if layer else x

    got = {"out": laid(out).view(st["grad"].shape)}
    if train:
        if layer:
            dq = _rope_backward((dq - (dq * q).sum(-1, keepdim=True) * q) * rq, c, s)
            dk = _rope_backward((dk - (dk * k).sum(-1, keepdim=True) * k) * rk, c, s)
        got.update(dq=laid(dq), dk=laid(dk), dv=laid(dv))
        if case["scale"] == "heads":
            got["dscale"] = dscale.view(B, H).sum(0).view(1, H, 1, 1)
            if purified:
                got["dtau"] = dtau.view(B, H).sum(0).view(1, H, 1, 1)
    return got
