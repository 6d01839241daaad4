"""Performance cases: the calls a user of this package makes, from the smallest to the largest.

Every pass is one call of a public entry point (``sol_attention``, ``dense_attention``,
``sol_attention_indexed``) on BF16 inputs that are resident on the GPU, with the output allocated by the
call, as in a model's forward pass.  The package is inference only, so there is no backward direction;
BF16 is its only input type.  Sizes are those of this repository's benchmark, receipts and tests, and odd
ones between them.  ``qk_precision="int8"`` and ``threshold_estimator="full_covariance"`` are opt-in
experiments and are left out.

Inputs are the benchmark's three kinds: block-smooth (64-token blocks around a centre each, noise 0.1),
random (iid normal) and a spatiotemporally smooth video field (noise 0.2).
"""

import math
import os
import sys

import torch
import torch.nn.functional as F

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if os.path.join(ROOT, "solattn-amd_amd") not in sys.path:
    sys.path.insert(0, os.path.join(ROOT, "solattn-amd_amd"))

from sol_attn_amd import IndexedPlan, dense_attention, sol_attention, sol_attention_indexed  # noqa: E402

BLOCK = 64


def _self(name, tokens, heads, dim, *, batch=1, beta=1.0, sinks=0, fill="block-smooth"):
    return dict(name=name, kind="sol", batch=batch, tq=tokens, tk=tokens, heads=heads, dim=dim, beta=beta,
                local=1, kv_sink=sinks, q_sink=sinks, head_stride=1, fill=fill)


def listed():
    return [
        # The smallest call: a short prompt against a short context with head-strided views (every other
        # head of a fused projection), odd lengths.  Latency and launches only.
        dict(name="tiny 193x317 h2 d64", kind="sol", batch=1, tq=193, tk=317, heads=2, dim=64, beta=1.0, local=1,
             kv_sink=64, q_sink=0, head_stride=2, fill="random"),
        # One image's tokens, a small model's heads, with text sinks: the benchmark's small self-attention.
        _self("self 1024 h8 d64", 1024, 8, 64, sinks=128),
        # The receipts' shapes: one tensor-parallel rank's four heads.
        _self("self 1024 h4 d128", 1024, 4, 128),
        _self("self 4096 h4 d128", 4096, 4, 128),
        # An ordinary batch of two images at an odd length and the smaller head dimension.
        _self("self 2x3001 h12 d64", 3001, 12, 64, batch=2, fill="random"),
        # Image self-attention at batch 2 (the benchmark's 4,096-token configuration).
        _self("self 2x4096 h16 d128", 4096, 16, 128, batch=2, sinks=128),
        # The same without routing: the dense entry point (guidance or full-precision layers).
        dict(name="dense 2x4096 h16 d128", kind="dense", batch=2, tq=4096, tk=4096, heads=16, dim=128,
             head_stride=1, fill="block-smooth"),
        # Cross-attention to a longer context whose length is no multiple of a block, head-strided Q.
        dict(name="cross 4096x10000 h24 d128", kind="sol", batch=1, tq=4096, tk=10000, heads=24, dim=128, beta=1.0,
             local=0, kv_sink=64, q_sink=0, head_stride=2, fill="random"),
        # A short video clip at an odd token count.
        _self("video 19003 h16 d128", 19003, 16, 128, fill="field"),
        # A long video: 21 x 48 x 84 tokens, text sinks (the headline configuration).
        _self("video 84672 h24 d128", 84672, 24, 128, sinks=128, fill="field"),
        # The same video as frame windows (frames 0, f-1, f, f+1), stored into the full sequence.
        dict(name="windows 21x4032 h24 d128", kind="windows", frames=21, tpf=4032, heads=24, dim=128, beta=1.0,
             head_stride=1, fill="field"),
        # Its anchor rows: the first frame's queries over every token, dense, into the full sequence.
        dict(name="anchors 4032x84672 h24", kind="anchors", frames=21, tpf=4032, heads=24, dim=128, beta=-math.inf,
             head_stride=1, fill="field"),
    ]


# Token pairs x heads of the largest listed case, weighted by the share that is attended exactly.
_MOST = 84672 ** 2 * 24 * 0.2


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("sol", "sol", "sol", "cross", "cross", "dense", "windows", "anchors"))
    heads, dim = rng.choice((1, 2, 3, 4, 8, 12, 16, 24)), rng.choice((64, 128, 128))
    fill = rng.choice(("block-smooth", "random", "field"))
    if kind in ("windows", "anchors"):
        frames, tpf = rng.randint(2, 21), _log_int(rng, 100, 4032)
        return dict(kind=kind, frames=frames, tpf=tpf, heads=heads, dim=dim,
                    beta=-math.inf if kind == "anchors" else rng.choice((0.0, 1.0, 1.0)),
                    head_stride=rng.choice((1, 1, 2)), fill=fill)
    tq = _log_int(rng, 100, 20000 if kind == "dense" else 84672)
    tk = _log_int(rng, 100, 40000) if kind == "cross" else tq
    beta = rng.choice((0.0, 0.5, 1.0, 1.0, 1.0, math.inf))
    case = dict(kind="dense" if kind == "dense" else "sol", batch=rng.choice((1, 1, 2)) if tq <= 8192 else 1, tq=tq,
                tk=tk, heads=heads, dim=dim, head_stride=rng.choice((1, 1, 2)), fill=fill)
    if kind != "dense":
        sink = rng.choice((0, 0, 64, 128))
        case.update(beta=beta, local=0 if kind == "cross" else 1, kv_sink=min(sink, tk),
                    q_sink=0 if kind == "cross" else min(sink, tq))
    while case["batch"] * tq * tk * case["heads"] * _density(case) > _MOST:
        case["heads"] = max(1, case["heads"] // 2)
    return case


# ---- inputs -----------------------------------------------------------------------------------------------


def _field(gen, tokens, heads, dim):
    """The benchmark's smooth video field over (frames, height, width), cut to `tokens` tokens."""
    frames = min(21, max(1, round(tokens / 4032)))
    area = -(-tokens // frames)
    height = max(1, round(math.sqrt(area * 4 / 7)))
    width = -(-area // height)
    grid = torch.randn((heads, dim, 6, 12, 21), generator=gen, device="cuda")
    up = F.interpolate(grid, size=(frames, height, width), mode="trilinear", align_corners=False)
    x = up.flatten(2).permute(2, 0, 1)[:tokens].contiguous()[None]
    return x + 0.2 * torch.randn(x.shape, generator=gen, device="cuda")


def _tensor(gen, fill, batch, tokens, heads, dim, head_stride=1):
    if fill == "field":
        x = torch.cat([_field(gen, tokens, heads, dim) for _ in range(batch)])
    else:
        x = torch.randn((batch, tokens, heads, dim), generator=gen, device="cuda")
        if fill == "block-smooth":
            centres = torch.randn((batch, -(-tokens // BLOCK), heads, dim), generator=gen, device="cuda")
            x = centres.repeat_interleave(BLOCK, 1)[:, :tokens] + 0.1 * x
    x = x.to(torch.bfloat16)
    if head_stride == 1:
        return x.contiguous()
    wide = torch.zeros((batch, tokens, heads * head_stride, dim), dtype=torch.bfloat16, device="cuda")
    wide[:, :, ::head_stride] = x
    return wide[:, :, ::head_stride]


def _window_indices(case):
    """Frame windows: window f's queries are frame f, its keys frames {0, f-1, f, f+1}."""
    frames, tpf = case["frames"], case["tpf"]
    rows = torch.arange(frames * tpf).view(frames, tpf)
    if case["kind"] == "anchors":
        return rows[:1], torch.arange(frames * tpf)[None]
    keys = [torch.cat([rows[x] for x in sorted({0, f - 1, f, f + 1} & set(range(frames)))]) for f in range(frames)]
    return rows, keys


def _plan(case):
    rows, keys = _window_indices(case)
    n = case["frames"] * case["tpf"]
    if case["kind"] == "anchors":
        return IndexedPlan.create(rows, keys, n)
    return IndexedPlan.create(rows, keys, n, protected_ranges=((0, case["tpf"]),), local_tokens=64)


def _inputs(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    if case["kind"] in ("windows", "anchors"):
        n = case["frames"] * case["tpf"]
        return [_tensor(gen, case["fill"], 1, n, case["heads"], case["dim"], case["head_stride"])[0] for _ in range(3)]
    stride = case["head_stride"]
    return [_tensor(gen, case["fill"], case["batch"], t, case["heads"], case["dim"], s)
            for t, s in ((case["tq"], stride), (case["tk"], 1 if case["tq"] != case["tk"] else stride),
                         (case["tk"], 1 if case["tq"] != case["tk"] else stride))]


def prepare(case, seed):
    q, k, v = _inputs(case, seed)
    state = dict(case=case, q=q, k=k, v=v)
    if case["kind"] in ("windows", "anchors"):
        # The plan is built once per sequence shape, and the adapter owns the full-sequence output.
        state["plan"] = _plan(case).to(q.device)
        state["out"] = torch.zeros(q.shape, dtype=q.dtype, device=q.device)
    return state


def run(state):
    case, q, k, v = state["case"], state["q"], state["k"], state["v"]
    if case["kind"] == "dense":
        return dense_attention(q, k, v)
    if case["kind"] == "sol":
        return sol_attention(q, k, v, beta=case["beta"], local_blocks=case["local"],
                             kv_sink_tokens=case["kv_sink"], query_sink_tokens=case["q_sink"])
    return sol_attention_indexed(q, k, v, state["plan"], beta=case["beta"], out=state["out"])


# ---- what a pass cannot do without ------------------------------------------------------------------------


def _density(case):
    """Share of the key blocks attended exactly: the share of a normal above `beta` (what the threshold
    aims at), at least the protected blocks."""
    beta = case.get("beta", -math.inf)
    if case["kind"] == "windows":
        # Frame 0 is protected in every window of 2 to 4 frames.
        return min(1.0, 0.5 * math.erfc(beta / math.sqrt(2)) + 0.25)
    share = 1.0 if beta == -math.inf else 0.5 * math.erfc(beta / math.sqrt(2))
    nkb = -(-case["tk"] // BLOCK) if "tk" in case else 1
    forced = 2 * case.get("local", 0) + 1 + -(-case.get("kv_sink", 0) // BLOCK) if case["kind"] == "sol" else 0
    sink = min(1.0, -(-case.get("q_sink", 0) // BLOCK) / -(-case["tq"] // BLOCK)) if "tq" in case else 0.0
    share = min(1.0, max(share, forced / nkb))
    return sink + (1.0 - sink) * share


def work(case):
    """Q, K and V read once and the output written once; the products of the exact blocks and, for the others,
    of one centroid each, and the routing products."""
    h, d = case["heads"], case["dim"]
    if case["kind"] in ("windows", "anchors"):
        n, tpf = case["frames"] * case["tpf"], case["tpf"]
        rows, keys = _window_indices(case)
        pairs = sum(tpf * len(x) for x in keys)
        queries = rows.numel()
        tokens = 2 * queries + 2 * n
        routed = 0 if case["kind"] == "anchors" else pairs
    else:
        b, tq, tk = case["batch"], case["tq"], case["tk"]
        pairs, tokens = b * tq * tk, b * (2 * tq + 2 * tk)
        routed = 0 if case["kind"] == "dense" else pairs
    share = _density(case)
    flops = 4.0 * pairs * h * d * share
    if routed:
        flops += 4.0 * pairs * h * d * (1.0 - share) / BLOCK + 2.0 * pairs * h * d / BLOCK ** 2
    return {"bytes": 2.0 * tokens * h * d, "flops": flops}


def tolerance(case):
    # BF16 probabilities and outputs with FP32 sums: 0.17% to 0.24% from the 64-bit result in every case, which
    # another order of the sums or of the rounding shows as well.  A block whose proxy lies within FP32
    # rounding of the cutoff may be routed the other way: few rows, of their own size.
    return {"rel": 8e-3, "max": 0.5}


# ---- the same in 64 bits ----------------------------------------------------------------------------------


def _block_means(x):
    """Means of 64-row blocks (the last may be shorter) of x [T, D]."""
    n = -(-x.shape[0] // BLOCK)
    total = F.pad(x, (0, 0, 0, n * BLOCK - x.shape[0])).view(n, BLOCK, -1).sum(1)
    lens = torch.full((n,), float(BLOCK), dtype=x.dtype, device=x.device)
    lens[-1] = x.shape[0] - BLOCK * (n - 1)
    return total / lens[:, None], lens


def _attend64(q, k, v, beta, scale, local=-1, kv_sink=0, q_sink=0, protected=None):
    """One head in 64 bits: q [Tq, D], k / v [Tk, D].  Centroids are BF16, as the method defines them."""
    q, k, v = (x.to(torch.float64) for x in (q, k, v))
    kt = k.t().contiguous()
    out = torch.empty_like(q)
    step = max(BLOCK, (1 << 28) // k.shape[0] // BLOCK * BLOCK)
    if beta == -math.inf:
        for i in range(0, q.shape[0], step):
            p = torch.softmax((q[i:i + step] @ kt) * scale, 1)
            out[i:i + step] = p @ v
        return out
    qc, _ = _block_means(q)
    kc, lens = _block_means(k)
    vc, _ = _block_means(v)
    kc, vc = (x.to(torch.bfloat16).to(torch.float64) for x in (kc, vc))
    nqb, nkb = qc.shape[0], kc.shape[0]
    dev = q.device
    sel = torch.zeros((nqb, nkb), dtype=torch.bool, device=dev)
    if beta != math.inf:
        mu = kc.mean(0)
        var = ((kc * kc).mean(0) - mu * mu).clamp_min(0)
        cut = qc @ mu + beta * torch.sqrt((qc * qc) @ var)
        sel = (qc @ kc.t().contiguous()) > cut[:, None]
    if local >= 0:
        sel |= (torch.arange(nqb, device=dev)[:, None] - torch.arange(nkb, device=dev)[None]).abs() <= local
    sel[:, :-(-kv_sink // BLOCK)] = True
    sel[:-(-q_sink // BLOCK)] = True
    if protected is not None:
        sel |= protected
    kct = kc.t().contiguous()
    loglen = torch.log(lens)
    for i in range(0, q.shape[0], step):
        qq = q[i:i + step]
        s = sel[i // BLOCK:i // BLOCK + -(-qq.shape[0] // BLOCK)]
        rows = s.repeat_interleave(BLOCK, 0)[:qq.shape[0]]
        exact = (qq @ kt) * scale
        exact.masked_fill_(~rows.repeat_interleave(BLOCK, 1)[:, :k.shape[0]], -math.inf)
        approx = (qq @ kct) * scale + loglen
        approx.masked_fill_(rows, -math.inf)
        m = torch.maximum(exact.amax(1), approx.amax(1))[:, None]
        exact.sub_(m).exp_()
        approx.sub_(m).exp_()
        den = exact.sum(1) + approx.sum(1)
        out[i:i + step] = (exact @ v + approx @ vc) / den[:, None]
    return out


def exact(case, seed):
    if "tq" in case and case["batch"] * case["heads"] * case["tq"] * case["tk"] > 2e11:
        return None  # longer than about 20 seconds in 64 bits
    q, k, v = _inputs(case, seed)
    h, d = case["heads"], case["dim"]
    scale = d ** -0.5
    if case["kind"] in ("windows", "anchors"):
        plan = _plan(case)
        rows, keys = _window_indices(case)
        out = torch.zeros(q.shape, dtype=torch.float64, device=q.device)
        for w, kw in enumerate(keys):
            r, kw = rows[w].to(q.device), kw.to(q.device)
            prot = plan.protected_blocks[w, :, :-(-len(kw) // BLOCK)].to(q.device)
            for i in range(h):
                out[r, i] = _attend64(q[r, i], k[kw, i], v[kw, i], case["beta"], scale, protected=prot)
        return out
    out = torch.empty((case["batch"], case["tq"], h, d), dtype=torch.float64, device=q.device)
    kw = {} if case["kind"] == "dense" else dict(local=case["local"], kv_sink=case["kv_sink"], q_sink=case["q_sink"])
    beta = case.get("beta", -math.inf)
    for b in range(case["batch"]):
        for i in range(h):
            out[b, :, i] = _attend64(q[b, :, i], k[b, :, i], v[b, :, i], beta, scale, **kw)
    return out
