"""The work a user of scratchtape_amd has it do, as cases that can be timed and compared.

Twelve listed cases over the package's public entry points, in the sizes of its own workloads (the d_model-256
byte-level language model over 32 windows of 128 tokens; the 125M-key 2-bit memory with 12,288 cells) and in generic
sizes to either side of them: one window or one decoding step, odd widths that no tile divides, wide layers.

- linear:       a Linear layer, forward (bias, ReLU) and backward (weight and bias gradients accumulated, input gradient)
- step_set:     every GEMM of one training step as one grouped call (five Linear layers, each forward, dX, dW)
- attn_fused:   causal attention forward and backward in the fused kernels
- attn:         the same through batched GEMMs and softmax, any sequence length and head width, f32 or f16 route
- layer_norm:   LayerNorm forward and backward
- ivf:          probe selection and the IVF scan of the 2-bit memory, top-k per query
- masked:       the exact search of each query's own key range plus a prefix (a document's tail)
- quantize:     f32 keys to 2-bit codes and scales (building the memory)

A case is a plain dict; `draw` makes more over the same ranges.  Every pass writes all of its outputs anew, so a state
can be run any number of times.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from scratchtape_amd import Epilogue, MatRef, matmul_grouped, matmul_with
from scratchtape_amd import attention, knn, rows

DEV = "cuda"
D_KEY = 256  # width of the 2-bit memory's keys


def listed():
    return [
        # One window of 128 tokens through the QKV projection: a single sequence, where launches and latency count.
        dict(name="linear_one_window", kind="linear", tokens=128, din=256, dout=768, f16=True, relu=False),
        # A wide feed-forward layer over 64 windows of 256 tokens: the largest matrix products.
        dict(name="linear_wide", kind="linear", tokens=16384, din=1024, dout=4096, f16=True, relu=True),
        # f32 with widths no tile divides and rows that are not 16-byte aligned (250 floats): what arbitrary layers give.
        dict(name="linear_odd_f32", kind="linear", tokens=3000, din=250, dout=1001, f16=False, relu=True),
        # The training step of the d_model-256 model over 32 windows x 128 tokens, its 15 GEMMs in one call.
        dict(name="step_set", kind="step_set", tokens=4096, d=256, vocab=256, f16=True),
        # The same model's attention, forward and backward: 32 windows x 4 heads x 128 tokens, head width 64.
        dict(name="attn_fused", kind="attn_fused", b=32, h=4, t=128, one=False),
        # Attention over windows cut at 200 tokens with 80-wide heads, which the fused kernels do not take, in f32.
        dict(name="attn_odd_f32", kind="attn", b=16, h=6, t=200, hd=80, f16=False),
        # LayerNorm over a large batch: 256 windows of 256 tokens, 768 wide.
        dict(name="layer_norm_large", kind="layer_norm", rows=65536, d=768),
        # One decoding step of a few sequences: 4 queries against the memory, where latency counts.
        dict(name="ivf_decode", kind="ivf", nq=4, nprobe=16, ncells=4096, mean_cell=5000, k=128),
        # The full memory, 125M keys in 12,288 cells, one batch of 256 queries probing 8 cells each.
        dict(name="ivf_batch", kind="ivf", nq=256, nprobe=8, ncells=12288, mean_cell=10172, k=128),
        # An evaluation pass, which asks for thousands of queries per call.
        dict(name="ivf_eval", kind="ivf", nq=4096, nprobe=8, ncells=12288, mean_cell=10172, k=128),
        # The tail search of 32 tokens: each sees up to 20,000 keys of its own document and a shared prefix.
        dict(name="masked_tail", kind="masked", nq=32, window=20000, always=1000, nkeys=4000000, k=128),
        # A tile of a million keys quantised while the memory is built.
        dict(name="quantize_tile", kind="quantize", n=1 << 20, d=256),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _width(rng, lo, hi):
    """A size from lo to hi: half of the time any, else a multiple of 32 or 64 as layers usually have."""
    n = _log_int(rng, lo, hi)
    step = rng.choice([1, 1, 32, 64])
    return max(step, n // step * step)


def draw(rng):
    kind = rng.choice(["linear", "linear", "linear", "step_set", "attn_fused", "attn", "layer_norm", "ivf", "ivf",
                       "masked", "quantize"])
    if kind == "linear":
        while True:
            f16 = rng.random() < 0.6
            c = dict(kind=kind, tokens=_width(rng, 64, 16384), din=_width(rng, 64, 4096), dout=_width(rng, 64, 4096),
                     f16=f16, relu=rng.random() < 0.5)
            # A drawn case costs no more than linear_wide; f32 products run at a fraction of the f16 rate.
            if c["tokens"] * c["din"] * c["dout"] <= (6.8e10 if f16 else 8e9):
                return c
    if kind == "step_set":
        return dict(kind=kind, tokens=_width(rng, 128, 8192), d=_width(rng, 64, 512),
                    vocab=rng.choice([256, 256, 257, 512, 1000]), f16=rng.random() < 0.7)
    if kind == "attn_fused":
        return dict(kind=kind, b=_log_int(rng, 1, 64), h=rng.randint(1, 12), t=32 * rng.randint(1, 8),
                    one=rng.random() < 0.3)
    if kind == "attn":
        return dict(kind=kind, b=_log_int(rng, 1, 32), h=rng.randint(1, 12), t=_width(rng, 32, 256),
                    hd=rng.choice([16, 24, 32, 40, 48, 64, 80, 96, 128]), f16=rng.random() < 0.4)
    if kind == "layer_norm":
        return dict(kind=kind, rows=_log_int(rng, 64, 65536), d=_width(rng, 33, 1536) if rng.random() < 0.5
                    else 4 * rng.randint(16, 256))
    if kind == "ivf":
        return dict(kind=kind, nq=_log_int(rng, 1, 4096), nprobe=rng.randint(1, 16), ncells=_log_int(rng, 64, 6000),
                    mean_cell=_log_int(rng, 300, 10000), k=rng.choice([1, 10, 64, 128, 128, 128]))
    if kind == "masked":
        return dict(kind=kind, nq=_log_int(rng, 1, 256), window=_log_int(rng, 500, 80000),
                    always=rng.choice([0, 256, 1000, 5000]), nkeys=_log_int(rng, 200000, 8000000),
                    k=rng.choice([10, 64, 128, 128]))
    return dict(kind="quantize", n=_log_int(rng, 1000, 1 << 20), d=rng.choice([64, 128, 256, 256]))


# ---- inputs ---------------------------------------------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 7919 + 17)
    return g


def _randn(g, *shape, std=1.0):
    return torch.randn(*shape, generator=g, device=DEV, dtype=torch.float32).mul_(std)


def _empty(*shape):
    return torch.empty(*shape, device=DEV, dtype=torch.float32)


def _step_layers(c):
    """(name, in width, out width) of the model's five Linear layers."""
    d = c["d"]
    return [("qkv", d, 3 * d), ("out", d, d), ("ffn1", d, 4 * d), ("ffn2", 4 * d, d), ("head", d, c["vocab"])]


def _linear_inputs(c, seed):
    g = _gen(seed)
    t, i, o = c["tokens"], c["din"], c["dout"]
    x = _randn(g, t, i)
    if c["relu"]:
        x = x.clamp_(min=0.0)  # the layer before ends in a ReLU too: its output masks the input gradient
    return x, _randn(g, i, o, std=0.02), _randn(g, o, std=0.02), _randn(g, t, o)


def _step_inputs(c, seed):
    g = _gen(seed)
    t = c["tokens"]
    return [(_randn(g, t, i), _randn(g, i, o, std=0.02), _randn(g, t, o)) for _, i, o in _step_layers(c)]


def _attn_inputs(c, seed):
    g = _gen(seed)
    b, h, t, hd = c["b"], c["h"], c["t"], c.get("hd", 64)
    return _randn(g, b * t, 3 * h * hd), _randn(g, b * t, h * hd)


def _ln_inputs(c, seed):
    g = _gen(seed)
    n, d = c["rows"], c["d"]
    params = _randn(g, 2 * d, std=0.1)
    params[:d] += 1.0
    return _randn(g, n, d), _randn(g, n, d), params


def _ivf_inputs(c, seed):
    """Cell bounds (host), centroids, and queries that lie near cells of their own."""
    g = _gen(seed)
    sizes = np.random.RandomState(seed % (1 << 31)).uniform(0.5, 1.5, c["ncells"]) * c["mean_cell"]
    bounds = np.concatenate([[0], np.cumsum(np.maximum(sizes.astype(np.int64), 130))])
    cent = _randn(g, c["ncells"], D_KEY)
    home = torch.randint(0, c["ncells"], (c["nq"],), generator=g, device=DEV)
    return bounds, cent, (cent[home] + _randn(g, c["nq"], D_KEY)).mul_(0.7)


def _masked_inputs(c, seed):
    g = _gen(seed)
    n, w = c["nkeys"], min(c["window"], c["nkeys"] - c["always"] - 1)
    length = torch.randint(max(128, w // 2), w + 1, (c["nq"],), generator=g, device=DEV)
    lo = c["always"] + (torch.rand(c["nq"], generator=g, device=DEV, dtype=torch.float64)
                        * (n - c["always"] - length)).long()
    return _randn(g, c["nq"], D_KEY), torch.stack([lo, lo + length], 1).contiguous()


def _store(seed, bounds):
    n = int(bounds[-1])
    codes = torch.empty((n, D_KEY // 4), dtype=torch.uint8, device=DEV)
    scales = _empty(n)
    knn.synth_store_2bit(seed + 1, 0, codes, scales)  # the codes and scales of N(0, 1) keys
    return knn.KnnStore2bit(codes, scales, bounds, D_KEY)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "linear":
        x, w, b, dy = _linear_inputs(case, seed)
        t, i, o = case["tokens"], case["din"], case["dout"]
        return dict(case=case, x=x, w=w, b=b, dy=dy, y=_empty(t, o), dx=_empty(t, i), grads=_empty(i * o + o))
    if kind == "step_set":
        bufs = [(x, w, dy, _empty(*dy.shape), _empty(*x.shape), _empty(*w.shape))
                for x, w, dy in _step_inputs(case, seed)]
        return dict(case=case, bufs=bufs)
    if kind == "attn_fused":
        qkv, dctx = _attn_inputs(case, seed)
        return dict(case=case, qkv=qkv, dctx=dctx,
                    buf=attention.FusedBuffers.empty(case["b"], case["h"], case["t"], 64, DEV))
    if kind == "attn":
        qkv, dctx = _attn_inputs(case, seed)
        return dict(case=case, qkv=qkv, dctx=dctx,
                    buf=attention.AttnBuffers.empty(case["b"], case["h"], case["t"], case["hd"], DEV))
    if kind == "layer_norm":
        x, dy, params = _ln_inputs(case, seed)
        return dict(case=case, x=x, dy=dy, params=params, grads=torch.zeros_like(params), dx=torch.empty_like(x))
    if kind == "ivf":
        bounds, cent, q = _ivf_inputs(case, seed)
        store = _store(seed, bounds)
        store.set_centroids(cent)
        return dict(case=case, store=store, q=q)
    if kind == "masked":
        q, lohi = _masked_inputs(case, seed)
        return dict(case=case, store=_store(seed, np.array([0, case["nkeys"]])), q=q, lohi=lohi)
    return dict(case=case, keys=_randn(_gen(seed), case["n"], case["d"]))


# ---- one pass ---------------------------------------------------------------------------------------------------

def run(state):
    c = state["case"]
    kind = c["kind"]
    if kind == "linear":
        t, i, o, f16 = c["tokens"], c["din"], c["dout"], c["f16"]
        x, w, dy, grads = MatRef(state["x"]), MatRef(state["w"]), MatRef(state["dy"]), state["grads"]
        matmul_with(x, w, MatRef(state["y"]), 1, t, i, o, Epilogue(bias=(state["b"], 0), relu=c["relu"]), f16)
        grads.zero_()  # the step's cleared gradients
        matmul_grouped([
            (x.with_(trans=True), dy, MatRef(grads), 1, i, t, o, Epilogue(accumulate=True, col_sum=(i * o, 0)), f16),
            (dy, w.with_(trans=True), MatRef(state["dx"]), 1, t, o, i,
             Epilogue(mask=(state["x"], 0)) if c["relu"] else None, f16)])
        return dict(y=state["y"], dx=state["dx"], dw=grads[:i * o], db=grads[i * o:])
    if kind == "step_set":
        t, f16, calls = c["tokens"], c["f16"], []
        for x, w, dy, y, dx, dw in state["bufs"]:
            i, o = w.shape
            calls += [(MatRef(x), MatRef(w), MatRef(y), 1, t, i, o, None, f16),
                      (MatRef(dy), MatRef(w, trans=True), MatRef(dx), 1, t, o, i, None, f16),
                      (MatRef(x, trans=True), MatRef(dy), MatRef(dw), 1, i, t, o, None, f16)]
        matmul_grouped(calls)
        return [list(b[3:]) for b in state["bufs"]]
    if kind == "attn_fused":
        attention.fused_step(state["qkv"], state["dctx"], state["buf"], c["b"], c["h"], c["t"], 64, c["one"])
        return dict(ctx=state["buf"].ctx, lse=state["buf"].lse, dqkv=state["buf"].dqkv)
    if kind == "attn":
        attention.step(state["qkv"], state["dctx"], state["buf"], c["b"], c["h"], c["t"], c["hd"], c["f16"])
        return dict(p=state["buf"].p, ctx=state["buf"].ctx, dqkv=state["buf"].dqkv)
    if kind == "layer_norm":
        n, d = c["rows"], c["d"]
        fwd = rows.layer_norm(state["x"], n, d, state["params"], 0)
        state["grads"].zero_()
        rows.layer_norm_backward(state["dy"], state["x"], fwd, n, d, state["params"], state["grads"], 0, state["dx"],
                                 False)
        return dict(y=fwd.y, mean=fwd.mean, rstd=fwd.rstd, dx=state["dx"], grads=state["grads"])
    if kind == "ivf":
        idx, dist = state["store"].search_ivf(state["q"], c["nprobe"], c["k"])
        return dict(idx=idx, dist=dist)
    if kind == "masked":
        idx, dist = state["store"].search_masked(state["q"], state["lohi"], c["always"], c["k"])
        return dict(idx=idx, dist=dist)
    codes, scales = knn.quantize_2bit(state["keys"])
    return dict(codes=codes, scales=scales)


# ---- what a pass cannot do without ---------------------------------------------------------------------------------

def work(case):
    kind = case["kind"]
    if kind == "linear":
        t, i, o = case["tokens"], case["din"], case["dout"]
        return dict(bytes=4 * (2 * t * i + 2 * t * o + 2 * i * o + 2 * o), flops=6 * t * i * o)
    if kind == "step_set":
        t = case["tokens"]
        return dict(bytes=sum(4 * (2 * t * i + 2 * t * o + 2 * i * o) for _, i, o in _step_layers(case)),
                    flops=sum(6 * t * i * o for _, i, o in _step_layers(case)))
    if kind in ("attn_fused", "attn"):
        b, h, t, hd = case["b"], case["h"], case["t"], case.get("hd", 64)
        tokens, causal = b * t * h * hd, b * h * t * (t + 1) // 2
        # Read qkv and dctx, write ctx and dqkv; with "attn" also the probabilities that it returns.
        extra = b * h * t if kind == "attn_fused" else b * h * t * t
        return dict(bytes=4 * (8 * tokens + extra), flops=6 * 2 * causal * hd)
    if kind == "layer_norm":
        n, d = case["rows"], case["d"]
        # x and dy in, y and dx out: the backward's second look at x is a read of its own (two calls).
        return dict(bytes=4 * (5 * n * d + 2 * n), flops=20 * n * d)
    if kind == "ivf":
        probes = case["nq"] * case["nprobe"]
        cells = case["ncells"] * (1.0 - (1.0 - 1.0 / case["ncells"]) ** probes)  # distinct cells, expected
        return dict(bytes=cells * case["mean_cell"] * 68 + case["ncells"] * 524 + case["nq"] * (1024 + 12 * case["k"]),
                    flops=512.0 * (probes * case["mean_cell"] + case["nq"] * case["ncells"]))
    if kind == "masked":
        keys = case["nq"] * 0.75 * min(case["window"], case["nkeys"])
        return dict(bytes=68 * (min(keys, case["nkeys"]) + case["always"]) + case["nq"] * (1040 + 12 * case["k"]),
                    flops=512.0 * (keys + case["nq"] * case["always"]))
    return dict(bytes=case["n"] * (4 * case["d"] + case["d"] // 4 + 4), flops=6 * case["n"] * case["d"])


def tolerance(case):
    kind = case["kind"]
    if kind in ("ivf", "masked", "quantize"):
        return "exact"  # integer scores, one fixed f32 expression per distance; the quantiser is fixed bit for bit
    if kind == "layer_norm":
        return {"rel": 1e-5}
    # Four times the measured distance from 64 bits where operands (and the fused kernels' probabilities) are rounded
    # to f16 and sums are f32: 2.9e-4 for the products, 4.7e-4 for the attention gradients.
    if kind == "attn_fused":
        return {"rel": 2e-3}
    if case["f16"]:
        return {"rel": 2e-3 if kind == "attn" else 1.2e-3}
    return {"rel": 1e-5}


# ---- the same in 64 bits ---------------------------------------------------------------------------------------------

def _exact_attn(case, seed, one):
    b, h, t, hd = case["b"], case["h"], case["t"], case.get("hd", 64)
    qkv, dctx = _attn_inputs(case, seed)
    q, k, v = (z.contiguous() for z in qkv.double().view(b, t, 3, h, hd).permute(2, 0, 3, 1, 4))
    do = dctx.double().view(b, t, h, hd).permute(0, 2, 1, 3).contiguous()
    scale = hd ** -0.5
    s = torch.matmul(q, k.transpose(-1, -2).contiguous()) * scale
    s = s.masked_fill(torch.ones(t, t, dtype=torch.bool, device=DEV).triu(1), -math.inf)
    m = s.amax(-1, keepdim=True)
    if one:
        m = m.clamp(min=0.0)
    e = torch.exp(s - m)
    z = e.sum(-1, keepdim=True) + (torch.exp(-m) if one else 0.0)
    p = e / z
    o = torch.matmul(p, v)
    dv = torch.matmul(p.transpose(-1, -2).contiguous(), do)
    dp = torch.matmul(do, v.transpose(-1, -2).contiguous())
    ds = scale * p * (dp - (dp * p).sum(-1, keepdim=True))
    dq, dk = torch.matmul(ds, k), torch.matmul(ds.transpose(-1, -2).contiguous(), q)
    merged = torch.stack([dq, dk, dv]).permute(1, 3, 0, 2, 4).reshape(-1)
    return p.reshape(-1), o.permute(0, 2, 1, 3).reshape(-1), (m + torch.log(z)).reshape(-1), merged


def _int16(v):
    """Rows as the search takes a query: integers of up to 15 bits and a power-of-two step per row."""
    top = v.abs().amax(1, keepdim=True).double()
    step = torch.exp2(torch.floor(torch.log2(top)) + 1 - 14)
    return torch.clamp(torch.round(v.double() / step), -16384, 16383) * step


def _decode(codes, scales):
    u = torch.stack([(codes >> s) & 3 for s in (0, 2, 4, 6)], -1).reshape(codes.shape[0], -1)
    return (u.double() - 1.5) * scales.double()[:, None]


def _nearest(store, q, spans, k):
    """The k smallest |q - key|^2 of each query over its row spans, ascending."""
    out = torch.full((q.shape[0], k), math.inf, dtype=torch.float64, device=DEV)
    for i, sp in enumerate(spans):
        d = torch.cat([(_decode(store.codes[a:b], store.scales[a:b]) - q[i]).square_().sum(1) for a, b in sp if b > a])
        near = torch.topk(d, min(k, d.numel()), largest=False).values
        out[i, :near.numel()] = near
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind == "linear":
        x, w, b, dy = (z.double() for z in _linear_inputs(case, seed))
        y = x @ w + b
        dx = dy @ w.t().contiguous()
        if case["relu"]:
            y = y.clamp(min=0.0)
            dx = torch.where(x > 0, dx, torch.zeros_like(dx))
        return dict(y=y, dx=dx, dw=(x.t().contiguous() @ dy).reshape(-1), db=dy.sum(0))
    if kind == "step_set":
        out = []
        for x, w, dy in _step_inputs(case, seed):
            x, w, dy = x.double(), w.double(), dy.double()
            out.append([x @ w, dy @ w.t().contiguous(), x.t().contiguous() @ dy])
        return out
    if kind == "attn_fused":
        _, ctx, lse, dqkv = _exact_attn(case, seed, case["one"])
        return dict(ctx=ctx, lse=lse, dqkv=dqkv)
    if kind == "attn":
        p, ctx, _, dqkv = _exact_attn(case, seed, False)
        return dict(p=p, ctx=ctx, dqkv=dqkv)
    if kind == "layer_norm":
        x, dy, params = (z.double() for z in _ln_inputs(case, seed))
        d = case["d"]
        gamma, beta = params[:d], params[d:]
        mean = x.mean(1, keepdim=True)
        rstd = 1.0 / torch.sqrt((x - mean).square().mean(1, keepdim=True) + 1e-5)
        xh = (x - mean) * rstd
        gy = dy * gamma
        dx = rstd * (gy - gy.mean(1, keepdim=True) - xh * (gy * xh).mean(1, keepdim=True))
        return dict(y=(xh * gamma + beta).reshape(-1), mean=mean.reshape(-1), rstd=rstd.reshape(-1), dx=dx,
                    grads=torch.cat([(dy * xh).sum(0), dy.sum(0)]))
    if kind == "ivf":
        if case["nq"] * case["nprobe"] > 4096:
            return None
        bounds, cent, q = _ivf_inputs(case, seed)
        store, qi, ci = _store(seed, bounds), _int16(q), _int16(cent)
        dd = ci.square().sum(1) - 2.0 * (qi @ ci.t().contiguous())
        cells = torch.sort(dd, dim=1, stable=True).indices[:, :case["nprobe"]].tolist()
        return dict(idx=None, dist=_nearest(store, qi, [[(int(bounds[p]), int(bounds[p + 1])) for p in row]
                                                        for row in cells], case["k"]))
    if kind == "masked":
        if case["nq"] * case["window"] > 20_000_000:
            return None
        q, lohi = _masked_inputs(case, seed)
        store = _store(seed, np.array([0, case["nkeys"]]))
        return dict(idx=None, dist=_nearest(store, _int16(q), [[(0, case["always"]), (int(a), int(b))]
                                                               for a, b in lohi.tolist()], case["k"]))
    keys = _randn(_gen(seed), case["n"], case["d"]).double()
    return dict(codes=None, scales=0.9957 * keys.square().mean(1).sqrt())
