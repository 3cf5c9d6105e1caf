"""The encoder forward's workloads at the sizes its users run, as timed and checked cases.

A case is a dict with a "kind":

  request    one row through a whole model, ids to option logits: HipModel.forward
  serve      rows in micro-batches, two in flight: HipModel.submit / collect
  batch      one packed batch through a whole model: HipModel.forward
  layer      the first encoder layer from token ids to the residual stream, kernel by kernel
  attention  attention over a packed batch (one launch)
  qkv        LayerNorm + Wqkv + RoPE of a few tokens (one launch)
  head       the marker rows' half of the last decision-head layer, and the scorer

"hidden" is 384 (the Julia-1 shape) or 768 (ModernBERT-base); the other sizes follow from it.  Row lengths are
drawn between "lo" and "hi" from "mix", so that a case has the same lengths whatever the seed of its inputs.
"""
import math
import os
import random
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "julia1-rs_amd"))

from julia1_amd import abi, hip, synth  # noqa: E402

INTER = 1152          # GEGLU width of both shapes
VOCAB = 50368
HALF_WINDOW = 64      # sliding-window layers: |i - j| <= 64
THETA = {True: 160000.0, False: 10000.0}  # global, sliding-window
EPS = 1e-5
SHAPES = {384: "julia1", 768: "modernbert-base"}
MICRO = 16            # rows per micro-batch of the serving path
WORKSPACE = 24 << 20  # FP32 partial sums of the small-batch GEMMs, as the model keeps
LONG = 4096           # rows from this length on run 256-query attention items


def listed():
    return [
        # One decision among 20 options, about 160 tokens: the latency a caller of the service sees.
        dict(name="request_384", kind="request", hidden=384, tokens=161, options=20),
        # Offline scoring: rows of 32 to 554 tokens in micro-batches of 16, the next packed while one runs.
        dict(name="serve_384", kind="serve", hidden=384, rows=64, lo=32, hi=554, mix=12),
        # The headline batch: 32 rows of 64 to 512 tokens, packed.
        dict(name="batch_768", kind="batch", hidden=768, rows=32, lo=64, hi=512, mix=1),
        # Attention of a single request's window layer: the smallest launch of the path.
        dict(name="attention_request", kind="attention", hidden=384, rows=1, lo=161, hi=161, mix=0, window=HALF_WINDOW),
        # Sliding-window attention of the headline batch (two layers of three).
        dict(name="attention_window", kind="attention", hidden=768, rows=32, lo=64, hi=512, mix=1, window=HALF_WINDOW),
        # Full attention of a request at the longest position the model takes.
        dict(name="attention_long", kind="attention", hidden=768, rows=1, lo=8192, hi=8192, mix=0, window=-1),
        # The first projection of a single request.
        dict(name="qkv_request", kind="qkv", hidden=384, tokens=161),
        # One layer of a serving micro-batch (16 rows).
        dict(name="layer_384", kind="layer", hidden=384, rows=16, lo=32, hi=554, mix=5, window=HALF_WINDOW),
        # One full-attention layer of a long document.
        dict(name="layer_384_long", kind="layer", hidden=384, rows=1, lo=3928, hi=3928, mix=0, window=-1),
        # One full-attention layer of the headline batch.
        dict(name="layer_768", kind="layer", hidden=768, rows=32, lo=64, hi=512, mix=1, window=-1),
        # One window layer of a router's batch: 256 rows of 32 to 1024 tokens.
        dict(name="layer_768_router", kind="layer", hidden=768, rows=256, lo=32, hi=1024, mix=4, window=HALF_WINDOW),
        # The options of the headline batch through the decision head's last layer.
        dict(name="head_768", kind="head", hidden=768, markers=382),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["request", "serve", "batch", "layer", "layer", "attention", "attention", "qkv", "head"])
    hidden = rng.choice([384, 768])
    c = dict(kind=kind, hidden=hidden)
    if kind == "request":
        c.update(tokens=_log_int(rng, 16, 1200), options=rng.randint(8, 20))
    elif kind == "qkv":
        c.update(tokens=_log_int(rng, 1, 512))
    elif kind == "head":
        c.update(markers=_log_int(rng, 2, 5120))
    else:
        # rows of one packed batch, up to the token count of the largest listed case of the kind
        most = {"serve": 18752, "batch": 9216, "layer": 131072, "attention": 32768}[kind]
        hi = _log_int(rng, 32, 1024 if kind in ("serve", "batch") else 8192)
        lo = max(1, _log_int(rng, max(1, hi // 8), hi))
        rows = max(1, min(256, _log_int(rng, 1, max(1, most // hi))))
        c.update(rows=rows, lo=lo, hi=hi, mix=rng.randint(0, 999))
        if kind in ("layer", "attention"):
            # full attention's work grows with the square of the length: the largest is attention_long's
            whole = rows * hi * hi <= 8192 * 8192
            c.update(window=rng.choice([HALF_WINDOW, -1]) if whole else HALF_WINDOW)
    return c


# ---------------------------------------------------------------- inputs

def lengths(case):
    if case["kind"] in ("request", "qkv"):
        return [case["tokens"]]
    r = random.Random(case["mix"])
    return [r.randint(case["lo"], case["hi"]) for _ in range(case["rows"])]


def option_counts(case, rows):
    if case["kind"] == "request":
        return [case["options"]]
    r = random.Random(case["mix"] + 1)
    return [r.randint(2, 20) for _ in range(rows)]


_models = {}


def model(hidden):
    """The loaded model of a shape, kept as a server keeps it: (its weights, the handle)."""
    if hidden not in _models:
        cfg = synth.model_config(SHAPES[hidden])
        ws = abi.WeightSet(cfg, synth.make_weights(cfg, seed=0))
        _models[hidden] = (ws, hip.HipModel(ws))
    return _models[hidden]


def batches(case, seed):
    """The packed batches of a whole-model case: one, or one per micro-batch of rows sorted by length."""
    lens = lengths(case)
    opts = option_counts(case, len(lens))
    step = len(lens)
    if case["kind"] == "serve":
        order = sorted(range(len(lens)), key=lambda i: lens[i])
        lens, opts, step = [lens[i] for i in order], [opts[i] for i in order], MICRO
    return [synth.make_batch(np.array(lens[i:i + step]), opts[i:i + step], VOCAB, seed * 1000 + i)
            for i in range(0, len(lens), step)]


class Draws:
    """Normal and integer device tensors from one seed; matrices as bf16, as the model keeps them."""

    def __init__(self, seed):
        self.g = torch.Generator("cuda").manual_seed(int(seed) + 1)

    def normal(self, *shape, std=1.0):
        return torch.randn(*shape, generator=self.g, device="cuda") * std

    def matrix(self, n, k):
        return (self.normal(n, k, std=0.02)).bfloat16()

    def below(self, bound, n):
        return torch.randint(0, bound, (n,), generator=self.g, device="cuda", dtype=torch.int32)


def tiles(lens, nq):
    """Attention work items of at most nq queries each, costliest first."""
    out, row = [], 0
    for n in lens:
        out += [(row + q, min(nq, n - q), row, n, q) for q in range(0, n, nq)]
        row += n
    out.sort(key=lambda t: -t[1] * t[3])
    return torch.tensor(out, dtype=torch.int32, device="cuda")


def positions(lens):
    return torch.cat([torch.arange(n, dtype=torch.int32) for n in lens]).cuda()


def rope(theta, n):
    c, s = hip.rope_table(theta, max(n, 64))
    return torch.from_numpy(c).cuda(), torch.from_numpy(s).cuda()


def weights(case, seed):
    """The layer's or head's own numbers (also what exact() computes from)."""
    d, h, kind = Draws(seed), case["hidden"], case["kind"]
    if kind == "layer":
        return dict(ids=d.below(VOCAB, sum(lengths(case))), table=d.normal(VOCAB, h, std=0.02),
                    emb_w=1 + d.normal(h, std=0.02), wqkv=d.matrix(3 * h, h), wo=d.matrix(h, h),
                    mlp_w=1 + d.normal(h, std=0.02), wi=d.matrix(2 * INTER, h), wo2=d.matrix(h, INTER))
    if kind == "attention":
        # q and k as Wqkv leaves them for normalised rows: standard deviation 0.02 * sqrt(hidden)
        return dict(qkv=d.normal(sum(lengths(case)), 3 * h, std=0.02 * math.sqrt(h)).bfloat16())
    if kind == "qkv":
        return dict(x=d.normal(case["tokens"], h), ln_w=1 + d.normal(h, std=0.02), wqkv=d.matrix(3 * h, h))
    m = case["markers"]
    return dict(x=d.normal(4 * m, h), rows=torch.sort(torch.randperm(4 * m, generator=d.g, device="cuda")[:m])[0].int(),
                ctx=d.normal(m, h, std=0.5).bfloat16(), out_w=d.matrix(h, h), out_b=d.normal(h, std=0.02),
                n2_w=1 + d.normal(h, std=0.02), n2_b=d.normal(h, std=0.02), lin1=d.matrix(4 * h, h),
                b1=d.normal(4 * h, std=0.02), lin2=d.matrix(h, 4 * h), b2=d.normal(h, std=0.02),
                sn_w=1 + d.normal(h, std=0.02), sn_b=d.normal(h, std=0.02), s_w1=d.matrix(h, h),
                s_b1=d.normal(h, std=0.02), s_w2=d.normal(h, std=0.02))


def few(rows, n):
    """Whether a projection's output is too small for the GPU without splitting K, as the model decides it."""
    return -(-n // 128) * -(-rows // 128) < 128


def linear(w, rows, workspace, epi):
    """run(x, out, **epilogue operands) of one projection as the model launches it: weight-stationary from a packed
    copy of W where that kernel takes the shape and the batch fills the GPU, the general entry point otherwise."""
    n, k = w.shape
    stationary = (k == 768 and n % 256 == 0) or (k == 1152 and n % 128 == 0 and epi == abi.EPI_RESID_F32)
    if stationary and not few(rows, n):
        packed = hip.pack_ws(w)
        return lambda x, out, **kw: hip.op_gemm_ws(epi, x, packed, n, k, out, **kw)
    return lambda x, out, **kw: hip.op_gemm_splitk(epi, x, w, out, workspace, **kw)


def empty(rows, n, dtype=torch.bfloat16):
    return torch.empty(rows, n, dtype=dtype, device="cuda")


def prepare(case, seed):
    kind, h = case["kind"], case["hidden"]
    if kind in ("request", "serve", "batch"):
        return dict(kind=kind, model=model(h)[1], batches=batches(case, seed))
    s = weights(case, seed)
    s.update(kind=kind, hidden=h)
    if kind == "qkv":
        s["cos"], s["sin"] = rope(THETA[False], case["tokens"])
        s["pos"] = positions([case["tokens"]])
        s["out"] = empty(case["tokens"], 3 * h)
        return s
    if kind in ("layer", "attention"):
        lens = lengths(case)
        t = sum(lens)
        s["window"] = case["window"]
        # full attention over long rows: 256-query items, and 128-query ones for the batch's other rows
        s["wide"] = case["window"] < 0 and min(lens) >= LONG
        s["tiles"] = tiles(lens, 256 if s["wide"] else 128)
        s["ctx"] = empty(t, h)
        if kind == "attention":
            return s
        ws = torch.empty(WORKSPACE // 4, device="cuda")
        wi = hip.interleave_geglu(s.pop("wi").float().cpu().numpy())
        s["qkv_of"] = linear(s["wqkv"], t, ws, abi.EPI_ROPE_BF16)
        s["wo_of"] = linear(s["wo"], t, ws, abi.EPI_RESID_F32)
        s["wi_of"] = linear(torch.from_numpy(wi).cuda().bfloat16(), t, ws, abi.EPI_GEGLU_BF16)
        s["wo2_of"] = linear(s["wo2"], t, ws, abi.EPI_RESID_F32)
        s["cos"], s["sin"] = rope(THETA[case["window"] < 0], max(lens))
        s["pos"] = positions(lens)
        s.update(x=empty(t, h, torch.float32), xn=empty(t, h), qkv=empty(t, 3 * h), g=empty(t, INTER))
        return s
    m = case["markers"]
    ws = torch.empty(WORKSPACE // 4, device="cuda")
    s["out_of"] = linear(s["out_w"], m, ws, abi.EPI_RESID_F32)
    s["lin1_of"] = linear(s["lin1"], m, ws, abi.EPI_BIAS_RELU_BF16)
    s["lin2_of"] = linear(s["lin2"], m, ws, abi.EPI_RESID_F32)
    s["scorer_of"] = linear(s["s_w1"], m, ws, abi.EPI_BIAS_F32)
    s.update(y=empty(m, h, torch.float32), yn=empty(m, h), hm=empty(m, 4 * h), z=empty(m, h, torch.float32),
             score=torch.empty(m, device="cuda"))
    return s


# ---------------------------------------------------------------- one pass

def run(s):
    kind = s["kind"]
    if kind in ("request", "batch"):
        return s["model"].forward(s["batches"][0])
    if kind == "serve":
        model_, out, flying = s["model"], [], []
        for b in s["batches"]:
            if len(flying) == 2:
                out.append(model_.collect(*flying.pop(0)))
            flying.append((model_.submit(b), b.marker_rows.size))
        return out + [model_.collect(*f) for f in flying]
    h = s["hidden"]
    if kind == "qkv":
        hip.op_gemm_ln(abi.EPI_ROPE_BF16, s["x"], s["wqkv"], s["out"], s["ln_w"], eps=EPS, pos=s["pos"], cos=s["cos"],
                       sin=s["sin"], rope_cols=2 * h)
        return s["out"]
    if kind == "attention":
        return attend(s)
    if kind == "layer":
        hip.op_embed_ln(s["ids"], s["table"], s["emb_w"], EPS, s["x"], s["xn"])
        s["qkv_of"](s["xn"], s["qkv"], pos=s["pos"], cos=s["cos"], sin=s["sin"], rope_cols=2 * h)
        attend(s)
        s["wo_of"](s["ctx"], s["x"])
        hip.op_layer_norm(s["x"], s["mlp_w"], None, EPS, s["xn"])
        s["wi_of"](s["xn"], s["g"])
        s["wo2_of"](s["g"], s["x"])
        return s["x"]
    hip.op_gather_f32(s["x"], s["rows"], s["y"])
    s["out_of"](s["ctx"], s["y"], bias=s["out_b"])
    hip.op_layer_norm(s["y"], s["n2_w"], s["n2_b"], EPS, s["yn"])
    s["lin1_of"](s["yn"], s["hm"], bias=s["b1"])
    s["lin2_of"](s["hm"], s["y"], bias=s["b2"])
    hip.op_layer_norm(s["y"], s["sn_w"], s["sn_b"], EPS, s["yn"])
    s["scorer_of"](s["yn"], s["z"], bias=s["s_b1"])
    hip.op_scorer(s["z"], s["s_w2"], 0.0, s["score"])
    return [s["y"], s["score"]]


def attend(s):
    h, q = s["hidden"], s["qkv"]
    hip.op_attention(q, 3 * h, q[:, h:], q[:, 2 * h:], 3 * h, s["ctx"], h, s["tiles"], h // 64, s["window"],
                     wide=s["wide"])
    return s["ctx"]


# ---------------------------------------------------------------- what a pass cannot do without

def pairs(n, window):
    """Attended (query, key) pairs of a row."""
    if window < 0:
        return n * n
    return sum(min(i + window, n - 1) - max(i - window, 0) + 1 for i in range(n))


def work(case):
    kind, h = case["kind"], case["hidden"]
    if kind == "head":
        m = case["markers"]
        params = 10 * h * h
        return dict(bytes=2 * params + m * h * (4 + 2 + 4) + 4 * m, flops=2 * m * params)
    lens = lengths(case)
    t = sum(lens)
    if kind == "qkv":
        return dict(bytes=t * h * 4 + 3 * h * h * 2 + t * 3 * h * 2, flops=2 * t * 3 * h * h)
    if kind == "attention":
        return dict(bytes=t * 4 * h * 2, flops=4 * h * sum(pairs(n, case["window"]) for n in lens))
    params = 4 * h * h + 3 * INTER * h  # of one encoder layer
    if kind == "layer":
        return dict(bytes=t * (h * 8 + 4) + 2 * params,
                    flops=2 * t * params + 4 * h * sum(pairs(n, case["window"]) for n in lens))
    opts = sum(option_counts(case, len(lens)))
    enc = 2 * t * 22 * params + 4 * h * sum(8 * pairs(n, -1) + 14 * pairs(n, HALF_WINDOW) for n in lens)
    head = 2 * t * 14 * h * h + 2 * opts * 11 * h * h + 4 * h * sum(pairs(n, -1) for n in lens)
    passes = len(lens) // MICRO if kind == "serve" else 1
    return dict(bytes=max(1, passes) * 2 * (22 * params + 25 * h * h) + t * (h * 4 + 4) + opts * 4, flops=enc + head)


def tolerance(case):
    # About four times what the model's two summation orders (split K on and off) differ by, and no less than twice
    # the distance to exact() that rounding to bf16 alone gives.
    if case["kind"] in ("request", "serve", "batch"):
        return {"rel": 1e-2, "max": 4e-2}  # logits behind 24 layers of bf16 activations (measured 2e-3)
    if case["kind"] == "layer":
        return {"rel": 1e-3, "max": 1e-2}  # FP32 residual rows plus bf16 branches (measured 4e-4)
    return {"rel": 6e-3, "max": 4e-2}      # bf16 outputs (measured 2.4e-3)


# ---------------------------------------------------------------- the same in 64 bits

def _f64(a):
    return (a if torch.is_tensor(a) else torch.from_numpy(np.ascontiguousarray(a))).cuda().double()


def _bf(a):
    """FP32 matrix -> its bf16 values, in 64 bits."""
    return torch.from_numpy(a).cuda().bfloat16().double()


def _norm(x, w, b=None, eps=EPS):
    y = (x - x.mean(1, keepdim=True)) / torch.sqrt(x.var(1, keepdim=True, unbiased=False) + eps) * w
    return y if b is None else y + b


def _table(theta, pos):
    """cos and sin rows [T, 32] of the tokens' positions; angles are FP32 products of FP32 frequencies, as the model's."""
    inv = np.float32(1) / np.power(np.float32(theta), np.arange(0, 64, 2, dtype=np.float32) / np.float32(64))
    a = (pos.cpu().numpy().astype(np.float32)[:, None] * inv.astype(np.float32)).astype(np.float64)
    return [torch.from_numpy(f(a)).cuda() for f in (np.cos, np.sin)]


def _rotate(x, cos, sin):
    """Rotate-half RoPE of [T, heads * 64] with per-token rows cos, sin [T, 32]."""
    t = x.view(x.shape[0], -1, 2, 32)
    c, s = cos[:, None], sin[:, None]
    return torch.stack([t[:, :, 0] * c - t[:, :, 1] * s, t[:, :, 1] * c + t[:, :, 0] * s], 2).reshape(x.shape)


def _attend(q, k, v, qrows, lens, window):
    """softmax(q k' / 8) v per head; qrows: per row of the batch, its queries' (first, count) in q."""
    out, row = torch.empty_like(q), 0
    for (q0, nq), n in zip(qrows, lens):
        for c in range(0, q.shape[1], 64):
            kk, vv = k[row:row + n, c:c + 64], v[row:row + n, c:c + 64]
            for a in range(0, nq, 2048):
                b = min(nq, a + 2048)
                s = q[q0 + a:q0 + b, c:c + 64] @ kk.T / 8
                if window >= 0:
                    i = torch.arange(a, b, device="cuda")[:, None]
                    s = s.masked_fill((i - torch.arange(n, device="cuda")).abs() > window, -math.inf)
                out[q0 + a:q0 + b, c:c + 64] = torch.softmax(s, 1) @ vv
        row += n
    return out


def _self_attend(qkv, lens, window):
    h = qkv.shape[1] // 3
    first = np.concatenate([[0], np.cumsum(lens)])
    return _attend(qkv[:, :h], qkv[:, h:2 * h], qkv[:, 2 * h:], list(zip(first, lens)), lens, window)


def _layer(x, xn, lens, window, table, wqkv, wo, mlp_w, wi, wo2):
    h = x.shape[1]
    qkv = xn @ wqkv.T
    qkv = torch.cat([_rotate(qkv[:, :h], *table), _rotate(qkv[:, h:2 * h], *table), qkv[:, 2 * h:]], 1)
    x = x + _self_attend(qkv, lens, window) @ wo.T
    u = _norm(x, mlp_w) @ wi.T
    return x + (torch.nn.functional.gelu(u[:, :INTER]) * u[:, INTER:]) @ wo2.T


def _forward(ws, b):
    """The whole model on one batch: embedding, encoder, decision head, scorer."""
    t, cfg = ws.tensors, ws.cfg
    f = lambda name: _f64(t[name])  # noqa: E731
    m = lambda name: _bf(t[name])   # noqa: E731
    lens = [int(n) for n in b.lens]
    table = {g: _table(THETA[g], positions(lens)) for g in (True, False)}
    ids = torch.from_numpy(b.ids.astype(np.int64))
    x = _norm(_f64(torch.from_numpy(t["encoder.embeddings.tok_embeddings.weight"])[ids]), f("encoder.embeddings.norm.weight"))
    for l in range(cfg.layers):
        p, g = f"encoder.layers.{l}.", bool(cfg.global_[l])
        xn = x if l == 0 else _norm(x, f(p + "attn_norm.weight"))
        x = _layer(x, xn, lens, -1 if g else HALF_WINDOW, table[g], m(p + "attn.Wqkv.weight"), m(p + "attn.Wo.weight"),
                   f(p + "mlp_norm.weight"), m(p + "mlp.Wi.weight"), m(p + "mlp.Wo.weight"))
    qt = torch.from_numpy(np.repeat(b.qtypes.astype(np.int64), b.lens)).cuda()
    x = _norm(x, f("encoder.final_norm.weight")) + f("type_emb.weight")[qt]
    rows = torch.from_numpy(b.marker_rows.astype(np.int64)).cuda()
    first = np.concatenate([[0], np.cumsum(lens)])
    for l in range(cfg.head_layers):
        p, last = f"head.layers.{l}.", l + 1 == cfg.head_layers
        w, bias = m(p + "self_attn.in_proj_weight"), f(p + "self_attn.in_proj_bias")
        qkv = _norm(x, f(p + "norm1.weight"), f(p + "norm1.bias")) @ w.T + bias
        h = x.shape[1]
        if last:
            q, x = qkv[rows, :h], x[rows]
            qrows = list(zip(b.marker_starts[:-1], np.diff(b.marker_starts)))
        else:
            q, qrows = qkv[:, :h], list(zip(first, lens))
        c = _attend(q, qkv[:, h:2 * h], qkv[:, 2 * h:], qrows, lens, -1)
        x = x + c @ m(p + "self_attn.out_proj.weight").T + f(p + "self_attn.out_proj.bias")
        u = torch.relu(_norm(x, f(p + "norm2.weight"), f(p + "norm2.bias")) @ m(p + "linear1.weight").T + f(p + "linear1.bias"))
        x = x + u @ m(p + "linear2.weight").T + f(p + "linear2.bias")
    z = _norm(x, f("scorer.0.weight"), f("scorer.0.bias")) @ m("scorer.1.weight").T + f("scorer.1.bias")
    return (torch.nn.functional.gelu(z) @ f("scorer.3.weight")[0] + f("scorer.3.bias")).cpu().numpy()


def exact(case, seed):
    kind, h = case["kind"], case["hidden"]
    if kind in ("request", "batch"):
        return _forward(model(h)[0], batches(case, seed)[0])
    if kind == "serve":
        return [_forward(model(h)[0], b) for b in batches(case, seed)]
    s = {k: v.double() if v.is_floating_point() else v for k, v in weights(case, seed).items()}
    if kind == "attention":
        return _self_attend(s["qkv"], lengths(case), case["window"])
    if kind == "qkv":
        table = _table(THETA[False], positions([case["tokens"]]))
        qkv = _norm(s["x"], s["ln_w"]) @ s["wqkv"].T
        return torch.cat([_rotate(qkv[:, :h], *table), _rotate(qkv[:, h:2 * h], *table), qkv[:, 2 * h:]], 1)
    if kind == "layer":
        lens = lengths(case)
        table = _table(THETA[case["window"] < 0], positions(lens))
        x = _norm(s["table"][s["ids"].long()], s["emb_w"])
        return _layer(x, x, lens, case["window"], table, s["wqkv"], s["wo"], s["mlp_w"], s["wi"], s["wo2"])
    y = s["x"][s["rows"].long()] + s["ctx"] @ s["out_w"].T + s["out_b"]
    u = torch.relu(_norm(y, s["n2_w"], s["n2_b"]) @ s["lin1"].T + s["b1"])
    y = y + u @ s["lin2"].T + s["b2"]
    z = _norm(y, s["sn_w"], s["sn_b"]) @ s["s_w1"].T + s["s_b1"]
    return [y, torch.nn.functional.gelu(z) @ s["s_w2"]]
