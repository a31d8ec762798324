"""The calls that a user of the Q8_0 linear path makes, as measurable cases.

A case is a dict of plain values; `prepare` sets up what a program holds
before the call (a context, registered weights, buffers and, where a step is
replayed, its captured graph), `run` is one pass through the public entry
points, `exact` the same function in float64 with plain torch.

Kinds
  linear     `weights` linears of one shape on one input, each its own call
             (add: the residual-add entry instead, no activation)
  mlp        `layers` SwiGLU MLPs, each on the same input
  layer      `layers` chained linear-attention layers of the model as the
             model builder emits them around the Q8_0 linears: input norm
             and in_proj group, gated norm (a fixed stand-in for the mixer's
             core, which is not on this path), out_proj + residual, post
             norm, SwiGLU, down_proj + residual
  lm_head    last-row logits and argmax over the vocabulary table
  embedding  the gather from that table

`graph` replays the pass from one captured graph, as a decode step or a
fixed-size prompt chunk is run; without it the calls are made one by one.
The dimensions are those of the 4B-class configuration in
llmcp_amd/model_arena.py and of bench.py; the ragged ones are generic.
"""
import math

import torch

import llmcp_amd as q8

EPS = 1e-6
ACTIVATIONS = ("none", "silu", "sigmoid", "softplus")


def _case(kind, **kw):
    c = {"kind": kind, "m": 1, "dtype": "f32", "platform": "aarch64", "accum": "exact",
         "graph": False}
    c.update(kw)
    return c


def _linear(m, n, k, **kw):
    return _case("linear", m=m, n=n, k=k, **dict({"act": "none", "add": False, "weights": 1}, **kw))


def _mlp(m, h, f, **kw):
    return _case("mlp", m=m, h=h, f=f, **dict({"layers": 1}, **kw))


def _layer(m, h, f, qkv, z, **kw):
    return _case("layer", m=m, h=h, f=f, qkv=qkv, z=z, dtype="bf16",
                 **dict({"layers": 1}, **kw))


def listed():
    return [
        # one projection of one token, called by itself: launch and latency
        dict(_linear(1, 2560, 2560), name="decode_linear_f32"),
        # the MLPs of a decode step (bench.py's headline step)
        dict(_mlp(1, 2560, 9216, layers=6, graph=True), name="decode_mlp_f32"),
        # four layers of a decode step with their norms, bf16 hidden state
        dict(_layer(1, 2560, 9216, 8192, 4096, layers=4, graph=True), name="decode_layers_bf16"),
        # the end of a decode step: logits over the tied table and the token
        dict(_case("lm_head", vocab=248320, h=2560, dtype="bf16"), name="decode_lm_head_bf16"),
        # a prompt of a few tokens (a chat turn's tail) through one layer
        dict(_layer(7, 2560, 9216, 8192, 4096, graph=True), name="prompt_layer_m7_bf16"),
        # a short prompt through one MLP
        dict(_mlp(19, 2560, 9216, graph=True), name="prompt_mlp_m19_f32"),
        # the gate projection of a small prompt chunk
        dict(_linear(64, 9216, 2560, weights=4, graph=True), name="prefill_linear_m64_f32"),
        # odd sizes on the x86 platform's arithmetic: K of 69 blocks, ragged
        # tiles in M and N, an activation
        dict(_linear(45, 1000, 2208, weights=4, act="sigmoid", platform="x86", dtype="bf16",
                     graph=True), name="ragged_linear_m45_x86_bf16"),
        # a prompt chunk with the split-K accumulation a program may opt into
        dict(_mlp(200, 2560, 9216, accum="split_k"), name="prefill_mlp_m200_split_f32"),
        # a prompt of a few hundred tokens through one layer
        dict(_layer(333, 2560, 9216, 8192, 4096), name="prefill_layer_m333_bf16"),
        # a long prompt chunk through one MLP (the largest)
        dict(_mlp(1024, 2560, 9216), name="prefill_mlp_m1024_f32"),
        # a long prompt's token embeddings
        dict(_case("embedding", m=1024, vocab=248320, h=2560, dtype="bf16"),
             name="prompt_embedding_m1024_bf16"),
    ]


def _log_int(rng, lo, hi, step=1):
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return min(hi, max(lo, int(round(v / step)) * step))


def draw(rng):
    kind = rng.choice(("linear", "linear", "linear", "mlp", "mlp", "layer", "layer", "lm_head",
                       "embedding"))
    dtype = rng.choice(("f32", "bf16"))
    platform = rng.choice(("aarch64", "aarch64", "x86"))
    accum = rng.choice(("exact", "exact", "split_k"))
    m = 1 if rng.random() < 0.2 else _log_int(rng, 2, 1024)
    opts = dict(dtype=dtype, platform=platform, accum=accum)
    if kind == "linear":
        add = rng.random() < 0.25
        return _linear(m, _log_int(rng, 256, 9216, 8), _log_int(rng, 256, 9216, 32), add=add,
                       act="none" if add else rng.choice(ACTIVATIONS), weights=4,
                       graph=m <= 128, **opts)
    if kind == "mlp":
        return _mlp(m, _log_int(rng, 512, 2560, 32), _log_int(rng, 1024, 9216, 32),
                    layers=4 if m == 1 else 1, graph=m <= 128, **opts)
    if kind == "layer":
        m = min(m, _log_int(rng, 256, 512))
        return _layer(m, _log_int(rng, 512, 2560, 32), _log_int(rng, 1024, 9216, 32),
                      _log_int(rng, 1024, 8192, 128), _log_int(rng, 512, 4096, 128),
                      layers=2 if m == 1 else 1, graph=m <= 128, platform=platform, accum=accum)
    vocab = _log_int(rng, 32000, 248320, 8)
    if kind == "lm_head":
        return _case("lm_head", vocab=vocab, h=_log_int(rng, 512, 2560, 32), dtype=dtype,
                     platform=platform)
    return _case("embedding", m=_log_int(rng, 1, 2048), vocab=vocab,
                 h=_log_int(rng, 512, 2560, 32), dtype=dtype)


# ------------------------------------------------------------- the inputs --

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 7919 + 17)
    return g


def _randn(g, *shape, scale=1.0):
    return torch.randn(*shape, generator=g, device="cuda") * scale


def _weight(g, n, k):
    """N(0, 0.02) weights as Q8_0: int8 values [n, k/32, 32] and f16 scales
    [n, k/32] (scale = max|w| / 127, rounding half away from zero)."""
    w = _randn(g, n, k, scale=0.02).view(n, k // 32, 32)
    scale = w.abs().amax(-1, keepdim=True) / 127.0
    r = w / scale
    q = torch.where(r < 0, -torch.floor(0.5 - r), torch.floor(0.5 + r)).to(torch.int8)
    return q, scale.squeeze(-1).to(torch.float16)


def _cast(x, dtype):
    return x.to(torch.bfloat16) if dtype == "bf16" else x


def _linear_shapes(c):
    """(name, n, k) of one layer's weights."""
    h, f = c["h"], c["f"]
    if c["kind"] == "mlp":
        return [("gate", f, h), ("up", f, h), ("down", h, f)]
    return [("qkv", c["qkv"], h), ("z", c["z"], h), ("a", 32, h), ("b", 32, h),
            ("out", h, c["z"]), ("gate", f, h), ("up", f, h), ("down", h, f)]


def _inputs(c, seed):
    g, m, dt, kind = _gen(seed), c["m"], c["dtype"], c["kind"]
    d = {}
    if kind == "linear":
        d["x"] = _cast(_randn(g, m, c["k"]), dt)
        if c["add"]:
            d["r"] = _cast(_randn(g, m, c["n"]), dt)
        d["w"] = [_weight(g, c["n"], c["k"]) for _ in range(c["weights"])]
    elif kind == "mlp":
        d["x"] = _cast(_randn(g, m, c["h"]), dt)
        d["w"] = [{s: _weight(g, n, k) for s, n, k in _linear_shapes(c)}
                  for _ in range(c["layers"])]
    elif kind == "layer":
        d["x"] = _cast(_randn(g, m, c["h"], scale=2.0), dt)
        d["v"] = _cast(_randn(g, m, c["z"]), dt)
        d["w"] = []
        for _ in range(c["layers"]):
            w = {s: _weight(g, n, k) for s, n, k in _linear_shapes(c)}
            w["ln"] = _cast(_randn(g, c["h"], scale=0.1), dt)
            w["post"] = _cast(_randn(g, c["h"], scale=0.1), dt)
            w["gn"] = _randn(g, 128, scale=0.1) + 1.0
            d["w"].append(w)
    else:
        d["w"] = _weight(g, c["vocab"], c["h"])
        if kind == "lm_head":
            d["x"] = _cast(_randn(g, 1, c["h"]), dt)
        else:
            d["ids"] = torch.randint(0, c["vocab"], (m,), generator=g, device="cuda")
    return d


# ---------------------------------------------------------- the framework --

class _Buf:
    """A torch tensor as the front end takes buffers (by address)."""

    def __init__(self, tensor):
        self.tensor, self.ptr = tensor, tensor.data_ptr()


_stream = None


def _program_stream():
    """The one stream that all passes are queued on, as one program queues
    its steps (contexts left on streams of their own would run side by
    side)."""
    global _stream
    if _stream is None:
        _stream = torch.cuda.Stream()
    return _stream.cuda_stream


class _State:
    """One program: its context, weights, buffers and captured pass."""

    def __init__(self, case):
        self.case, self.graph, self.keep = case, None, []
        self.ctx = q8.Context(0)
        q8.check(q8.lib().llmcp_q8_ctx_set_stream(self.ctx.handle, _program_stream()))
        self.ctx.set_platform(case["platform"])
        self.ctx.set_accumulation(case["accum"])

    def buf(self, tensor):
        self.keep.append(_Buf(tensor))
        return self.keep[-1]

    def out(self, *shape, dtype=None):
        dt = dtype or self.case["dtype"]
        return self.buf(torch.empty(*shape, device="cuda",
                                    dtype=torch.bfloat16 if dt == "bf16" else torch.float32))

    def weight(self, qd):
        """Registers Q8_0 values and scales, packed as the arena's q8_0_p4
        records (4 scales, then 8 chunks of 4 rows x 4 values)."""
        q, d = qd
        n, b = d.shape
        rec = torch.empty(n // 4, b, 136, dtype=torch.uint8, device="cuda")
        rec[:, :, :8] = d.view(n // 4, 4, b).transpose(1, 2).contiguous().view(torch.uint8)
        rec[:, :, 8:] = (q.view(n // 4, 4, b, 8, 4).permute(0, 2, 3, 1, 4)
                         .reshape(n // 4, b, 128).view(torch.uint8))
        torch.cuda.synchronize()
        return self.ctx.register_device_p4(self.buf(rec), n, 32 * b)

    def __del__(self):
        try:
            if self.graph is not None:
                self.ctx.sync()
                self.ctx.graph_destroy(self.graph)
            self.ctx.close()
        except Exception:
            pass


def prepare(case, seed):
    c, m, dt, kind = case, case["m"], case["dtype"], case["kind"]
    d = _inputs(c, seed)
    s = _State(c)
    ctx, mode = s.ctx, "decode" if m == 1 else "prefill"
    if kind == "linear":
        x = s.buf(d["x"])
        ws = [s.weight(w) for w in d["w"]]
        ys = [s.out(m, c["n"]) for _ in ws]
        r = s.buf(d["r"]) if c["add"] else None

        def calls():
            for w, y in zip(ws, ys):
                if r is not None:
                    ctx.linear_add(x, w, r, y, m, mode=mode, dtype=dt)
                else:
                    ctx.linear(x, w, y, m, activation=c["act"], mode=mode, dtype=dt)
        s.outputs = [y.tensor for y in ys]
    elif kind == "mlp":
        x = s.buf(d["x"])
        ws = [{k: s.weight(v) for k, v in w.items()} for w in d["w"]]
        hs = [s.out(m, c["f"]) for _ in ws]
        ys = [s.out(m, c["h"]) for _ in ws]

        def calls():
            for w, h, y in zip(ws, hs, ys):
                ctx.mlp(x, w["gate"], w["up"], w["down"], y, h=h, m=m, mode=mode, dtype=dt)
        s.outputs = [t.tensor for t in hs + ys]
    elif kind == "layer":
        h, z, group = c["h"], c["z"], ("qkv", "z", "a", "b")
        v = s.buf(d["v"])
        hidden = [s.buf(d["x"])] + [s.out(m, h) for _ in d["w"]]
        ws = [{k: s.buf(t) if k in ("ln", "post", "gn") else s.weight(t) for k, t in w.items()}
              for w in d["w"]]
        outs = [[s.out(m, w[k].rows) for k in group] for w in ws]
        mid = [s.out(m, h) for _ in ws]
        n1, n2, gated, up = s.out(m, h), s.out(m, h), s.out(m, z), s.out(m, c["f"])

        def calls():
            for i, w in enumerate(ws):
                ctx.rmsnorm_linear_group(hidden[i], w["ln"], n1, [w[k] for k in group], outs[i],
                                         m, eps=EPS, zero_centered=True, mode=mode, dtype=dt)
                ctx.gated_rmsnorm(v, outs[i][1], w["gn"], gated, m, z, 128, eps=EPS, dtype=dt)
                ctx.linear_add(gated, w["out"], hidden[i], mid[i], m, mode=mode, dtype=dt)
                ctx.rmsnorm(mid[i], w["post"], n2, m, h, eps=EPS, zero_centered=True, dtype=dt)
                ctx.swiglu(n2, w["gate"], w["up"], up, m, mode=mode, dtype=dt)
                ctx.linear_add(up, w["down"], mid[i], hidden[i + 1], m, mode=mode, dtype=dt)
        s.outputs = [[t.tensor for t in o + [a, b]] for o, a, b in zip(outs, mid, hidden[1:])]
    elif kind == "lm_head":
        x, w = s.buf(d["x"]), s.weight(d["w"])
        logits = s.out(1, c["vocab"], dtype="f32")
        token = s.buf(torch.zeros(1, dtype=torch.int64, device="cuda"))

        def calls():
            ctx.lm_head(x, w, logits, 1, argmax=token, dtype=dt)
        s.outputs = [logits.tensor, token.tensor]
    else:
        ids, w, y = s.buf(d["ids"]), s.weight(d["w"]), s.out(m, c["h"])

        def calls():
            ctx.embedding(ids, m, w, y, dtype=dt)
        s.outputs = [y.tensor]
    s.calls = calls
    torch.cuda.synchronize()
    if c["graph"]:
        # once outside the capture: the workspace grows to this size
        calls()
        ctx.sync()
        ctx.graph_begin()
        calls()
        s.graph = ctx.graph_end()
    return s


def run(state):
    if state.graph is not None:
        state.ctx.graph_launch(state.graph)
    else:
        state.calls()
    return state.outputs


# ------------------------------------------------------------ the yardstick --

def work(case):
    c, m, kind = case, case["m"], case["kind"]
    e = 2 if c["dtype"] == "bf16" else 4
    q = lambda n, k: n * k * 34 // 32  # noqa: E731
    if kind == "linear":
        n, k, t = c["n"], c["k"], c["weights"]
        byt = t * (q(n, k) + m * n * e) + m * k * e + (m * n * e if c["add"] else 0)
        return {"bytes": byt, "flops": 2 * m * n * k * t}
    if kind in ("mlp", "layer"):
        shapes, t = _linear_shapes(c), c["layers"]
        byt = t * sum(q(n, k) for _, n, k in shapes)
        if kind == "mlp":
            byt += m * e * (c["h"] + t * (c["f"] + c["h"]))
        else:
            byt += m * e * (c["h"] + c["z"] + t * (2 * c["h"] + c["qkv"] + c["z"] + 64))
        return {"bytes": byt, "flops": t * sum(2 * m * n * k for _, n, k in shapes)}
    if kind == "lm_head":
        return {"bytes": q(c["vocab"], c["h"]) + c["vocab"] * 4 + c["h"] * e,
                "flops": 2 * c["vocab"] * c["h"]}
    return {"bytes": m * (q(1, c["h"]) + c["h"] * e + 8), "flops": m * c["h"]}


def tolerance(case):
    """f32 sums in another order move a linear's output by a few 1e-7 (1.6e-7
    from float64 at K = 2560); in an MLP they also move values of h across a
    rounding of the activation quantizer now and then, one int8 step of one
    value of thousands (5e-5 from float64).  A bf16 result may round the
    other way (one step of 2^-8 or 2^-7 of the value, for about one value in
    ten thousand), and in the chained layers the steps that follow see it."""
    kind, bf16 = case["kind"], case["dtype"] == "bf16"
    if kind == "embedding":
        return "exact"
    if kind == "lm_head":
        return {"rel": 2e-6}
    if kind == "linear":
        return {"rel": 2e-4, "max": 1e-2} if bf16 else {"rel": 2e-6}
    if kind == "mlp":
        return {"rel": 2e-3, "max": 3e-2} if bf16 else {"rel": 3e-4, "max": 1e-2}
    return {"rel": 1e-2, "max": 1e-1}


def _rnd(x, dtype):
    """The stored value of a float64 result: bf16 rows are rounded as such."""
    return x.float().to(torch.bfloat16).double() if dtype == "bf16" else x


def _q8_1(x):
    """Q8_1 activations: per 32 values d = max|x| / 127 and round(x / d) half
    to even, in f32 as the format defines them; returned dequantized."""
    v = x.float().view(x.shape[0], -1, 32)
    d = v.abs().amax(-1, keepdim=True) / 127.0
    inv = torch.where(d == 0, torch.zeros_like(d), 1.0 / d)
    return (torch.round(v * inv).double() * d.double()).reshape(x.shape)


def _matmul(x, qd):
    q, d = qd
    n, b = d.shape
    xq, step = _q8_1(x), 32768
    return torch.cat([xq @ (q[i:i + step].double() * d[i:i + step, :, None].double())
                      .reshape(-1, 32 * b).t() for i in range(0, n, step)], 1)


def _act(v, name):
    if name == "silu":
        return v / (1.0 + torch.exp(-v))
    if name == "sigmoid":
        return 1.0 / (1.0 + torch.exp(-v))
    if name == "softplus":
        return torch.log1p(torch.exp(v))
    return v


def _norm(x, w):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * w


def exact(case, seed):
    c, dt, kind = case, case["dtype"], case["kind"]
    d = _inputs(c, seed)
    if kind == "linear":
        x = d["x"].double()
        ys = [_act(_matmul(x, w), c["act"]) for w in d["w"]]
        return [y + d["r"].double() if c["add"] else y for y in ys]
    if kind == "mlp":
        x, hs, ys = d["x"].double(), [], []
        for w in d["w"]:
            g = _rnd(_act(_matmul(x, w["gate"]), "silu"), dt)
            hs.append(_rnd(g * _rnd(_matmul(x, w["up"]), dt), dt))
            ys.append(_matmul(hs[-1], w["down"]))
        return hs + ys
    if kind == "layer":
        x, v, outs = d["x"].double(), d["v"].double(), []
        for w in d["w"]:
            n1 = _rnd(_norm(x, w["ln"].double() + 1.0), dt)
            o = [_rnd(_matmul(n1, w[k]), dt) for k in ("qkv", "z", "a", "b")]
            gated = _rnd((_norm(v.view(-1, 128), w["gn"].double())
                          * _act(o[1].view(-1, 128), "silu")).view(v.shape), dt)
            mid = _rnd(_rnd(_matmul(gated, w["out"]), dt) + x, dt)
            n2 = _rnd(_norm(mid, w["post"].double() + 1.0), dt)
            g = _rnd(_act(_matmul(n2, w["gate"]), "silu"), dt)
            up = _rnd(g * _rnd(_matmul(n2, w["up"]), dt), dt)
            x = _rnd(_rnd(_matmul(up, w["down"]), dt) + mid, dt)
            outs.append(o + [mid, x])
        return outs
    q, s = d["w"]
    if kind == "lm_head":
        return [_matmul(d["x"].double(), d["w"]), None]
    ids = d["ids"]
    return [(q[ids].double() * s[ids][:, :, None].double()).reshape(len(ids), -1)]
