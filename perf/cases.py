"""What a program that serves quantized models has this framework do, as cases that can be timed.

Each case is one step of such a program through `metaltile_amd.ops`, on weights that are resident in the packed format:

  delta     one token through a linear-attention layer: its input projections, and its gated norm with the output projection
  decode    1..32 tokens through the projections of some dense layers (attention and MLP)
  prefill   the same projections of one layer for a prompt of 33..4096 tokens
  moe       tokens through an expert layer: router, expert sort, permute, gate / up / down experts, unpermute
  vocab     both ends of a model: a prompt's embedding rows, and the final norm with the output head for the last token
  convert   a weight matrix quantized into the packed format, and read back

What lies between these calls in a model (attention, activation functions, residuals) is not the framework's, so the inputs
of each call are at hand when a step begins. Weights, scales and activations have the distributions of
`metaltile_amd.synth`: uniform codes, scale = 0.02 |N(0,1)| + 1e-3, bias = -2^(bits-1) scale + 1e-3 N(0,1), x ~ N(0,1).
"""
import math

import torch

from metaltile_amd import DType, ops

DTYPES = {"bf16": (DType.BF16, torch.bfloat16), "f16": (DType.F16, torch.float16), "f32": (DType.F32, torch.float32)}


def listed():
    return [
        # One stream through a small linear-attention layer: two short calls, nothing but latency.
        dict(name="delta_1_token", kind="delta", dtype="bf16", bits=4, group=64, hidden=2048, hv=16, dv=128),
        # One stream through eight layers of an 8B model, norms fused into the projections that follow them. The weights (1 GB a
        # pass) come from memory, as in a decode loop.
        dict(name="decode_1_token", kind="decode", dtype="bf16", bits=4, group=64, rows=1, layers=8, hidden=4096, inter=14336, q=4096, kv=1024),
        # A few streams at once, 8-bit weights, row lengths that are no power of two; separate projections.
        dict(name="decode_4_tokens_8_bit", kind="decode", dtype="f16", bits=8, group=64, rows=4, layers=2, hidden=3584, inter=18944, q=3584, kv=512),
        # A full decode batch on a 13B model's layers.
        dict(name="decode_16_tokens", kind="decode", dtype="bf16", bits=4, group=128, rows=16, layers=3, hidden=5120, inter=13824, q=5120, kv=5120),
        # A short prompt of an odd length on 6-bit weights.
        dict(name="prefill_77_tokens_6_bit", kind="prefill", dtype="f16", bits=6, group=64, rows=77, layers=1, hidden=3584, inter=18944, q=3584, kv=512),
        # The usual prefill chunk.
        dict(name="prefill_512_tokens", kind="prefill", dtype="bf16", bits=4, group=64, rows=512, layers=1, hidden=4096, inter=14336, q=4096, kv=1024),
        # A long prompt.
        dict(name="prefill_4096_tokens", kind="prefill", dtype="bf16", bits=4, group=64, rows=4096, layers=1, hidden=4096, inter=14336, q=4096, kv=1024),
        # One stream through a layer of many small experts.
        dict(name="moe_1_token", kind="moe", dtype="bf16", bits=4, group=64, tokens=1, hidden=2048, inter=768, experts=128, top=8),
        # A decode batch through a layer of few large experts.
        dict(name="moe_16_tokens", kind="moe", dtype="bf16", bits=4, group=64, tokens=16, hidden=4096, inter=14336, experts=8, top=2),
        # A prompt through a layer of many small experts.
        dict(name="moe_2048_tokens", kind="moe", dtype="bf16", bits=4, group=64, tokens=2048, hidden=2048, inter=768, experts=128, top=8),
        # A prompt's embedding rows, and the output head.
        dict(name="vocab_512_tokens", kind="vocab", dtype="bf16", bits=4, group=64, tokens=512, hidden=4096, vocab=128256),
        # A checkpoint's matrix into the packed format and back.
        dict(name="convert_f32", kind="convert", dtype="f32", bits=4, group=64, rows=14336, cols=4096),
    ]


# The largest listed case's products: a drawn one has no more.
MOST_MACS = 4096 * (4096 * (4096 + 2 * 1024) + 4096 * 4096 + 3 * 4096 * 14336)


def _spread(rng, lo, hi, step=1):
    """A whole multiple of `step` from lo to hi, spread over the logarithm."""
    return min(hi, max(lo, int(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.5))) / step + 0.5) * step))


def _format(rng):
    return dict(dtype=rng.choice(("bf16", "bf16", "f16")), bits=rng.choice((4, 4, 4, 4, 8, 8, 6, 5, 3, 2)), group=rng.choice((64, 64, 128, 32)))


def draw(rng):
    kind = rng.choice(("delta", "decode", "decode", "decode", "prefill", "prefill", "prefill", "moe", "moe", "vocab", "convert"))
    c = dict(kind=kind, **_format(rng))
    if kind == "delta":
        c.update(bits=4, hidden=_spread(rng, 1024, 5120, 128), hv=rng.choice((8, 12, 16, 24, 32, 48)), dv=128)
    elif kind in ("decode", "prefill"):
        hidden = _spread(rng, 1024, 8192, 128)
        inter = min(28672, int(hidden * rng.uniform(2.0, 4.5)) // 128 * 128)
        heads, shared = hidden // 128, rng.choice((1, 2, 4, 8))
        c.update(hidden=hidden, inter=inter, q=heads * 128, kv=max(1, heads // shared) * 128)
        codes = _codes(c)
        if kind == "decode":
            rows = rng.choice((1, 1, _spread(rng, 2, 32), _spread(rng, 2, 32)))
            c.update(rows=rows, layers=max(1, min(8, (1 << 31) // codes, rng.randint(1, 8))))
        else:
            c.update(rows=min(_spread(rng, 33, 4096), MOST_MACS // codes), layers=1)
    elif kind == "moe":
        experts = rng.choice((8, 16, 32, 60, 64, 128))
        hidden = _spread(rng, 1024, 4096, 128)
        inter = _spread(rng, 512, min(14336, (7 << 28) // (4 * experts * hidden) // 128 * 128), 128)
        top = rng.choice((1, 2, 4, 6, 8))
        c.update(bits=rng.choice((4, 4, 4, 8)), hidden=hidden, inter=inter, experts=experts, top=top)
        c.update(tokens=min(rng.choice((1, _spread(rng, 2, 64), _spread(rng, 64, 4096))), MOST_MACS // (3 * top * hidden * inter)))
    elif kind == "vocab":
        c.update(bits=rng.choice((4, 4, 8, 6)), tokens=_spread(rng, 1, 4096), hidden=_spread(rng, 1024, 8192, 128), vocab=_spread(rng, 32000, 152064))
    else:
        c.update(dtype=rng.choice(("bf16", "f16", "f32")), rows=_spread(rng, 256, 14336), cols=_spread(rng, 1024, 8192, 128))
    return c


def _codes(c):
    """Weights of one dense layer."""
    return c["hidden"] * (c["q"] + 2 * c["kv"]) + c["q"] * c["hidden"] + 3 * c["hidden"] * c["inter"]


def _fused(c):
    """Whether a decode step has its norms inside the projections: only one row can."""
    return c["rows"] == 1


class Maker:
    """Inputs on the GPU from a seed."""

    def __init__(self, case, seed):
        self.gen = torch.Generator("cuda").manual_seed(seed)
        self.dtype, self.t = DTYPES[case["dtype"]]
        self.bits, self.group = case.get("bits"), case.get("group")
        self.keep = []  # what the addresses in the state point at

    def held(self, t):
        self.keep.append(t)
        return t

    def values(self, *shape, dtype=None):
        return self.held(torch.randn(shape, generator=self.gen, device="cuda", dtype=torch.float32).to(dtype or self.t))

    def norm_weight(self, n):
        return self.held((1.0 + 0.1 * torch.randn(n, generator=self.gen, device="cuda")).to(self.t))

    def matrix(self, n, k):
        """(weights, scales, biases) addresses of an [n, k] matrix in the packed format."""
        w = self.held(torch.randint(-(1 << 31), 1 << 31, (n * (k * self.bits // 32),), generator=self.gen, device="cuda", dtype=torch.int32))
        s = 0.02 * torch.randn(n * (k // self.group), generator=self.gen, device="cuda").abs_() + 1e-3
        b = s * -float(1 << (self.bits - 1)) + 1e-3 * torch.randn(s.numel(), generator=self.gen, device="cuda")
        return w.data_ptr(), self.held(s.to(self.t)).data_ptr(), self.held(b.to(self.t)).data_ptr()

    def out(self, *shape, dtype=None):
        return self.held(torch.zeros(shape, device="cuda", dtype=dtype or self.t))

    def scalar(self, v):
        return self.held(torch.full((1,), v, device="cuda", dtype=torch.float32)).data_ptr()


def prepare(case, seed):
    m = Maker(case, seed)
    s = dict(case=case, make=m, dtype=m.dtype, fmt=(m.dtype, m.bits, m.group), eps=m.scalar(1e-5))
    s.update({"delta": _delta, "decode": _dense, "prefill": _dense, "moe": _moe, "vocab": _vocab, "convert": _convert}[case["kind"]](case, m))
    return s


def _delta(c, m):
    inner, n = c["hv"] * c["dv"], (2 * c["hv"] * c["dv"], c["hv"] * c["dv"], c["hv"], c["hv"])
    outs = [m.out(k) for k in n]
    result = m.out(c["hidden"])
    mats = [m.matrix(k, c["hidden"]) for k in n]
    return dict(n=n, ws=[w for w, _, _ in mats], ss=[s for _, s, _ in mats], bs=[b for _, _, b in mats], x=m.values(c["hidden"]).data_ptr(),
                y=m.values(c["hv"], c["dv"], dtype=torch.float32).data_ptr(), z=m.values(inner).data_ptr(), norm=m.norm_weight(c["dv"]).data_ptr(),
                o=m.matrix(c["hidden"], inner), outs=[t.data_ptr() for t in outs], out=result.data_ptr(), result=outs + [result])


def _dense(c, m):
    rows, hidden, inter, q, kv = (c[k] for k in ("rows", "hidden", "inter", "q", "kv"))
    layers, result = [], []

    def out(n):
        t = m.out(rows, n)
        result.append(t)
        return t.data_ptr()

    for _ in range(c["layers"]):
        at = dict(x=m.values(rows, hidden).data_ptr(), attn=m.values(rows, q).data_ptr(), h=m.values(rows, hidden).data_ptr(), act=m.values(rows, inter).data_ptr(),
                  o=m.matrix(hidden, q), down=m.matrix(hidden, inter), o_out=out(hidden), down_out=out(hidden))
        if _fused(c):
            at.update(norm1=m.norm_weight(hidden).data_ptr(), norm2=m.norm_weight(hidden).data_ptr(), qkv=m.matrix(q + 2 * kv, hidden), qkv_out=out(q + 2 * kv),
                      gate_up=m.matrix(2 * inter, hidden), gate_up_out=out(2 * inter))
        else:
            for name, ns in (("qkv", (q, kv, kv)), ("gate_up", (inter, inter))):
                mats = [m.matrix(n, hidden) for n in ns]
                at[name] = ([w for w, _, _ in mats], [s for _, s, _ in mats], [b for _, _, b in mats])
                at[name + "_outs"] = [out(n) for n in ns]
        layers.append(at)
    return dict(layers=layers, result=result)


def _moe(c, m):
    tokens, hidden, inter, experts, top = (c[k] for k in ("tokens", "hidden", "inter", "experts", "top"))
    rows = tokens * top
    whole = dict(dtype=torch.int32)
    t = dict(ids=m.out(tokens, top, **whole), weights=m.out(tokens, top), rows_in=m.out(rows, hidden), gate_out=m.out(rows, inter), up_out=m.out(rows, inter),
             out=m.out(tokens, hidden))
    if not _one_token(c):
        t.update(order=m.out(rows, **whole), inverse=m.out(tokens, top, **whole), offsets=m.out(experts + 1, **whole), down_out=m.out(rows, hidden))
    s = {k: v.data_ptr() for k, v in t.items()}
    s.update(logits=m.values(tokens, experts).data_ptr(), x=m.values(tokens, hidden).data_ptr(), act=m.values(rows, inter).data_ptr(),
             first=m.out(top, **whole).data_ptr(), gate=m.matrix(experts * inter, hidden), up=m.matrix(experts * inter, hidden),
             down=m.matrix(experts * hidden, inter), result=t)
    if _one_token(c):
        size = t["gate_out"].element_size() * inter
        s.update(gates=[s["gate_out"] + j * size for j in range(top)], ups=[s["up_out"] + j * size for j in range(top)])
    return s


def _one_token(c):
    """Whether the step is one token's whose down projection can have the activation and the weighted sum inside it."""
    return c["tokens"] == 1 and c["top"] <= 8 and c["bits"] == 4 and c["inter"] <= 4096


def _vocab(c, m):
    rows, logits = m.out(c["tokens"], c["hidden"]), m.out(c["vocab"])
    ids = m.held(torch.randint(0, c["vocab"], (c["tokens"],), generator=m.gen, device="cuda", dtype=torch.int32))
    return dict(table=m.matrix(c["vocab"], c["hidden"]), ids=ids.data_ptr(), rows=rows.data_ptr(), x=m.values(c["hidden"]).data_ptr(),
                norm=m.norm_weight(c["hidden"]).data_ptr(), logits=logits.data_ptr(), result=[rows, logits])


def _convert(c, m):
    n = c["rows"] * c["cols"]
    w = m.held((0.05 * torch.randn(n, generator=m.gen, device="cuda")).to(m.t))
    t = [m.out(n * m.bits // 32, dtype=torch.int32), m.out(n // m.group), m.out(n // m.group), m.out(n)]
    return dict(n=n, w=w.data_ptr(), to=[x.data_ptr() for x in t], result=t)


def run(state):
    c, fmt = state["case"], state["fmt"]
    kind = c["kind"]
    if kind == "delta":
        ops.qmv_batched(*fmt, state["ws"], state["ss"], state["bs"], state["x"], state["outs"], state["n"], c["hidden"])
        ops.gated_rms_norm_qmv(state["dtype"], c["group"], state["y"], state["z"], state["norm"], state["eps"], *state["o"], state["out"], c["hv"], c["dv"], c["hidden"])
    elif kind in ("decode", "prefill"):
        rows, hidden, inter, q, kv = c["rows"], c["hidden"], c["inter"], c["q"], c["kv"]
        for at in state["layers"]:
            if _fused(c):
                ops.rms_norm_qmv(*fmt, at["x"], at["norm1"], *at["qkv"], at["qkv_out"], state["eps"], q + 2 * kv, hidden)
                ops.qmv(*fmt, *at["o"], at["attn"], at["o_out"], 1, hidden, q)
                ops.rms_norm_qmv(*fmt, at["h"], at["norm2"], *at["gate_up"], at["gate_up_out"], state["eps"], 2 * inter, hidden)
                ops.qmv(*fmt, *at["down"], at["act"], at["down_out"], 1, hidden, inter)
            else:
                ops.qmm_batched(*fmt, *at["qkv"], at["x"], at["qkv_outs"], (q, kv, kv), rows, hidden)
                ops.qmm(*fmt, *at["o"], at["attn"], at["o_out"], rows, hidden, q)
                ops.qmm_batched(*fmt, *at["gate_up"], at["h"], at["gate_up_outs"], (inter, inter), rows, hidden)
                ops.qmm(*fmt, *at["down"], at["act"], at["down_out"], rows, hidden, inter)
    elif kind == "moe":
        d, tokens, hidden, inter, experts, top = state["dtype"], c["tokens"], c["hidden"], c["inter"], c["experts"], c["top"]
        rows = tokens * top
        ops.moe_router_topk(d, state["logits"], state["ids"], state["weights"], tokens, experts, top)
        if _one_token(c):
            ops.moe_permute(d, state["x"], state["first"], state["rows_in"], 1, top, hidden)
            ops.gather_qmv_indices(*fmt, state["rows_in"], *state["gate"], state["ids"], state["gate_out"], top, inter, hidden, experts)
            ops.gather_qmv_indices(*fmt, state["rows_in"], *state["up"], state["ids"], state["up_out"], top, inter, hidden, experts)
            ops.moe_down_swiglu_accum(d, c["group"], state["gates"], state["ups"], state["ids"], state["weights"], *state["down"], state["out"], inter, hidden, experts)
        else:
            ops.moe_sort_by_expert(state["ids"], tokens, top, experts, state["order"], state["inverse"], state["offsets"])
            ops.moe_permute(d, state["x"], state["order"], state["rows_in"], tokens, rows, hidden)
            ops.gather_qmv_csr(*fmt, state["rows_in"], *state["gate"], state["offsets"], state["gate_out"], rows, inter, hidden, experts)
            ops.gather_qmv_csr(*fmt, state["rows_in"], *state["up"], state["offsets"], state["up_out"], rows, inter, hidden, experts)
            ops.gather_qmv_csr(*fmt, state["act"], *state["down"], state["offsets"], state["down_out"], rows, hidden, inter, experts)
            ops.moe_unpermute(d, state["down_out"], state["inverse"], state["weights"], state["out"], tokens, rows, hidden, top)
    elif kind == "vocab":
        ops.dequant_gather(*fmt, *state["table"], state["ids"], state["rows"], c["tokens"], c["hidden"], c["vocab"])
        ops.rms_norm_qmv(*fmt, state["x"], state["norm"], *state["table"], state["logits"], state["eps"], c["vocab"], c["hidden"])
    else:
        words, scales, biases, back = state["to"]
        ops.affine_quantize(*fmt, state["w"], words, scales, biases, state["n"])
        ops.affine_dequantize(*fmt, words, scales, biases, back, state["n"])
    return state["result"]


def work(case):
    c = case
    size = 4 if c["dtype"] == "f32" else 2
    per_code = c["bits"] / 8 + 2 * size / c["group"]  # a packed weight with its share of scale and bias
    kind = c["kind"]
    if kind == "delta":
        inner = c["hv"] * c["dv"]
        codes = c["hidden"] * (3 * inner + 2 * c["hv"] + inner)
        return dict(bytes=codes * per_code + size * (2 * c["hidden"] + 4 * inner + 2 * c["hv"] + c["dv"]) + 4 * inner, flops=2 * codes)
    if kind in ("decode", "prefill"):
        codes, rows = _codes(c), c["rows"]
        values = 4 * c["hidden"] + 2 * c["q"] + 2 * c["kv"] + 3 * c["inter"]  # inputs and outputs of the four steps, per row
        return dict(bytes=c["layers"] * (codes * per_code + rows * values * size), flops=2.0 * c["layers"] * codes * rows)
    if kind == "moe":
        tokens, hidden, inter, experts, top = (c[k] for k in ("tokens", "hidden", "inter", "experts", "top"))
        rows = tokens * top
        hit = experts * (1 - (1 - min(1, top / experts)) ** tokens)  # experts that some token picks, expected
        codes = 3 * hidden * inter
        values = tokens * (experts + 2 * hidden + top) + rows * (hidden + 2 * inter)
        if not _one_token(c):
            values += rows * (hidden + inter)
        return dict(bytes=hit * codes * per_code + values * size + 4 * rows, flops=2.0 * rows * codes)
    if kind == "vocab":
        codes = c["vocab"] * c["hidden"]
        return dict(bytes=(codes + c["tokens"] * c["hidden"]) * per_code + size * (c["tokens"] * c["hidden"] + 2 * c["hidden"] + c["vocab"]), flops=2.0 * codes)
    n = c["rows"] * c["cols"]
    return dict(bytes=2 * n * size + 2 * n * per_code, flops=8.0 * n)


def tolerance(case):
    """16-bit results: a rounding of the weight, where a product takes them rounded, and one of the result. 32-bit ones: the
    order of sums. Experts, orders and packed codes are whole numbers that do not depend on either."""
    return dict(rel={"bf16": 1e-2, "f16": 2e-3, "f32": 1e-5}[case["dtype"]])


class Exact:
    """The same inputs in plain torch, in 64 bits."""

    def __init__(self, case, make):
        self.bits, self.group = case["bits"], case["group"]
        self.at = {t.data_ptr(): t for t in make.keep}

    def value(self, address, *shape):
        return self.at[address].double().reshape(shape or (-1,))

    def rows(self, matrix, k, lo, hi):
        """Rows lo..hi of a matrix in the packed format, k columns."""
        w, s, b = (self.at[p] for p in matrix)
        words = w.reshape(-1, k * self.bits // 32)[lo:hi].reshape(-1, self.bits).long() & 0xFFFFFFFF
        codes = torch.empty(words.shape[0], 32, dtype=torch.float64, device=w.device)
        for i in range(32):  # 32 codes of any width are a whole number of words
            at, shift = divmod(i * self.bits, 32)
            c = words[:, at] >> shift
            if shift + self.bits > 32:
                c = c | words[:, at + 1] << (32 - shift)
            codes[:, i] = (c & ((1 << self.bits) - 1)).double()
        s, b = (t.reshape(-1, k // self.group)[lo:hi].double().reshape(-1, 1) for t in (s, b))
        return (codes.reshape(-1, self.group) * s + b).reshape(hi - lo, k)

    def product(self, matrix, x, n, first=0):
        """x [m, k] times the transpose of the matrix's n rows from `first` on."""
        step = max(1, (1 << 24) // x.shape[1])
        return torch.cat([x @ self.rows(matrix, x.shape[1], first + lo, first + min(n, lo + step)).T for lo in range(0, n, step)], 1)

    def rms_norm(self, x, weight):
        return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + float(torch.tensor(1e-5, dtype=torch.float32))) * weight


def exact(case, seed):
    """What `run` returns for these inputs in 64 bits; None where it returns whole numbers."""
    c, s = case, prepare(case, seed)
    e = Exact(c, s["make"])
    kind = c["kind"]
    if kind == "delta":
        x = e.value(s["x"], 1, -1)
        z = e.value(s["z"], c["hv"], -1)
        inner = e.rms_norm(e.value(s["y"], c["hv"], -1), e.value(s["norm"])) * z * torch.sigmoid(z)
        return [e.product(m, x, n)[0] for m, n in zip(zip(s["ws"], s["ss"], s["bs"]), s["n"])] + [e.product(s["o"], inner.reshape(1, -1), c["hidden"])[0]]
    if kind in ("decode", "prefill"):
        q, kv, hidden, inter, got = c["q"], c["kv"], c["hidden"], c["inter"], []
        for at in s["layers"]:
            x, h, attn, act = (e.value(at[name], c["rows"], -1) for name in ("x", "h", "attn", "act"))
            got += [e.product(at["o"], attn, hidden), e.product(at["down"], act, hidden)]
            if _fused(c):
                got += [e.product(at["qkv"], e.rms_norm(x, e.value(at["norm1"])), q + 2 * kv), e.product(at["gate_up"], e.rms_norm(h, e.value(at["norm2"])), 2 * inter)]
            else:
                got += [e.product(m, x, n) for m, n in zip(zip(*at["qkv"]), (q, kv, kv))] + [e.product(m, h, inter) for m in zip(*at["gate_up"])]
        return got
    if kind == "moe":
        tokens, hidden, inter, experts, top = (c[k] for k in ("tokens", "hidden", "inter", "experts", "top"))
        logits = e.value(s["logits"], tokens, experts)
        ids = torch.sort(logits, dim=1, descending=True, stable=True)[1][:, :top]  # of equal ones the first
        weights = torch.softmax(logits.gather(1, ids), 1)
        order = torch.sort(ids.reshape(-1), stable=True)[1] if not _one_token(c) else torch.arange(top, device=ids.device)
        chosen = ids.reshape(-1)[order].tolist()
        rows_in, act = e.value(s["x"], tokens, hidden)[order // top], e.value(s["act"], tokens * top, inter)
        got = dict(ids=None, weights=weights, rows_in=rows_in)

        def through(matrix, x, n):
            out = torch.empty(x.shape[0], n, dtype=x.dtype, device=x.device)
            for expert in sorted(set(chosen)):
                at = torch.tensor([p for p, i in enumerate(chosen) if i == expert], device=x.device)
                out[at] = e.product(matrix, x[at], n, first=expert * n)
            return out

        got.update(gate_out=through(s["gate"], rows_in, inter), up_out=through(s["up"], rows_in, inter))
        down = through(s["down"], act if not _one_token(c) else got["gate_out"] * torch.sigmoid(got["gate_out"]) * got["up_out"], hidden)
        got["out"] = (down[torch.argsort(order)].reshape(tokens, top, hidden) * weights[:, :, None]).sum(1)
        if not _one_token(c):
            got.update(order=None, inverse=None, offsets=None, down_out=down)
        return got
    if kind == "vocab":
        ids = e.at[s["ids"]].tolist()
        x = e.rms_norm(e.value(s["x"], 1, -1), e.value(s["norm"]))
        return [torch.cat([e.rows(s["table"], c["hidden"], i, i + 1) for i in ids]), e.product(s["table"], x, c["vocab"])[0]]
    v = e.value(s["w"], -1, c["group"])
    low, high, most = v.amin(1, keepdim=True), v.amax(1, keepdim=True), (1 << c["bits"]) - 1
    scale = (high - low) / most
    scale = torch.where(scale < 1e-7, torch.ones_like(scale), scale)
    codes = torch.floor(((v - low) / scale + 0.5).clamp(0, most))
    held = [t.to(DTYPES[c["dtype"]][1]).double() for t in (scale, low)]  # the packed format holds them in the element type
    return [None, scale.reshape(-1), low.reshape(-1), (codes * held[0] + held[1]).reshape(-1)]
