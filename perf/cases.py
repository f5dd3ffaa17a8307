"""Performance cases of the quantized-matmul backend, each one pass through the
package's public entry points.

Six kinds of work, by what a program on this library spends its time on:
  mv      one decode matvec (``mv``): the smallest call there is;
  layer   the matrix products of one transformer layer for `tokens` tokens: a
          decode step's launches (``mv_multi``, ``mv``, ``mv_add``) for one
          token, with lm_head where `V` is set, or a chunk's GEMMs
          (``batch_mv_ws``) for several;
  moe     one whole MoE layer (``moe_layer``), decode, a few tokens, prefill;
  codec   packing: quantize a matrix, and read it back dequantised;
  engine  a prompt and then single tokens through a four-layer model.
Sizes are those of the Qwen3.5-9B (Q8_0), Qwen3.8-27B (Q4_0) and
Qwen3.6-35B-A3B (Q4_0) configurations in ``qwen3x_amd/workloads.py`` and the
tests; ``draw`` spreads them over the ranges that these stand for.
"""
import math

import numpy as np
import torch

import qwen3x_amd as q3x

Q8, Q4 = q3x.MATRIX_Q8_0, q3x.MATRIX_Q4_0
DEVICE = "cuda"
EPS = 1e-6
THETA = 10000000.0

# The layer widths of the models: H, I, rows of the query and key/value
# projections, input width of the output projection.
LAYER_9B = dict(type=Q8, H=4096, I=12288, Q=8192, KV=1024, O=4096)
LAYER_27B = dict(type=Q4, H=5120, I=17408, Q=12288, KV=1024, O=6144)
MOE_35B = dict(type=Q4, experts=256, top_k=8, H=2048, I=512, shared_I=512)
ENGINE_9B = dict(type=Q8, H=4096, I=12288, AH=16, KVH=4, KH=16, VH=32)
ENGINE_27B = dict(type=Q4, H=5120, I=17408, AH=24, KVH=4, KH=16, VH=48)

MOST_PRODUCTS = 7e11  # multiplications of a drawn case: fewer than the largest listed one has


def listed():
    return [
        # One 4096 x 4096 matrix for one token: a launch and its latency.
        dict(name="mv_q8_4096", kind="mv", type=Q8, rows=4096, cols=4096),
        # A decode step's matvec set of a 9B-class layer with lm_head.
        dict(name="decode_9b_q8", kind="layer", tokens=1, V=151936, **dict(LAYER_9B, Q=4096, KV=4096)),
        # A decode step's matrices of a 27B attention layer.
        dict(name="decode_27b_q4", kind="layer", tokens=1, V=0, **LAYER_27B),
        # A very short prompt, or a few drafted tokens to verify.
        dict(name="layer_9b_q8_7tok", kind="layer", tokens=7, V=0, **LAYER_9B),
        # A chat turn of a sentence or two: an odd number of tokens.
        dict(name="layer_27b_q4_77tok", kind="layer", tokens=77, V=0, **LAYER_27B),
        # A page of prompt.
        dict(name="layer_27b_q4_512tok", kind="layer", tokens=512, V=0, **LAYER_27B),
        # A full prefill chunk of a long prompt.
        dict(name="layer_9b_q8_4096tok", kind="layer", tokens=4096, V=0, **LAYER_9B),
        # A MoE layer in decode, over a short turn, and over a long prompt.
        dict(name="moe_35b_1tok", kind="moe", tokens=1, **MOE_35B),
        dict(name="moe_35b_19tok", kind="moe", tokens=19, **MOE_35B),
        dict(name="moe_35b_2048tok", kind="moe", tokens=2048, **MOE_35B),
        # Packing one BF16 feed-forward matrix to Q4_0 and reading it back.
        dict(name="codec_q4_17408x5120", kind="codec", type=Q4, source="bf16", rows=17408, cols=5120),
        # A prompt of some hundred tokens, then eight generated tokens.
        dict(name="engine_9b_500_8", kind="engine", prompt=500, decode=8, **ENGINE_9B),
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _width(rng, low, high):
    """A row length: mostly a multiple of 256, as models have, else of 32."""
    step = 32 if rng.random() < 0.25 else 256
    return max(step, _log(rng, low, high) // step * step)


def draw(rng):
    kind = rng.choice(["mv", "layer1", "layer", "layer", "moe", "moe", "codec", "engine"])
    type_ = rng.choice([Q8, Q4])
    if kind == "mv":
        return dict(kind="mv", type=type_, rows=_log(rng, 64, 160000), cols=_width(rng, 256, 8192))
    if kind in ("layer1", "layer"):
        H = _width(rng, 1024, 6144)
        I = _width(rng, 2 * H, 4 * H)
        Q, KV, O = _log(rng, H // 2, 2 * H), _log(rng, 128, H), _width(rng, H // 2, 2 * H)
        most = int(MOST_PRODUCTS / (H * (Q + 2 * KV + O) + 3 * H * I))
        tokens = 1 if kind == "layer1" else _log(rng, 2, min(4096, most))
        return dict(kind="layer", type=type_, tokens=tokens, H=H, I=I, Q=Q, KV=KV, O=O,
                    V=_log(rng, 1000, 160000) if tokens == 1 and rng.random() < 0.5 else 0)
    if kind == "moe":
        experts = rng.choice([8, 32, 60, 128, 256])
        I = 32 * _log(rng, 4, 32)
        H = 256 * rng.randint(4, 12)
        return dict(kind="moe", type=type_, experts=experts, top_k=rng.randint(1, 8), H=H, I=I,
                    shared_I=I if rng.random() < 0.6 else max(32, I // 64 * 32),
                    tokens=1 if rng.random() < 0.25 else _log(rng, 2, 2500))
    if kind == "codec":
        return dict(kind="codec", type=type_, source=rng.choice(["bf16", "f32"]), rows=_log(rng, 1, 20000),
                    cols=_width(rng, 256, 8192))
    model = rng.choice([ENGINE_9B, ENGINE_27B])
    most = int(MOST_PRODUCTS / _engine_matrices(model))
    return dict(kind="engine", prompt=_log(rng, 2, min(1200, most)), decode=rng.randint(1, 12), **model)


# ---------------------------------------------------------------- inputs

def _generator(seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(int(seed))
    return g


def _pack(type_, w):
    """Blocks (uint8 [n, 34 or 18]) of FP32 values w [n, 32], as the packer
    quantizes them: Q8_0 d = max|w| / 127, Q4_0 d = (value of largest
    magnitude) / -8."""
    if type_ == Q8:
        d = w.abs().amax(1, keepdim=True) / 127.0
        inv = torch.where(d != 0, 1.0 / d, torch.zeros_like(d))
        v = w * inv
        q = torch.copysign(torch.floor(v.abs() + 0.5), v).clamp_(-127, 127).to(torch.int8).view(torch.uint8)
    else:
        d = w.gather(1, w.abs().argmax(1, keepdim=True)) / -8.0
        inv = torch.where(d != 0, 1.0 / d, torch.zeros_like(d))
        n = torch.trunc(w * inv + 8.5).clamp_(0, 15).to(torch.uint8)
        q = n[:, :16] | (n[:, 16:] << 4)
    return torch.cat([d.to(torch.float16).view(torch.uint8), q], 1)


def _matrix(g, type_, rows, cols, std):
    """Bytes of a quantized matrix of N(0, std) weights."""
    out = torch.empty((rows * cols // 32, 34 if type_ == Q8 else 18), dtype=torch.uint8, device=DEVICE)
    step = 1 << 21
    for b in range(0, out.shape[0], step):
        n = min(step, out.shape[0] - b)
        out[b:b + n] = _pack(type_, torch.randn((n, 32), generator=g, device=DEVICE).mul_(std))
    return out.view(-1)


def _linear(g, type_, rows, cols, std=0.02):
    return q3x.Linear(_matrix(g, type_, rows, cols, std), rows, cols, type_)


def _bf16(g, shape, std):
    """BF16 bits (int16) of N(0, std) values."""
    return torch.randn(shape, generator=g, device=DEVICE).mul_(std).to(torch.bfloat16).view(torch.int16)


def _randn(g, *shape):
    return torch.randn(shape, generator=g, device=DEVICE)


def _empty(*shape):
    return torch.empty(shape, device=DEVICE)


def _engine_fields(c):
    return dict(V=1024, N=4, AI=4, AD=256, RD=64, KD=128, VD=128, CK=4, experts=0, top_k=0, shared_I=0,
                tied_embeddings=0, id=11, matrix_type=c["type"], H=c["H"], I=c["I"], AH=c["AH"], KVH=c["KVH"],
                KH=c["KH"], VH=c["VH"])


def prepare(case, seed):
    c, g = case, _generator(seed)
    s = dict(case=case)
    if c["kind"] == "mv":
        s.update(w=_linear(g, c["type"], c["rows"], c["cols"]), x=_randn(g, c["cols"]), y=_empty(c["rows"]))
    elif c["kind"] == "layer":
        t, H, I, T = c["type"], c["H"], c["I"], c["tokens"]
        s["q"], s["k"], s["v"] = (_linear(g, t, rows, H) for rows in (c["Q"], c["KV"], c["KV"]))
        s["o"] = _linear(g, t, H, c["O"])
        s["gate"], s["up"] = _linear(g, t, I, H), _linear(g, t, I, H)
        s["down"] = _linear(g, t, H, I)
        if c["V"]:
            s["lm_head"] = _linear(g, t, c["V"], H)
            s["logits"] = _empty(c["V"])
        s.update(x=_randn(g, T, H), a=_randn(g, T, c["O"]), h=_randn(g, T, I))
        s["outs"] = [_empty(T, rows) for rows in (c["Q"], c["KV"], c["KV"], I, I)]
        s["y"] = _empty(T, H)
        if T > 1:  # one workspace for the layer's GEMMs, which run in order
            need = max(q3x.gemm_workspace_bytes(s[m], T) for m in ("q", "k", "v", "o", "gate", "up", "down"))
            s["ws"] = torch.empty(need, dtype=torch.uint8, device=DEVICE) if need else None
    elif c["kind"] == "moe":
        t, E, H, I, SI, T = c["type"], c["experts"], c["H"], c["I"], c["shared_I"], c["tokens"]
        top_k = min(c["top_k"], E)
        layer = q3x.MoeLayer(_bf16(g, (E, H), H ** -0.5), _matrix(g, t, E * 2 * I, H, 0.02),
                             _matrix(g, t, E * H, I, 0.02), _matrix(g, t, SI, H, 0.02), _matrix(g, t, SI, H, 0.02),
                             _matrix(g, t, H, SI, 0.02), _bf16(g, (1, H), 0.02), t, E, top_k, H, I, SI)
        s.update(layer=layer, X=_randn(g, T, H), Y=_empty(T, H), weights=_empty(T, top_k),
                 ids=torch.empty((T, top_k), dtype=torch.int32, device=DEVICE),
                 ws=torch.empty(q3x.moe_layer_workspace_bytes(layer, T), dtype=torch.uint8, device=DEVICE))
    elif c["kind"] == "codec":
        rows, cols = c["rows"], c["cols"]
        src = _randn(g, rows, cols).mul_(0.02)
        s["src"] = src.to(torch.bfloat16) if c["source"] == "bf16" else src
        s["blocks"] = torch.empty(rows * cols // 32 * (34 if c["type"] == Q8 else 18), dtype=torch.uint8,
                                  device=DEVICE)
        s["out"] = _empty(rows, cols)
    else:
        fields = _engine_fields(c)
        config = q3x.make_config(**fields)
        table, nbytes = q3x.model_schema(config)
        image = torch.zeros(nbytes, dtype=torch.uint8, device=DEVICE)
        H = c["H"]
        for t in table:
            role = q3x.TENSOR_ROLES[t.role]
            n = t.rows * t.cols
            if t.type in (Q8, Q4):
                data = _matrix(g, t.type, t.rows, t.cols, 1.0 if role == "embedding" else t.cols ** -0.5)
            elif t.type == q3x.TENSOR_F32:
                data = _randn(g, n).mul_(0.2).add_(-1.0 if role == "delta_alog" else 1.0).view(torch.uint8)
            else:
                data = _bf16(g, (n,), 0.5 if role in ("delta_conv", "delta_dt") else 0.1).view(torch.uint8)
            image[t.offset:t.offset + t.bytes] = data
        torch.cuda.synchronize()
        count = c["prompt"] + c["decode"]
        tokens = np.random.default_rng(int(seed)).integers(0, fields["V"], count).astype(np.int32)
        s.update(image=image, table=table, tokens=tokens, engine=q3x.Engine(config, image, count))
    return s


def run(state):
    s, c = state, state["case"]
    if c["kind"] == "mv":
        return q3x.mv(s["w"], s["x"], s["y"])
    if c["kind"] == "layer":
        T, outs, y = c["tokens"], s["outs"], s["y"]
        if T == 1:
            q3x.mv_multi([s["q"], s["k"], s["v"]], s["x"], outs[:3])
            q3x.mv(s["o"], s["a"], y)
            q3x.mv_multi([s["gate"], s["up"]], s["x"], outs[3:])
            q3x.mv_add(s["down"], s["h"], y)
            if c["V"]:
                q3x.mv(s["lm_head"], s["x"], s["logits"])
                return outs + [y, s["logits"]]
            return outs + [y]
        for name, out in zip(("q", "k", "v"), outs):
            q3x.batch_mv_ws(s[name], s["x"], out, T, s["ws"])
        q3x.batch_mv_ws(s["o"], s["a"], y, T, s["ws"])
        for name, out in zip(("gate", "up"), outs[3:]):
            q3x.batch_mv_ws(s[name], s["x"], out, T, s["ws"])
        q3x.batch_mv_ws(s["down"], s["h"], y, T, s["ws"], add=True)
        return outs + [y]
    if c["kind"] == "moe":
        q3x.moe_layer(s["layer"], s["X"], c["tokens"], s["Y"], s["ids"], s["weights"], s["ws"])
        return [s["Y"], s["ids"], s["weights"]]
    if c["kind"] == "codec":
        pack = q3x.quantize_bf16 if c["source"] == "bf16" else q3x.quantize
        pack(c["type"], s["src"], c["rows"], c["cols"], s["blocks"])
        q3x.dequant(q3x.Linear(s["blocks"], c["rows"], c["cols"], c["type"]), 0, c["rows"], s["out"])
        return [s["blocks"], s["out"]]
    e, tokens, prompt = s["engine"], s["tokens"], c["prompt"]
    e.reset()
    e.forward(tokens[:prompt])
    logits = [e.logits()]
    for t in range(prompt, len(tokens)):
        e.forward(tokens[t:t + 1])
        logits.append(e.logits())
    return np.stack(logits)


# ------------------------------------------------------------ work, tolerance

def _bytes(type_, n):
    return n // 32 * (34 if type_ == Q8 else 18)


def _engine_matrices(c):
    """Weights of the four layers and lm_head of an engine case's model."""
    DO, DK, AS, KVW = c["VH"] * 128, c["KH"] * 128, c["AH"] * 256, c["KVH"] * 256
    H = c["H"]
    delta = H * (2 * DK + 2 * DO + 2 * c["VH"]) + DO * H
    attention = H * (2 * AS + 2 * KVW) + AS * H
    return 3 * delta + attention + 4 * 3 * H * c["I"] + 1024 * H


def work(case):
    c = case
    if c["kind"] == "mv":
        n = c["rows"] * c["cols"]
        return dict(bytes=_bytes(c["type"], n) + 4 * (c["rows"] + c["cols"]), flops=2 * n)
    if c["kind"] == "layer":
        H, I, T = c["H"], c["I"], c["tokens"]
        n = H * (c["Q"] + 2 * c["KV"] + c["O"] + c["V"]) + 3 * H * I
        values = T * (H + c["O"] + I + c["Q"] + 2 * c["KV"] + 2 * I + H) + c["V"]
        return dict(bytes=_bytes(c["type"], n) + 4 * values, flops=2 * T * n)
    if c["kind"] == "moe":
        E, H, I, SI, T = c["experts"], c["H"], c["I"], c["shared_I"], c["tokens"]
        k = min(c["top_k"], E)
        used = E * (1.0 - (1.0 - k / E) ** T)  # experts that T tokens select, on average
        return dict(bytes=_bytes(c["type"], 3 * H * I) * used + _bytes(c["type"], 3 * H * SI) + 2 * (E + 1) * H +
                    8 * T * (H + k), flops=2 * T * (3 * H * (I * k + SI) + (E + 1) * H))
    if c["kind"] == "codec":
        n = c["rows"] * c["cols"]
        return dict(bytes=n * (2 if c["source"] == "bf16" else 4) + 2 * _bytes(c["type"], n) + 4 * n, flops=0)
    n = _engine_matrices(c)
    return dict(bytes=_bytes(c["type"], n) * (1 + c["decode"]) + 4 * 1024 * (1 + c["decode"]),
                flops=2 * (n * (c["prompt"] + c["decode"])))


def tolerance(case):
    # About four times what the path differs from exact() by (1e-7 to 3.5e-7
    # of the result for single products, 4e-7 for a MoE layer, 5e-7 through
    # four layers of a model): FP32 sums, whatever their order.
    if case["kind"] == "codec":
        return "exact"
    if case["kind"] == "moe":
        return dict(rel=2e-6, differ=1e-3)  # ids may differ where two probabilities tie
    if case["kind"] == "engine":
        return dict(rel=3e-6)
    return dict(rel=1.5e-6)


# ------------------------------------------------------------------ exact

def _values(type_, data, rows, cols):
    """float64 [rows, cols] of a quantized matrix's bytes."""
    b = data.view(-1, 34 if type_ == Q8 else 18)
    d = b[:, :2].contiguous().view(torch.float16).double()
    if type_ == Q8:
        q = b[:, 2:].contiguous().view(torch.int8).double()
    else:
        n = b[:, 2:]
        q = torch.cat([n & 15, n >> 4], 1).double() - 8.0
    return (q * d).view(rows, cols)


def _bits64(t):
    """float64 of BF16 bits."""
    return t.view(torch.bfloat16).double()


def _apply(m, x):
    return x.double() @ _values(m.type, m.weight, m.rows, m.columns).T


def _silu(x):
    return x * torch.sigmoid(x)


def exact(case, seed):
    c = case
    s = prepare(case, seed)
    if c["kind"] == "mv":
        return _apply(s["w"], s["x"])
    if c["kind"] == "layer":
        outs = [_apply(s[m], s["x"]) for m in ("q", "k", "v", "gate", "up")]
        outs.append(_apply(s["o"], s["a"]) + _apply(s["down"], s["h"]))
        return outs + ([_apply(s["lm_head"], s["x"])[0]] if c["V"] else [])
    if c["kind"] == "moe":
        return _exact_moe(s["layer"], s["X"].double())
    if c["kind"] == "codec":
        blocks = _pack(c["type"], s["src"].float().view(-1, 32)).view(-1)
        return [None, _values(c["type"], blocks, c["rows"], c["cols"])]
    return _exact_engine(c, s)


def _exact_moe(m, X):
    p = torch.softmax(X @ _bits64(m.router).T, 1)
    top, ids = p.topk(m.top_k, 1)
    weights = top / top.sum(1, keepdim=True)
    Y = torch.zeros_like(X)
    gu = m.gate_up.view(m.experts, -1)
    dn = m.down.view(m.experts, -1)
    for e in range(m.experts):
        token, slot = (ids == e).nonzero(as_tuple=True)
        if token.numel():
            v = X[token] @ _values(m.type, gu[e], 2 * m.I, m.H).T
            v = (_silu(v[:, :m.I]) * v[:, m.I:]) @ _values(m.type, dn[e], m.H, m.I).T
            Y.index_add_(0, token, weights[token, slot, None] * v)
    v = _silu(X @ _values(m.type, m.shared_gate, m.shared_I, m.H).T) * (
        X @ _values(m.type, m.shared_up, m.shared_I, m.H).T)
    Y += torch.sigmoid(X @ _bits64(m.shared_scale).T) * (v @ _values(m.type, m.shared_down, m.H, m.shared_I).T)
    return [Y, None, weights]


def _exact_engine(c, s):
    tensors = {(q3x.TENSOR_ROLES[t.role], t.layer): t for t in s["table"]}

    def get(role, layer=-1):
        t = tensors[role, layer]
        data = s["image"][t.offset:t.offset + t.bytes]
        if t.type in (Q8, Q4):
            return _values(t.type, data, t.rows, t.cols)
        return data.view(torch.float32).double() if t.type == q3x.TENSOR_F32 else _bits64(data.view(torch.int16))

    def norm(x, w):
        return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w

    KH, VH, AH, KVH, KD, AD, RD = c["KH"], c["VH"], c["AH"], c["KVH"], 128, 256, 64
    tokens = torch.from_numpy(s["tokens"].astype(np.int64)).to(DEVICE)
    T = tokens.numel()
    x = get("embedding")[tokens]
    for i in range(4):
        n = norm(x, 1.0 + get("input_norm", i))
        if i % 4 != 3:
            qkv = n @ get("delta_qkv", i).T
            w = get("delta_conv", i).view(-1, 4)
            padded = torch.cat([torch.zeros_like(qkv[:3]), qkv])
            qkv = _silu(sum(padded[j:j + T] * w[:, j] for j in range(4)))
            q, k, v = qkv.split([KH * KD, KH * KD, VH * KD], 1)
            q, k, v = q.view(T, KH, KD), k.view(T, KH, KD), v.view(T, VH, KD)
            q = q * torch.rsqrt(q.square().sum(-1, keepdim=True) + EPS) / KD ** 0.5
            k = k * torch.rsqrt(k.square().sum(-1, keepdim=True) + EPS)
            q, k = (t.repeat_interleave(VH // KH, 1) for t in (q, k))
            beta = torch.sigmoid(n @ get("delta_b", i).T)
            decay = torch.exp(-torch.exp(get("delta_alog", i)) *
                              torch.nn.functional.softplus(n @ get("delta_a", i).T + get("delta_dt", i)))
            S = torch.zeros((VH, KD, KD), dtype=torch.float64, device=DEVICE)
            o = torch.empty((T, VH, KD), dtype=torch.float64, device=DEVICE)
            for t in range(T):
                S = S * decay[t, :, None, None]
                delta = beta[t, :, None] * (v[t] - (S * k[t, :, :, None]).sum(1))
                S = S + k[t, :, :, None] * delta[:, None, :]
                o[t] = (S * q[t, :, :, None]).sum(1)
            z = (n @ get("delta_z", i).T).view(T, VH, KD)
            mixed = (norm(o, get("delta_norm", i)) * _silu(z)).view(T, -1) @ get("delta_out", i).T
        else:
            qg = (n @ get("attn_q", i).T).view(T, AH, 2, AD)
            q = norm(qg[:, :, 0], 1.0 + get("attn_qnorm", i))
            k = norm((n @ get("attn_k", i).T).view(T, KVH, AD), 1.0 + get("attn_knorm", i))
            v = (n @ get("attn_v", i).T).view(T, KVH, AD)
            # The model's rotation angles are 32-bit values.
            base = torch.tensor([THETA ** (2.0 * j / RD) for j in range(RD // 2)], dtype=torch.float32, device=DEVICE)
            angle = (torch.arange(T, dtype=torch.float32, device=DEVICE)[:, None, None] / base).double()
            cos, sin = angle.cos(), angle.sin()
            q, k = (torch.cat([t[..., :RD // 2] * cos - t[..., RD // 2:RD] * sin,
                               t[..., RD // 2:RD] * cos + t[..., :RD // 2] * sin, t[..., RD:]], -1) for t in (q, k))
            mask = torch.ones((T, T), dtype=torch.bool, device=DEVICE).tril()
            heads = []
            for h in range(AH):
                kv = h // (AH // KVH)
                score = (q[:, h] @ k[:, kv].T / AD ** 0.5).masked_fill(~mask, -math.inf)
                heads.append(torch.softmax(score, 1) @ v[:, kv])
            mixed = (torch.stack(heads, 1) * torch.sigmoid(qg[:, :, 1])).reshape(T, -1) @ get("attn_out", i).T
        x = x + mixed
        n = norm(x, 1.0 + get("post_norm", i))
        x = x + (_silu(n @ get("ffn_gate", i).T) * (n @ get("ffn_up", i).T)) @ get("ffn_down", i).T
    last = x[c["prompt"] - 1:]
    return (norm(last, 1.0 + get("final_norm")) @ get("lm_head").T).cpu().numpy()
