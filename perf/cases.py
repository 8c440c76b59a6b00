"""Performance cases of the engine: what a serving process asks of it, through the public entry points.

A case is one call (or the calls of one request) on a model of a few layers with the real widths of the supported
workloads, either as a pipeline stage (activations in, activations out) or as a whole model (token ids in, logits out):

  part      "stage": a middle pipeline stage; "model": embedding, layers, head
  call      "prefill": a new request's prompt (its session is opened for it); "step": one decode / verify / batched step
  shape     a row of SHAPES; "small" is a generic 64-wide-head model
  type      the linear layers' tensor type
  layers    layers of the stage or model
  sessions  sequences of the step (1 for a prefill)
  rows      prompt tokens of a prefill, token rows per session of a step
  position  cached positions before a step (0 for a prefill)
"""
from __future__ import annotations

import dataclasses
import functools
import math
import zlib

import numpy as np
import torch

import jetsonfabric_amd as jf
from jetsonfabric_amd.configs import CONFIGS

JFM = {"q4_k": jf.Q4_K, "q6_k": jf.Q6_K, "q8_0": jf.Q8_0, "q2_k": jf.Q2_K, "f32": jf.F32}
BITS = {"q4_k": 4.5, "q6_k": 6.5625, "q8_0": 8.5, "q2_k": 2.625}

# (widths, embedding type, head type)
SHAPES = {
    "1.5b": (CONFIGS["qwen2.5-1.5b-q4k"].model, "q8_0", "q8_0"),
    "7b": (CONFIGS["qwen2.5-7b-q4k"].model, "q4_k", "q6_k"),
    "14b": (CONFIGS["qwen2.5-14b-q4k"].model, "q4_k", "q4_k"),
    "32b": (CONFIGS["qwen2.5-32b-q2k"].model, "q2_k", "q6_k"),
    "small": (jf.ModelConfig(n_layer=2, n_embd=512, n_ff=1536, n_head=8, n_head_kv=2, n_vocab=8192, n_ctx=8192),
              "q4_k", "q6_k"),
}


def _case(name, part, call, shape, type_, layers, sessions, rows, position):
    return {"name": name, "part": part, "call": call, "shape": shape, "type": type_, "layers": layers,
            "sessions": sessions, "rows": rows, "position": position}


def listed():
    return [
        # one request's next token on one stage of a small model: launches and latency
        _case("decode-1.5b", "stage", "step", "1.5b", "q4_k", 4, 1, 1, 256),
        # continuous batching at concurrency 2, the benchmark's step
        _case("decode-7b-x2", "stage", "step", "7b", "q4_k", 4, 2, 1, 1100),
        # whole decode call with logits (sampling on the host), tied Q8_0 head
        _case("logits-1.5b", "model", "step", "1.5b", "q4_k", 2, 1, 1, 333),
        # prompt-lookup draft of 4 verified in one pass
        _case("verify-7b", "stage", "step", "7b", "q4_k", 4, 1, 5, 1024),
        # two requests with drafts of 8 at a long context
        _case("verify-14b-x2", "stage", "step", "14b", "q4_k", 2, 2, 9, 4096),
        # eight requests on the 2-bit model
        _case("decode-32b-x8", "stage", "step", "32b", "q2_k", 2, 8, 1, 2176),
        # a short chat prompt: one ragged chunk
        _case("prompt-7b-100", "stage", "prefill", "7b", "q4_k", 4, 1, 100, 0),
        # prompts on the 8-bit and 6-bit formats, odd lengths
        _case("prompt-1.5b-q8-333", "stage", "prefill", "1.5b", "q8_0", 4, 1, 333, 0),
        _case("prompt-7b-q6-777", "stage", "prefill", "7b", "q6_k", 2, 1, 777, 0),
        # the benchmark's prompt, whole call with logits
        _case("prompt-7b-1024", "model", "prefill", "7b", "q4_k", 2, 1, 1024, 0),
        # a long document: attention grows to thousands of keys
        _case("prompt-14b-4096", "model", "prefill", "14b", "q4_k", 2, 1, 4096, 0),
        # the 2-bit model's prompt
        _case("prompt-32b-q2-2048", "model", "prefill", "32b", "q2_k", 2, 1, 2048, 0),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    most = max(work(c)["flops"] for c in listed())
    while True:
        shape = rng.choice(["1.5b", "1.5b", "7b", "7b", "14b", "32b", "small"])
        type_ = rng.choice(["q4_k", "q4_k", "q4_k", "q6_k", "q8_0", "q2_k"])
        call = rng.choice(["prefill", "step"])
        c = _case("", "stage", call, shape, type_, rng.randint(1, 4), 1, 1, 0)
        del c["name"]
        if call == "prefill":
            c["rows"] = _log(rng, 20, 4096)
            c["part"] = rng.choice(["stage", "model"]) if shape in ("1.5b", "small") and c["layers"] < 3 else "stage"
        else:
            c["sessions"] = rng.choice([1, 1, 2, 3, 5, 8])
            c["rows"] = rng.choice([1, 1, rng.randint(2, 9)])
            c["position"] = _log(rng, 30, 4096)
        if work(c)["flops"] <= most:
            return c


# ---------------------------------------------------------------- weights

def _seed(*parts):
    return zlib.crc32(repr(parts).encode())


def _gen(*parts):
    return torch.Generator(device="cuda").manual_seed(_seed(*parts))


def _f16(x):
    return x.to(torch.float16)


def _bytes16(x):
    """f16 [...] -> uint8 [..., 2] (little endian)"""
    return x.contiguous().view(torch.uint8).reshape(*x.shape, 2)


def _min_max(w, sub, levels, top):
    """Affine sub-blocks of `sub` values: codes, 'top'-level scales and mins, f16 super-block factors."""
    b = w.reshape(-1, 256 // sub, sub)
    lo = b.amin(-1).clamp(max=0.0)
    scale = (b.amax(-1) - lo) / levels
    d, dmin = _f16(scale.amax(-1) / top), _f16((-lo).amax(-1) / top)
    df, mf = d.float().clamp(min=1e-12).unsqueeze(-1), dmin.float().clamp(min=1e-12).unsqueeze(-1)
    sc, mn = (scale / df).round().clamp(0, top), (-lo / mf).round().clamp(0, top)
    s, m = (d.float().unsqueeze(-1) * sc).unsqueeze(-1), (dmin.float().unsqueeze(-1) * mn).unsqueeze(-1)
    q = ((b + m) / s.clamp(min=1e-12)).round().clamp(0, levels)
    value = d.double()[:, None, None] * sc.double().unsqueeze(-1) * q.double() - \
        dmin.double()[:, None, None] * mn.double().unsqueeze(-1)
    return q.to(torch.uint8), sc.to(torch.uint8), mn.to(torch.uint8), d, dmin, value.reshape(w.shape)


def _encode(type_, w):
    """w f32 [n, cols] -> (GGML blocks uint8 [n, row bytes], the values they stand for, f64 [n, cols])"""
    n = w.shape[0]
    if type_ == "q8_0":
        b = w.reshape(-1, 32)
        d = _f16(b.abs().amax(-1) / 127.0)
        q = (b / d.float().clamp(min=1e-12).unsqueeze(-1)).round().clamp(-127, 127)
        return (torch.cat([_bytes16(d), q.to(torch.int8).view(torch.uint8)], -1).reshape(n, -1),
                (d.double().unsqueeze(-1) * q.double()).reshape(w.shape))
    if type_ == "q4_k":
        q, sc, mn, d, dmin, value = _min_max(w, 32, 15, 63)
        packed = torch.empty(q.shape[0], 12, dtype=torch.uint8, device=w.device)
        packed[:, 0:4] = sc[:, :4] | (sc[:, 4:] >> 4) << 6
        packed[:, 4:8] = mn[:, :4] | (mn[:, 4:] >> 4) << 6
        packed[:, 8:12] = (sc[:, 4:] & 15) | (mn[:, 4:] & 15) << 4
        qs = (q[:, 0::2] | q[:, 1::2] << 4).reshape(-1, 128)
        return torch.cat([_bytes16(d), _bytes16(dmin), packed, qs], -1).reshape(n, -1), value
    if type_ == "q2_k":
        q, sc, mn, d, dmin, value = _min_max(w, 16, 3, 15)
        f = q.reshape(-1, 2, 4, 32)  # half, shift, value
        qs = f[:, :, 0] | f[:, :, 1] << 2 | f[:, :, 2] << 4 | f[:, :, 3] << 6
        return torch.cat([sc | mn << 4, qs.reshape(-1, 64), _bytes16(d), _bytes16(dmin)], -1).reshape(n, -1), value
    if type_ == "q6_k":
        b = w.reshape(-1, 16, 16)
        scale = b.abs().amax(-1) / 31.0
        d = _f16(scale.amax(-1) / 127.0)
        sc = (scale / d.float().clamp(min=1e-12).unsqueeze(-1)).round().clamp(1, 127)
        q = (b / (d.float()[:, None] * sc).clamp(min=1e-12).unsqueeze(-1)).round().clamp(-32, 31)
        value = (d.double()[:, None, None] * sc.double().unsqueeze(-1) * q.double()).reshape(w.shape)
        f = (q + 32).to(torch.uint8).reshape(-1, 2, 4, 32)  # half, quarter, value
        ql = torch.stack([f[:, :, 0] & 15 | (f[:, :, 2] & 15) << 4, f[:, :, 1] & 15 | (f[:, :, 3] & 15) << 4], 2)
        qh = f[:, :, 0] >> 4 | (f[:, :, 1] >> 4) << 2 | (f[:, :, 2] >> 4) << 4 | (f[:, :, 3] >> 4) << 6
        return (torch.cat([ql.reshape(-1, 128), qh.reshape(-1, 64), sc.to(torch.uint8), _bytes16(d)], -1).reshape(n, -1),
                value)
    raise ValueError(type_)


def _matrix(type_, rows, cols, *key):
    """Blocks (uint8 [rows, row bytes]) and f64 values, in pieces of rows."""
    g = _gen("matrix", type_, rows, cols, *key)
    step = max(1, (64 << 20) // cols)
    for r in range(0, rows, step):
        yield _encode(type_, torch.randn(min(step, rows - r), cols, generator=g, device="cuda") * 0.02)


def _vector(n, mean, std, *key):
    return mean + std * torch.randn(n, generator=_gen("vector", n, *key), device="cuda")


def _config(case):
    """The model the engine is built on: a middle stage has a layer before and one after it."""
    m = SHAPES[case["shape"]][0]
    if case["part"] == "stage":
        return dataclasses.replace(m, n_layer=case["layers"] + 2, n_vocab=256)
    return dataclasses.replace(m, n_layer=case["layers"])


def _layer_matrices(m):
    h, kv, f = m.n_embd, m.n_head_kv * m.head_dim, m.n_ff
    return {"attn_q": (h, h), "attn_k": (kv, h), "attn_v": (kv, h), "attn_output": (h, h), "ffn_gate": (f, h),
            "ffn_up": (f, h), "ffn_down": (h, f)}


def _layer_vectors(m):
    h, kv = m.n_embd, m.n_head_kv * m.head_dim
    return {"attn_norm.weight": (h, 1.0, 0.1), "ffn_norm.weight": (h, 1.0, 0.1), "attn_q.bias": (h, 0.0, 0.2),
            "attn_k.bias": (kv, 0.0, 0.2), "attn_v.bias": (kv, 0.0, 0.2)}


@functools.lru_cache(maxsize=1)
def _engine(part, shape, type_, layers):
    """The engine a serving process keeps for its model (the weights are the same for every request)."""
    m = _config({"part": part, "shape": shape, "layers": layers})
    _, embd, head = SHAPES[shape]

    def blocks(t, rows, cols, *key):
        return b"".join(b.cpu().numpy().tobytes() for b, _ in _matrix(t, rows, cols, *key))

    def tensors():
        yield "token_embd.weight", JFM[embd], (m.n_embd, m.n_vocab), blocks(embd, m.n_vocab, m.n_embd, "embd")
        yield "output.weight", JFM[head], (m.n_embd, m.n_vocab), blocks(head, m.n_vocab, m.n_embd, "head")
        yield "output_norm.weight", JFM["f32"], (m.n_embd,), _vector(m.n_embd, 1.0, 0.1, "norm").cpu().numpy().tobytes()
        # the layers around a middle stage are not part of its engine: they repeat its first layer
        first = 1 if part == "stage" else 0
        for name, (rows, cols) in _layer_matrices(m).items():
            for k in range(layers):
                data = blocks(type_, rows, cols, name, k)
                for l in [first + k] + ([0, layers + 1] if part == "stage" and k == 0 else []):
                    yield f"blk.{l}.{name}.weight", JFM[type_], (cols, rows), data
        for name, (n, mean, std) in _layer_vectors(m).items():
            for l in range(m.n_layer):
                v = _vector(n, mean, std, name, max(0, l - first))
                yield f"blk.{l}.{name}", JFM["f32"], (n,), v.cpu().numpy().tobytes()

    model = jf.Model.build(m, tensors())
    if part == "stage":
        whole, model = model, model.slice(1, 1 + layers)
        whole.close()
    engine = jf.NativeEngine(model)
    model.close()
    torch.cuda.empty_cache()
    return engine


# ---------------------------------------------------------------- a request

def _inputs(case, seed):
    """Per session: token ids or activation rows, and the cached keys and values [layer][kv head][position][dim]."""
    m = _config(case)
    g = _gen("inputs", seed)
    out = []
    for _ in range(case["sessions"]):
        if case["part"] == "model":
            x = torch.randint(0, m.n_vocab, (case["rows"],), generator=g, device="cuda")
        else:  # a residual stream after many layers: several times one layer's update, a few channels much larger
            x = torch.randn(case["rows"], m.n_embd, generator=g, device="cuda") * 8.0
            x[:, torch.randint(0, m.n_embd, (8,), generator=g, device="cuda")] *= 8.0
        kv = None
        if case["position"]:
            size = (2, case["layers"], m.n_head_kv, case["position"], m.head_dim)
            kv = (torch.randn(size, generator=g, device="cuda") * 1.2).to(torch.float16)
        out.append((x, kv))
    return out


def prepare(case, seed):
    engine = _engine(case["part"], case["shape"], case["type"], case["layers"])
    state = {"case": case, "engine": engine, "sessions": [], "inputs": []}
    for x, kv in _inputs(case, seed):
        if kv is not None:
            s = engine.create_session(case["position"] + case["rows"] + 64)
            k, v = kv.cpu().numpy().view(np.uint16)
            s.import_kv(k, v)
            state["sessions"].append(s)
        state["inputs"].append(x.cpu().tolist() if case["part"] == "model" else x.cpu().numpy())
    return state


def run(state):
    case, engine, xs = state["case"], state["engine"], state["inputs"]
    model, n = case["part"] == "model", case["rows"]
    if case["call"] == "prefill":
        s = engine.create_session(n + 64)
        out = s.prefill_greedy(xs[0], logits=True)[1] if model else s.prefill_stage(activations=xs[0])
        s.close()
        return [out]
    sessions = state["sessions"]
    if len(sessions) == 1 and n == 1:
        out = [sessions[0].decode_greedy(xs[0][0], logits=True)[1] if model
               else sessions[0].decode_stage(activation=xs[0])]
    elif model:
        out = engine.step_batch(sessions, xs, logits=True)[2]
    else:
        out = engine.stage_step_batch(sessions, activations=xs)
    for s in sessions:  # the next pass takes the same step
        s.rollback(n)
    return out


def work(case):
    m = _config(case)
    rows = case["sessions"] * case["rows"]
    weights = sum(r * c for r, c in _layer_matrices(m).values())
    byte = case["layers"] * weights * BITS[case["type"]] / 8
    flop = case["layers"] * 2.0 * weights * rows
    kv = m.n_head_kv * m.head_dim * 2 * 2  # bytes of a position's keys and values
    seen = case["sessions"] * sum(case["position"] + i + 1 for i in range(case["rows"]))  # (row, key) pairs
    byte += case["layers"] * case["sessions"] * (case["position"] + case["rows"]) * kv
    flop += case["layers"] * 4.0 * m.n_embd * seen
    if case["part"] == "stage":
        byte += 2 * rows * m.n_embd * 4
    else:
        outs = 1 if case["call"] == "prefill" else rows
        byte += m.n_vocab * m.n_embd * BITS[SHAPES[case["shape"]][2]] / 8 + outs * m.n_vocab * 4
        flop += 2.0 * m.n_vocab * m.n_embd * outs
    return {"bytes": byte, "flops": flop}


def tolerance(case):
    # Every linear layer rounds its inputs to 8-bit codes, and sums in another order move a few codes by one. Measured
    # with inputs changed by 2e-7 of themselves and prompts cut into other chunks: up to 0.004 of the output per stage
    # layer (0.012 over four, largest value 0.06), 0.011 over two layers of a whole model, whose residual is small.
    if case["part"] == "model":
        return {"rel": 0.03, "max": 0.2}
    return {"rel": min(0.03, 0.012 * case["layers"]), "max": 0.2}


# ---------------------------------------------------------------- in 64 bits

def _apply(x, type_, rows, cols, *key):
    return torch.cat([x @ v.T for _, v in _matrix(type_, rows, cols, *key)], -1)


def _norm(x, gain, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * gain


def _rope(x, pos, base):
    """x [rows, heads, dim]: value i pairs with value i + dim / 2"""
    half = x.shape[-1] // 2
    f = base ** (-torch.arange(half, dtype=torch.float64, device=x.device) / half)
    a = (pos.double()[:, None] * f)[:, None, :]
    lo, hi = x[..., :half], x[..., half:]
    return torch.cat([lo * a.cos() - hi * a.sin(), lo * a.sin() + hi * a.cos()], -1)


def exact(case, seed):
    m, type_ = _config(case), case["type"]
    _, embd, head = SHAPES[case["shape"]]
    hd, group = m.head_dim, m.n_head // m.n_head_kv
    inputs = _inputs(case, seed)
    n, p0 = case["rows"], case["position"]
    if case["part"] == "model":
        ids = torch.cat([x for x, _ in inputs])
        h, at = torch.empty(len(ids), m.n_embd, dtype=torch.float64, device="cuda"), 0
        for _, v in _matrix(embd, m.n_vocab, m.n_embd, "embd"):
            here = (ids >= at) & (ids < at + len(v))
            h[here] = v[ids[here] - at]
            at += len(v)
    else:
        h = torch.cat([x for x, _ in inputs]).double()
    pos = torch.arange(p0, p0 + n, device="cuda").repeat(len(inputs))
    sizes = _layer_matrices(m)
    for k in range(case["layers"]):
        vec = {name: _vector(*size, name, k).double() for name, size in _layer_vectors(m).items()}

        def linear(name, x):
            return _apply(x, type_, *sizes[name], name, k)

        x = _norm(h, vec["attn_norm.weight"], m.rms_eps)
        q = _rope((linear("attn_q", x) + vec["attn_q.bias"]).reshape(-1, m.n_head, hd), pos, m.rope_base)
        key = _rope((linear("attn_k", x) + vec["attn_k.bias"]).reshape(-1, m.n_head_kv, hd), pos, m.rope_base)
        val = (linear("attn_v", x) + vec["attn_v.bias"]).reshape(-1, m.n_head_kv, hd)
        att = torch.empty_like(q)
        for i, (_, kv) in enumerate(inputs):
            r = slice(i * n, (i + 1) * n)
            for a in range(m.n_head):
                kk, vv = key[r, a // group], val[r, a // group]
                if kv is not None:
                    kk = torch.cat([kv[0, k, a // group].double(), kk])
                    vv = torch.cat([kv[1, k, a // group].double(), vv])
                s = q[r, a] @ kk.T / math.sqrt(hd)
                s.masked_fill_(torch.arange(len(kk), device="cuda") > pos[r][:, None], -math.inf)
                att[r, a] = torch.softmax(s, -1) @ vv
        h = h + linear("attn_output", att.reshape(len(h), -1))
        x = _norm(h, vec["ffn_norm.weight"], m.rms_eps)
        h = h + linear("ffn_down", torch.nn.functional.silu(linear("ffn_gate", x)) * linear("ffn_up", x))
    if case["part"] == "model":
        if case["call"] == "prefill":
            h = h[-1:]
        h = _apply(_norm(h, _vector(m.n_embd, 1.0, 0.1, "norm").double(), m.rms_eps), head, m.n_vocab, m.n_embd, "head")
        if case["call"] == "prefill" or len(h) == 1:
            return [h[0].cpu().numpy()]
    h = h.cpu().numpy()
    if case["call"] == "prefill":
        return [h]
    return [h[i * n:(i + 1) * n] for i in range(len(inputs))]
