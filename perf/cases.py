"""The work a user of this framework has it do, as cases that can be timed and
compared: the blocks of the 0.8B hybrid (MLP, Gated DeltaNet layer, attention
layer) through the bridge's calls in the order the engine makes them, and
whole conversation turns through the engine.

Blocks run over 1 to a few thousand tokens: one token is a step of the op
sequence (captured and edited steps, engines without the one-launch step),
2-8 a verify pass, tens a short prompt, 128 the default prefill chunk
(`Model.new_run`), thousands a long prompt in one chunk. Formats are the three
the engine loads: fp32, BF16 (the checkpoints' own) and int8 per row.
`prepared` says whether the matrices were prepared (qr_gemm_*_prepare), as
this repository's engine does after an upload; an engine that binds only the
reference's symbols does not.
"""
import math
import sys
from pathlib import Path

import numpy as np
import torch

_PKG = Path(__file__).resolve().parent.parent / "qwen-rust-inference_amd"
if str(_PKG) not in sys.path:
    sys.path.insert(0, str(_PKG))

from qwen_mi355x import engine as E  # noqa: E402
from qwen_mi355x import model as M  # noqa: E402
from qwen_mi355x.bridge import Bridge  # noqa: E402

C = M.config_qwen08b()
H, I = C.hidden_size, C.intermediate_size
KD, VD = C.key_heads * C.key_dim, C.value_heads * C.value_dim
CH = 2 * KD + VD
Q, KV, D = C.num_heads * C.head_dim, C.num_kv_heads * C.head_dim, C.head_dim
EPS = C.rms_norm_eps
STD = 0.02  # the random init of the matrices
F64 = torch.float64
ELEMENT = {"f32": 4.0, "bf16": 2.0, "i8": 1.0}
FORMAT = {"f32": E.F32, "bf16": E.BF16_EXACT, "i8": E.INT8}


def listed():
    return [
        # one token of the op sequence through an MLP: the smallest call, latency and launches
        {"name": "mlp bf16 1", "block": "mlp", "fmt": "bf16", "tokens": 1, "prepared": True},
        # a short prompt of a chat
        {"name": "mlp f32 23", "block": "mlp", "fmt": "f32", "tokens": 23, "prepared": True},
        # the reference engine's prefill chunk on its own symbols, int8 weights
        {"name": "mlp i8 128 plain", "block": "mlp", "fmt": "i8", "tokens": 128, "prepared": False},
        # a long prompt in one chunk
        {"name": "mlp f32 2644", "block": "mlp", "fmt": "f32", "tokens": 2644, "prepared": True},
        # a prompt of a few sentences
        {"name": "delta bf16 77", "block": "delta", "fmt": "bf16", "tokens": 77, "prepared": True},
        # the engine's default prefill chunk
        {"name": "delta f32 128", "block": "delta", "fmt": "f32", "tokens": 128, "prepared": True},
        # a long prompt in one chunk
        {"name": "delta i8 2644", "block": "delta", "fmt": "i8", "tokens": 2644, "prepared": True},
        # one token of the op sequence over a long context
        {"name": "attention f32 1 at 8191", "block": "attention", "fmt": "f32", "tokens": 1, "past": 8191,
         "prepared": True},
        # a middle chunk of a chunked prefill
        {"name": "attention bf16 128 at 1920", "block": "attention", "fmt": "bf16", "tokens": 128, "past": 1920,
         "prepared": True},
        # a long prompt in one chunk
        {"name": "attention f32 2644", "block": "attention", "fmt": "f32", "tokens": 2644, "past": 0,
         "prepared": True},
        # whole turns at the default chunk: a fresh conversation's prompt, then greedy decoding
        {"name": "turn f32 454+32", "block": "turn", "fmt": "f32", "tokens": 454, "new": 32},
        {"name": "turn bf16 37+16", "block": "turn", "fmt": "bf16", "tokens": 37, "new": 16},
    ]


def _spread(rng, lo, hi):
    """A whole number of [lo, hi], even over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    block = rng.choice(["mlp", "mlp", "delta", "delta", "attention", "attention", "turn"])
    fmt = rng.choice(["f32", "bf16", "i8"])
    if block == "turn":
        return {"block": block, "fmt": fmt, "tokens": _spread(rng, 8, 454), "new": _spread(rng, 2, 32)}
    case = {"block": block, "fmt": fmt, "tokens": _spread(rng, 1, 2644), "prepared": rng.random() < 0.75}
    if block == "attention":
        case["past"] = 0 if rng.random() < 0.4 else _spread(rng, 1, 8192 if case["tokens"] <= 256 else 2644)
    return case


# ---------------------------------------------------------------- device data

_BRIDGE = []


def _bridge():
    """The bridge context that a program opens once."""
    if not _BRIDGE:
        _BRIDGE.append(Bridge())
    return _BRIDGE[0]


class _Words:
    """A bridge buffer as an array torch can view (the view keeps it alive)."""

    def __init__(self, buf, shape, kind):
        self.buf = buf
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": kind, "data": (buf.ptr, False),
                                         "strides": None, "version": 3}


def _view(buf, *shape):
    return torch.as_tensor(_Words(buf, shape, "<f4"), device="cuda")


def _alloc(n):
    return _bridge().alloc(int(n))


def _upload(t):
    """A torch tensor of 32-bit words in a bridge buffer of its own."""
    t = t.contiguous()
    buf = _alloc(t.numel())
    words = torch.as_tensor(_Words(buf, (t.numel(),), "<i4"), device="cuda")
    words.copy_(t.view(torch.int32).reshape(-1))
    return buf


class _Draws:
    """Normal values from a seed, in the order they are asked for."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(int(seed))

    def normal(self, *shape, std=1.0):
        return torch.randn(shape, generator=self.g, device="cuda", dtype=torch.float32) * std


def _int8(w):
    """Row-wise symmetric int8 as the engine quantises (fp32 quotients, rounded
    half to even): the scales and the values."""
    scale = (w.abs().amax(dim=1).clamp_min(1e-30).to(F64) / 127.0).to(torch.float32)
    q = torch.empty(w.shape, dtype=torch.int8, device=w.device)
    for r in range(0, w.shape[0], 16384):  # the quotients in 64 bits, then rounded to 32
        part = (w[r:r + 16384].to(F64) / scale[r:r + 16384, None].to(F64)).to(torch.float32)
        q[r:r + 16384] = torch.round(part).clamp(-127, 127).to(torch.int8)
    return scale, q


def _matrix(g, rows, cols, fmt):
    """A random matrix: (its words as the engine uploads them, its values in 64 bits on demand)."""
    w = g.normal(rows, cols, std=STD)
    if fmt == "f32":
        return w, lambda: w.to(F64)
    if fmt == "bf16":
        b = w.to(torch.bfloat16)
        return b.view(torch.int32), lambda: b.to(F64)
    scale, q = _int8(w)
    words = torch.cat([scale.view(torch.int32), q.reshape(-1).view(torch.int32)])
    return words, lambda: scale.to(F64)[:, None] * q.to(F64)


def _names(block):
    if block == "mlp":
        return {"gate": (I, H), "up": (I, H), "down": (H, I)}
    if block == "delta":
        return {"qkv": (CH, H), "z": (VD, H), "a": (C.value_heads, H), "b": (C.value_heads, H), "out": (H, VD)}
    return {"q": (2 * Q, H), "k": (KV, H), "v": (KV, H), "o": (H, Q)}


def _inputs(case, seed):
    """Matrices and vectors of a block and its input, from the seed alone."""
    g, t, block = _Draws(seed), case["tokens"], case["block"]
    mats = {n: _matrix(g, r, c, case["fmt"]) for n, (r, c) in _names(block).items()}
    vec = {"x": g.normal(t, H), "norm": g.normal(H, std=STD)}
    if block == "mlp":
        vec["mixed"] = g.normal(t, H)
    elif block == "delta":
        vec["conv"] = g.normal(CH, C.conv_kernel, std=0.3)
        vec["history"] = g.normal(CH, C.conv_kernel - 1)
        vec["state"] = g.normal(C.value_heads, C.key_dim, C.value_dim, std=0.3)
        vec["gates"] = g.normal(2, C.value_heads, std=0.3)
        vec["delta_norm"] = 1.0 + g.normal(C.value_dim, std=0.1)
    else:
        vec["qk_norm"] = g.normal(2, D, std=0.1)
        vec["keys"] = g.normal(case["past"] + t, KV)
        vec["values"] = g.normal(case["past"] + t, KV)
    return mats, vec


# ---------------------------------------------------------------- whole models

_MODELS = {}


def _weights(fmt, device="cuda"):
    """Random-init weights of the whole model (seed 0, not the case's: one model
    serves every prompt), tensor by tensor: (spec, values on the device)."""
    g = torch.Generator(device=device)
    g.manual_seed(0)
    for s in M.tensor_specs(C):
        if s.kind == "norm_zero":
            yield s, torch.zeros(s.shape, device=device)
        elif s.kind == "norm_direct":
            yield s, torch.ones(s.shape, device=device)
        else:
            w = torch.randn(s.shape, generator=g, device=device) * STD
            yield s, w.to(torch.bfloat16).to(torch.float32) if fmt == "bf16" else w


def _model(fmt):
    """The loaded model that a program keeps for all its conversations."""
    if fmt not in _MODELS:
        w = M.Weights(C, {s.index: np.ascontiguousarray(v.cpu().numpy().reshape(-1)) for s, v in _weights(fmt)})
        _MODELS[fmt] = E.Model(w, fmt=FORMAT[fmt])
    return _MODELS[fmt]


def _prompt(case, seed):
    return np.random.default_rng(seed).integers(0, C.vocab_size, case["tokens"]).astype(np.uint32)


# ---------------------------------------------------------------- prepare

def prepare(case, seed):
    if case["block"] == "turn":
        # the model, a run for conversations of up to 1024 tokens, a prompt
        return {"case": case, "run": _model(case["fmt"]).new_run(1024), "prompt": _prompt(case, seed)}
    b, t, fmt = _bridge(), case["tokens"], case["fmt"]
    mats, vec = _inputs(case, seed)
    s = {"case": case, "bridge": b, "w": {n: _upload(words) for n, (words, _) in mats.items()},
         "v": {n: _upload(v) for n, v in vec.items()}}
    sizes = {"normed": t * H, "y": t * H}
    if case["block"] == "mlp":
        sizes |= {"sum": t * H, "gate_y": t * I, "up_y": t * I, "product": t * I}
    elif case["block"] == "delta":
        sizes |= {"projected": t * CH, "convolved": t * CH, "zs": t * VD, "as": t * C.value_heads,
                  "bs": t * C.value_heads, "query": t * C.value_heads * C.key_dim,
                  "key": t * C.value_heads * C.key_dim, "core": t * VD, "gated": t * VD}
    else:
        sizes |= {"qg": t * 2 * Q, "k": t * KV, "vv": t * KV, "query": t * Q, "gate": t * Q, "context": t * Q,
                  "scores": C.num_heads * max(case["past"] + t, 16 * (D + 2))}
    s["b"] = {n: _alloc(k) for n, k in sizes.items()}
    torch.cuda.synchronize()  # the uploads above, before the bridge's own stream reads them
    if case["prepared"]:
        for n, (rows, cols) in _names(case["block"]).items():
            if rows > 16:
                b.prepare(s["w"][n], rows, cols, fmt)
    b.sync()
    return s


# ---------------------------------------------------------------- run

def run(s):
    case = s["case"]
    return {"mlp": _run_mlp, "delta": _run_delta, "attention": _run_attention, "turn": _run_turn}[case["block"]](s)


def _run_mlp(s):
    """Residual add + norm, silu(x G^T) * (x U^T), down projection."""
    b, w, v, o, fmt, t = s["bridge"], s["w"], s["v"], s["b"], s["case"]["fmt"], s["case"]["tokens"]
    b.run("ADD_RMS_NORM", t, [o["sum"], v["x"], v["mixed"], o["normed"], v["norm"]], [H], [EPS, 1.0])
    b.glu(o["product"], o["gate_y"], o["up_y"], w["gate"], w["up"], o["normed"], I, H, t, kind=fmt)
    b.gemm(o["y"], w["down"], o["product"], H, I, t, kind=fmt)
    return {"sum": _view(o["sum"], t, H), "y": _view(o["y"], t, H)}


def _run_delta(s):
    """Norm, the four input projections, the Gated DeltaNet mixer, the output
    projection; the convolution history and the recurrent state advance."""
    b, w, v, o, fmt, t = s["bridge"], s["w"], s["v"], s["b"], s["case"]["fmt"], s["case"]["tokens"]
    b.run("RMS_NORM", t, [o["normed"], v["x"], v["norm"]], [H], [EPS, 1.0])
    b.group([(o["projected"], w["qkv"], CH), (o["zs"], w["z"], VD), (o["as"], w["a"], C.value_heads),
             (o["bs"], w["b"], C.value_heads)], o["normed"], H, t, kind=fmt)
    b.delta_mixer(convolved=o["convolved"], projected=o["projected"], conv_w=v["conv"], conv_state=v["history"],
                  query=o["query"], key=o["key"], core=o["core"], recurrent=v["state"], a=o["as"], b=o["bs"],
                  gates=v["gates"], gated=o["gated"], norm_w=v["delta_norm"], z=o["zs"], key_heads=C.key_heads,
                  value_heads=C.value_heads, key_dim=C.key_dim, value_dim=C.value_dim, kernel=C.conv_kernel, tokens=t,
                  channels=CH, eps=EPS)
    b.gemm(o["y"], w["out"], o["gated"], H, VD, t, kind=fmt)
    return {"y": _view(o["y"], t, H), "history": _view(v["history"], CH, C.conv_kernel - 1),
            "state": _view(v["state"], C.value_heads, C.key_dim, C.value_dim)}


def _run_attention(s):
    """Norm, q / k / v projections, q and k norms with RoPE and the cache
    append, the gated attention read, the output projection."""
    b, w, v, o, fmt, t = s["bridge"], s["w"], s["v"], s["b"], s["case"]["fmt"], s["case"]["tokens"]
    past = s["case"]["past"]
    b.run("RMS_NORM", t, [o["normed"], v["x"], v["norm"]], [H], [EPS, 1.0])
    b.group([(o["qg"], w["q"], 2 * Q), (o["k"], w["k"], KV), (o["vv"], w["v"], KV)], o["normed"], H, t, kind=fmt)
    b.run("ATTENTION_QUERY_KV", (C.num_heads + C.num_kv_heads) * t,
          [o["query"], o["qg"], v["qk_norm"], o["gate"], v["keys"], o["k"], o["vv"], v["values"]],
          [D, C.rotary_dim, past, C.num_heads, C.num_kv_heads, t], [EPS, C.rope_theta])
    b.run("ATTENTION_READ", C.num_heads, [o["context"], o["query"], v["keys"], v["values"], o["gate"], o["scores"]],
          [D, C.num_heads, C.num_kv_heads, past + 1, past + t, t, o["scores"].n // C.num_heads])
    b.gemm(o["y"], w["o"], o["context"], H, Q, t, kind=fmt)
    return {"y": _view(o["y"], t, H), "keys": _view(v["keys"], past + t, KV), "values": _view(v["values"], past + t, KV)}


def _run_turn(s):
    """A new conversation: its prompt, greedy tokens, and a sampled step's logits."""
    r, new = s["run"], s["case"]["new"]
    r.reset()
    first = r.prefill(s["prompt"])
    ids, _ = r.decode_greedy(int(np.argmax(first)), new)
    last = r.step(ids[-1])
    return {"first": first, "ids": np.array(ids, dtype=np.int64), "last": last}


# ---------------------------------------------------------------- work and tolerance

def _block_bytes(case):
    t, e = case["tokens"], ELEMENT[case["fmt"]]
    shapes = _names(case["block"]).values()
    weights = sum(r * c * e + (4 * r if case["fmt"] == "i8" else 0) for r, c in shapes)
    macs = t * sum(r * c for r, c in shapes)
    if case["block"] == "mlp":
        return weights + 4.0 * t * H * 4, 2.0 * macs
    if case["block"] == "delta":
        state = VD * C.key_dim + CH * (C.conv_kernel - 1)
        rule = 4 * t * VD * C.key_dim  # the recurrence: decay, S^T k, the update, S^T q
        return weights + 4.0 * (2 * t * H + 2 * state), 2.0 * macs + 2.0 * rule
    pairs = t * case["past"] + t * (t + 1) // 2
    cache = (case["past"] + 2 * t) * KV * 2
    return weights + 4.0 * (2 * t * H + cache), 2.0 * macs + 4.0 * pairs * Q


def work(case):
    if case["block"] != "turn":
        b, f = _block_bytes(case)
        return {"bytes": b, "flops": f}
    # the prompt reads every matrix once, each new token once more (lm_head: the tied embedding)
    e, head = ELEMENT[case["fmt"]], C.vocab_size * H
    layers = sum(int(np.prod(s.shape)) for s in M.tensor_specs(C) if s.kind == "matrix") - head
    steps, attn = case["new"], sum(1 for k in C.layer_types if k == "full_attention")
    delta = C.num_layers - attn
    state = delta * (VD * C.key_dim + CH * (C.conv_kernel - 1))
    per = (layers + head) * e + 8.0 * state + 4.0 * C.vocab_size
    cache = 8.0 * attn * KV * (case["tokens"] * (steps + 1) + steps * (steps + 1) // 2)
    n = case["tokens"] + steps
    macs = n * layers + (steps + 1) * head + 4 * n * delta * VD * C.key_dim + attn * Q * n * (n + 1)
    return {"bytes": (1 + steps) * per + cache, "flops": 2.0 * macs}


def tolerance(case):
    # fp32 sums in another order: a block's outputs were up to 1e-6 (2-norm)
    # off 64 bits, and attention's over thousands of positions 2e-6; in a whole
    # model the roundings of 24 layers meet (3.3e-6)
    if case["block"] == "turn":
        return {"rel": 2e-5, "max": 8e-4, "differ": 0.01}
    return {"rel": 1e-5, "max": 4e-4}


# ---------------------------------------------------------------- 64 bits

def _silu(x):
    return x * torch.sigmoid(x)


def _rms(x, w):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * w


def _mlp64(x, w):
    return (_silu(x @ w("gate").T) * (x @ w("up").T)) @ w("down").T


def _delta64(x, w, v, history, state):
    """x [t, H] normalised; returns the output rows, the history and the state."""
    t, heads, dk, dv, k = x.shape[0], C.value_heads, C.key_dim, C.value_dim, C.conv_kernel
    line = torch.cat([history.T, x @ w("qkv").T])  # [k - 1 + t, CH]
    conv = _silu(sum(line[i:i + t] * v["conv"][:, i] for i in range(k)))
    q, key, val = conv[:, :KD].view(t, heads, dk), conv[:, KD:2 * KD].view(t, heads, dk), conv[:, 2 * KD:].view(t, heads, dv)
    q = q * torch.rsqrt((q * q).sum(-1, keepdim=True) + 1e-6) / math.sqrt(dk)
    key = key * torch.rsqrt((key * key).sum(-1, keepdim=True) + 1e-6)
    decay = torch.exp(-torch.exp(v["gates"][1]) * torch.nn.functional.softplus(x @ w("a").T + v["gates"][0]))
    beta = torch.sigmoid(x @ w("b").T)
    state, out = state.clone(), torch.empty(t, heads, dv, dtype=F64, device=x.device)
    for i in range(t):
        state *= decay[i][:, None, None]
        d = (val[i] - (state * key[i][:, :, None]).sum(1)) * beta[i][:, None]
        state += key[i][:, :, None] * d[:, None, :]
        out[i] = (state * q[i][:, :, None]).sum(1)
    z = (x @ w("z").T).view(t, heads, dv)
    gated = _rms(out, v["delta_norm"]) * _silu(z)
    return gated.reshape(t, VD) @ w("out").T, line[t:].T.contiguous(), state


def _rope64(x, past):
    """x [t, heads, D] rotated in its first rotary_dim elements (halves paired).
    The angle itself is an fp32 value, as the model defines it: the position
    over theta^(2 i / rotary_dim), both in fp32."""
    half = C.rotary_dim // 2
    base = (C.rope_theta ** (torch.arange(half, device=x.device, dtype=F64) * 2 / C.rotary_dim)).to(torch.float32)
    at = torch.arange(past, past + x.shape[0], device=x.device)
    angle = (at.to(F64)[:, None] / base.to(F64)).to(torch.float32).to(F64)
    c, s = torch.cos(angle)[:, None], torch.sin(angle)[:, None]
    a, b = x[..., :half], x[..., half:2 * half]
    return torch.cat([a * c - b * s, b * c + a * s, x[..., 2 * half:]], -1)


def _attention64(x, w, v, keys, values, past):
    """x [t, H] normalised; keys / values [past + t, KV], the last t rows set here."""
    t, group = x.shape[0], C.num_heads // C.num_kv_heads
    qg = (x @ w("q").T).view(t, C.num_heads, 2 * D)
    q = _rope64(_rms(qg[..., :D], 1 + v["qk_norm"][0]), past)
    keys[past:] = _rope64(_rms((x @ w("k").T).view(t, C.num_kv_heads, D), 1 + v["qk_norm"][1]), past).reshape(t, KV)
    values[past:] = x @ w("v").T
    seen = torch.arange(past + t, device=x.device)[None] <= torch.arange(past, past + t, device=x.device)[:, None]
    context = torch.empty(t, C.num_heads, D, dtype=F64, device=x.device)
    for h in range(C.num_heads):
        k = slice(h // group * D, (h // group + 1) * D)
        score = (q[:, h] @ keys[:, k].T / math.sqrt(D)).masked_fill(~seen, -math.inf)
        context[:, h] = torch.softmax(score, -1) @ values[:, k]
    return (context * torch.sigmoid(qg[..., D:])).reshape(t, Q) @ w("o").T


def exact(case, seed):
    if case["block"] == "turn":
        return _exact_turn(case, seed)
    mats, vec = _inputs(case, seed)
    v = {n: t.to(F64) for n, t in vec.items()}

    def w(name):
        return mats[name][1]()
    if case["block"] == "mlp":
        total = v["x"] + v["mixed"]
        return {"sum": total, "y": _mlp64(_rms(total, 1 + v["norm"]), w)}
    x = _rms(v["x"], 1 + v["norm"])
    if case["block"] == "delta":
        y, history, state = _delta64(x, w, v, v["history"], v["state"])
        return {"y": y, "history": history, "state": state}
    y = _attention64(x, w, v, v["keys"], v["values"], case["past"])
    return {"y": y, "keys": v["keys"], "values": v["values"]}


def _exact_turn(case, seed):
    fmt, dev = case["fmt"], "cuda"
    tensors = {s.index: v for s, v in _weights(fmt)}
    head32 = tensors[0]

    def matrix(index):
        m = tensors[index]
        if fmt != "i8":
            return m.to(F64)
        scale, q = _int8(m)
        return scale.to(F64)[:, None] * q.to(F64)
    head = matrix(0)
    if fmt == "i8":  # the engine keeps the int8 model's embedding rows in BF16 where they are exact, else in fp32
        embed = head32.to(F64)
    else:
        embed = head
    conv0 = torch.zeros(CH, C.conv_kernel - 1, dtype=F64, device=dev)
    caches = []
    for kind in C.layer_types:
        if kind == "full_attention":
            caches.append([torch.zeros(0, KV, dtype=F64, device=dev)] * 2)
        else:
            caches.append([conv0, torch.zeros(C.value_heads, C.key_dim, C.value_dim, dtype=F64, device=dev)])
    position = 0

    def forward(ids):
        nonlocal position
        x = embed[torch.as_tensor(np.asarray(ids, dtype=np.int64), device=dev)]
        t = x.shape[0]
        for layer, kind in enumerate(C.layer_types):
            base = M.QW_SLOTS_BASE + layer * M.QW_SLOTS_LAYER
            xn = _rms(x, 1 + tensors[base + M.INPUT_NORM].to(F64))
            if kind == "full_attention":
                slot = {"q": M.Q, "k": M.K, "v": M.V, "o": M.O}
                v = {"qk_norm": torch.stack([tensors[base + M.Q_NORM], tensors[base + M.K_NORM]]).to(F64)}
                grown = [torch.cat([c, torch.zeros(t, KV, dtype=F64, device=dev)]) for c in caches[layer]]
                x = x + _attention64(xn, lambda n: matrix(base + slot[n]), v, grown[0], grown[1], position)
                caches[layer] = grown
            else:
                slot = {"qkv": M.QKV, "z": M.Z, "a": M.A, "b": M.B, "out": M.OUT}
                v = {"conv": tensors[base + M.CONV].to(F64), "delta_norm": tensors[base + M.DELTA_NORM].to(F64),
                     "gates": torch.stack([tensors[base + M.DT], tensors[base + M.A_LOG]]).to(F64)}
                y, history, state = _delta64(xn, lambda n: matrix(base + slot[n]), v, *caches[layer])
                x, caches[layer] = x + y, [history, state]
            slot = {"gate": M.GATE, "up": M.UP, "down": M.DOWN}
            x = x + _mlp64(_rms(x, 1 + tensors[base + M.POST_NORM].to(F64)), lambda n: matrix(base + slot[n]))
        position += t
        return head @ _rms(x[-1], 1 + tensors[1].to(F64))

    first = forward(_prompt(case, seed))
    ids = [int(first.argmax())]
    while len(ids) < case["new"]:
        ids.append(int(forward(ids[-1:]).argmax()))
    return {"first": first, "ids": np.array(ids, dtype=np.int64), "last": forward(ids[-1:])}
