"""What a program that runs a local Gemma-like GGUF model has this framework do, as timed cases.

Sizes are those of the model the benchmark and the tests use (hidden 2560, 8 query heads over 2 KV heads, FFN
10240, vocabulary 262144, KV rings of 4096 slots) and of the smaller shapes of the tests.  Kinds of work:

* ``proj``: one projection launch, device pointers (Q/K/V together, O, or down);
* ``ffn``: gate/up + GeGLU, then down;
* ``head``: the output head, top-k candidates and the sampled token of every column;
* ``attention``: head norms, RoPE and the cache append, then GQA attention over the ring;
* ``layers``: a segment of decoder layers for the tokens of one call (a token, a draft, a prompt), with the final
  norm, and with ``head`` the logits too;
* ``runner``: the host-buffer projection call of the engine's runner API (numpy in, numpy out).

Weights: ``file`` are Q4_K / Q6_K blocks quantised from N(0, 1/k) weights as a GGUF quantiser does it (a Q6_K
block's largest sub-block takes scale -128 and the others spread below it); ``synthetic`` are the uniform random
blocks of the benchmark, whose Q6_K scales stay within -32..31 (single projections, FFN and head only).
"""
import ctypes
import math

import numpy as np
import torch

from heliopause_amd import hip_kernels as H
from heliopause_amd.decode import ModelShape

MODEL = {"hidden": 2560, "heads": 8, "kv_heads": 2, "ffn": 10240, "vocab": 262144, "capacity": 4096}
EPSILON = 1e-6
FREQ_BASE = 10000.0
SEED_RNG = 0x48454C49  # the engine's default sampling seed


def _case(kind, **fields):
    c = {"kind": kind, "weights": "file"}
    for name in {"proj": ("hidden", "heads", "kv_heads", "ffn"), "runner": ("hidden", "heads", "kv_heads"),
                 "ffn": ("hidden", "ffn"), "head": ("hidden", "vocab"),
                 "attention": ("heads", "kv_heads", "capacity"),
                 "layers": ("hidden", "heads", "kv_heads", "ffn", "vocab", "capacity")}[kind]:
        c[name] = MODEL[name]
    if kind in ("attention", "layers"):
        c["window"] = 0
    if kind == "attention":
        del c["weights"]
    c.update(fields)
    return c


def listed():
    return [
        # one generated token: its Q/K/V launch, its FFN, its attention over a full ring, the head with its
        # sampled token, and the whole step through all layers to the logits
        _case("proj", name="qkv_token", set="qkv", tokens=1),
        _case("ffn", name="ffn_token", tokens=1),
        _case("attention", name="attention_token", tokens=1, position=5000),
        _case("head", name="head_token", tokens=1, k=64),
        _case("layers", name="decode_step", layers=42, tokens=1, position=4096, head=True),
        # a draft being verified: five tokens through a segment, and the head's candidates for each of them
        _case("layers", name="draft_5", layers=3, tokens=5, position=2000, head=False),
        _case("head", name="head_draft_5", tokens=5, k=40),
        # a chat turn of a sentence or a short paragraph, late in a conversation and at its start
        _case("layers", name="prompt_21", layers=3, tokens=21, position=1500, head=False),
        _case("layers", name="prompt_150", layers=3, tokens=150, position=0, head=False),
        # a full prefill chunk of a long document, and its attention alone
        _case("layers", name="chunk_512", layers=3, tokens=512, position=3584, head=False),
        _case("attention", name="attention_512", tokens=512, position=3584),
        # the engine's runner API from host buffers, a 40-token turn
        _case("runner", name="runner_qkv_40", tokens=40),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["layers"] * 6 + ["proj"] * 3 + ["ffn"] * 2 + ["attention"] * 2 + ["head"] * 2 + ["runner"])
    weights = "synthetic" if rng.random() < 0.2 else "file"
    hidden = rng.choice([1024, 2048, 2560, 2560, 3840])
    heads, kv_heads = rng.choice([(8, 2), (8, 2), (8, 4), (4, 1), (8, 1)])
    ffn = rng.choice([2 * hidden, 10240])
    tokens = _log(rng, 1, 512)
    capacity = rng.choice([4096, 4096, 1024, _log(rng, 512, 4608)])
    window = rng.choice([0, 0, 512])
    position = rng.choice([0, rng.randrange(0, capacity), rng.randrange(0, 2 * capacity)])
    if kind == "proj":
        return _case(kind, weights=weights, hidden=hidden, heads=heads, kv_heads=kv_heads, ffn=ffn, tokens=tokens,
                     set=rng.choice(["qkv", "o", "down"]))
    if kind == "runner":
        return _case(kind, weights=weights, hidden=hidden, heads=heads, kv_heads=kv_heads,
                     tokens=min(tokens, 200))
    if kind == "ffn":
        return _case(kind, weights=weights, hidden=hidden, ffn=ffn, tokens=tokens)
    if kind == "head":
        return _case(kind, weights=weights, hidden=hidden, vocab=_log(rng, 16000, 170000), tokens=_log(rng, 1, 8),
                     k=rng.choice([1, 40, 64]))
    if kind == "attention":
        return _case(kind, heads=heads, kv_heads=kv_heads, capacity=capacity, window=window, tokens=tokens,
                     position=position)
    return _case(kind, layers=rng.choice([1, 2, 3]), hidden=hidden, heads=heads, kv_heads=kv_heads,
                 ffn=ffn, capacity=capacity, window=window, tokens=tokens, position=position, head=False)


# ---- inputs ------------------------------------------------------------------------------------------------

def _generator(seed, label):
    g = torch.Generator(device="cuda:0")
    g.manual_seed((int(seed) * 1000003 + sum((i + 1) * ord(ch) for i, ch in enumerate(label))) & 0x7FFFFFFFFFFF)
    return g


def _normal(g, *shape):
    return torch.randn(*shape, device="cuda:0", generator=g)


def _half_bytes(x):
    return x.half().contiguous().view(torch.uint8).view(*x.shape, 2)


def _q4_k(g, rows, k, synthetic):
    """Q4_K blocks [rows * k/256][144]."""
    n = rows * (k // 256)
    out = torch.empty(n, 144, dtype=torch.uint8, device="cuda:0")
    if synthetic:
        d = _normal(g, n).abs() * 0.01
        dmin = _normal(g, n).abs() * 0.01
        sc = torch.randint(0, 64, (n, 8), device="cuda:0", generator=g)
        mn = torch.randint(0, 64, (n, 8), device="cuda:0", generator=g)
        out[:, 16:] = torch.randint(0, 256, (n, 128), dtype=torch.uint8, device="cuda:0", generator=g)
    else:
        w = _normal(g, n, 8, 32) / math.sqrt(k)
        low = w.amin(2).clamp(max=0)
        scale, low = (w.amax(2) - low) / 15, -low
        d, dmin = (scale.amax(1) / 63).half().float(), (low.amax(1) / 63).half().float()
        sc = (scale / d[:, None]).round().clamp(0, 63).long()
        mn = (low / dmin[:, None]).round().clamp(0, 63).long()
        step = (d[:, None] * sc).clamp(min=1e-12)[:, :, None]
        q = ((w + (dmin[:, None] * mn)[:, :, None]) / step).round().clamp(0, 15).to(torch.uint8)
        out[:, 16:] = (q[:, 0::2] | (q[:, 1::2] << 4)).reshape(n, 128)
        del w, q
    out[:, 0:2], out[:, 2:4] = _half_bytes(d), _half_bytes(dmin)
    out[:, 4:8] = (sc[:, :4] | ((sc[:, 4:] >> 4) << 6)).to(torch.uint8)
    out[:, 8:12] = (mn[:, :4] | ((mn[:, 4:] >> 4) << 6)).to(torch.uint8)
    out[:, 12:16] = ((sc[:, 4:] & 15) | ((mn[:, 4:] & 15) << 4)).to(torch.uint8)
    return out


def _q6_k(g, rows, k, synthetic):
    """Q6_K blocks [rows * k/256][210]."""
    n = rows * (k // 256)
    out = torch.empty(n, 210, dtype=torch.uint8, device="cuda:0")
    if synthetic:
        out[:, :192] = torch.randint(0, 256, (n, 192), dtype=torch.uint8, device="cuda:0", generator=g)
        sc = torch.randint(-32, 32, (n, 16), device="cuda:0", generator=g)
        d = _normal(g, n).abs() * 0.005
    else:
        w = _normal(g, n, 16, 16) / math.sqrt(k)
        big = w.gather(2, w.abs().argmax(2, keepdim=True))[:, :, 0]  # each sub-block's largest value, signed
        scale = big / -32
        top = scale.gather(1, scale.abs().argmax(1, keepdim=True))[:, 0]
        d = (top / -128).half().float()
        sc = (scale / d[:, None]).round().clamp(-128, 127).long()
        step = d[:, None] * sc
        step = torch.where(step == 0, torch.full_like(step, 1e-12), step)[:, :, None]
        q = ((w / step).round().clamp(-32, 31) + 32).to(torch.uint8).view(n, 2, 4, 32)  # [half][t][32]
        lo, hi = q & 15, q >> 4
        out[:, :128] = torch.cat([lo[:, :, 0:2] | (lo[:, :, 2:4] << 4)], 2).reshape(n, 128)
        out[:, 128:192] = (hi[:, :, 0] | (hi[:, :, 1] << 2) | (hi[:, :, 2] << 4) | (hi[:, :, 3] << 6)).reshape(n, 64)
        del w, q, lo, hi
    out[:, 192:208] = sc.to(torch.int8).view(torch.uint8)
    out[:, 208:210] = _half_bytes(d)
    return out


_ROWS_AT_ONCE = 1 << 28  # weights of one piece (the quantiser's temporaries are several times that)


def _blocks(seed, label, kind, rows, k, weights):
    """One tensor's GGUF bytes on the GPU, [rows][row bytes]."""
    g = _generator(seed, label)
    make = _q4_k if kind == "Q4_K" else _q6_k
    at_once = max(1, _ROWS_AT_ONCE // 4 // k)
    parts = [make(g, min(at_once, rows - r), k, weights == "synthetic") for r in range(0, rows, at_once)]
    return (parts[0] if len(parts) == 1 else torch.cat(parts)).view(rows, -1)


def _projections(case):
    """name -> (type, rows, input size) of the case's projections."""
    s = ModelShape(hidden=case["hidden"], head_count=case.get("heads", 8), head_count_kv=case.get("kv_heads", 2),
                   ffn=case.get("ffn", 10240))
    return {name: (t, rows, k) for name, t, rows, k in s.projections()}


_SETS = {"qkv": ("attn_q", "attn_k", "attn_v"), "o": ("attn_output",), "down": ("ffn_down",),
         "ffn": ("ffn_gate", "ffn_up", "ffn_down")}


def _tensors(case, seed):
    """[(label, type, rows, k)] of every weight tensor of a case, in upload order."""
    kind = case["kind"]
    if kind == "attention":
        return []
    if kind == "head":
        return [("head", "Q6_K", case["vocab"], case["hidden"])]
    p = _projections(case)
    if kind == "layers":
        got = [("%d.%s" % (i, n), *p[n]) for i in range(case["layers"]) for n in p]
        return got + ([("head", "Q6_K", case["vocab"], case["hidden"])] if case["head"] else [])
    return [(n, *p[n]) for n in _SETS[{"proj": case.get("set"), "runner": "qkv", "ffn": "ffn"}[kind]]]


def _norm_weights(case, seed):
    """Norm weights of the case (all f32): per layer, and the output norm."""
    got = {}
    for i in range(case.get("layers", 1)):
        g = _generator(seed, "norms %d" % i)
        for name in ("attn_norm", "post_attention_norm", "ffn_norm", "post_ffw_norm"):
            if case["kind"] == "layers":
                got["%d.%s" % (i, name)] = 1 + 0.1 * _normal(g, case["hidden"])
        got["%d.attn_q_norm" % i] = 0.25 * (1 + 0.1 * _normal(g, 256))  # scores of a few units
        got["%d.attn_k_norm" % i] = 1 + 0.1 * _normal(g, 256)
    if case["kind"] == "layers":
        got["output_norm"] = 1 + 0.1 * _normal(_generator(seed, "output norm"), case["hidden"])
    return got


def _rings(case, seed):
    """f16 key and value rings, [layers][2][kv heads][capacity][256], filled as far as the conversation went."""
    n, kv, cap = case.get("layers", 1), case["kv_heads"], case["capacity"]
    rings = torch.zeros(n, 2, kv, cap, 256, dtype=torch.float16, device="cuda:0")
    used = min(cap, case["position"])
    for i in range(n):
        rings[i, :, :, :used] = _normal(_generator(seed, "ring %d" % i), 2, kv, used, 256).half()
    return rings


def _inputs(case, seed):
    """The call's activations."""
    g, t = _generator(seed, "input"), case["tokens"]
    if case["kind"] == "attention":
        return {"q": 2 * _normal(g, t, case["heads"], 256), "k": 2 * _normal(g, t, case["kv_heads"], 256),
                "v": 2 * _normal(g, t, case["kv_heads"], 256)}
    if case["kind"] == "proj":
        return {"x": _normal(g, t, _tensors(case, seed)[0][3])}
    return {"x": _normal(g, t, case["hidden"]) * (4 if case["kind"] == "layers" else 1)}


_stream = None


def _the_stream():
    """The program's stream: every pass of this process is queued on it."""
    global _stream
    if _stream is None:
        _stream = torch.cuda.Stream()
    return _stream


class State:
    def __init__(self):
        self.handles = []

    def __del__(self):
        try:
            torch.cuda.synchronize()
            for h in self.handles:
                H.releaseHipQuantizedWeightHandle(h)
        except Exception:
            pass


def _upload(kind, blocks, k, rows):
    torch.cuda.current_stream().synchronize()
    out = ctypes.c_uint64(0)
    H.assertHipOk(H.lib().hp_hip_weight_upload_device(H.TYPE_IDS[kind], blocks.data_ptr(), blocks.numel(), k, rows,
                                                      ctypes.byref(out)), "upload")
    return H.HipQuantizedWeightHandle(out.value, kind, blocks.numel(), rows, k)


def prepare(case, seed):
    s = State()
    s.case, s.stream = case, _the_stream()
    s.weights = {}
    for label, kind, rows, k in _tensors(case, seed):
        s.weights[label] = _upload(kind, _blocks(seed, label, kind, rows, k, case["weights"]), k, rows)
        s.handles.append(s.weights[label])
    s.inputs = _inputs(case, seed)
    kind, t = case["kind"], case["tokens"]
    f32 = lambda *shape: torch.empty(*shape, device="cuda:0")  # noqa: E731
    if kind == "runner":
        s.x = s.inputs["x"].cpu().numpy()
    elif kind == "proj":
        s.out = {n: f32(t, w.rowCount) for n, w in s.weights.items()}
    elif kind == "ffn":
        s.mid, s.out = f32(t, case["ffn"]), f32(t, case["hidden"])
    if kind in ("attention", "layers"):
        s.norms = _norm_weights(case, seed)
        s.rings = _rings(case, seed)
        s.position = torch.full((1,), case["position"], dtype=torch.int32, device="cuda:0")
        s.config = H.attention_config(case["heads"], case["kv_heads"], case["capacity"], rope_freq_base=FREQ_BASE,
                                      sliding_window=case["window"], epsilon=EPSILON)
    if kind == "attention":
        s.q, s.out = f32(t, case["heads"], 256), f32(t, case["heads"], 256)
    if kind == "layers":
        s.hidden, s.normed = f32(t, case["hidden"]), f32(t, case["hidden"])
        s.layers = []
        for i in range(case["layers"]):
            layer = H.HipDecodeLayer()
            for n in _projections(case):
                setattr(layer, n, s.weights["%d.%s" % (i, n)].handle)
            for n in ("attn_norm", "attn_q_norm", "attn_k_norm", "post_attention_norm", "ffn_norm", "post_ffw_norm"):
                setattr(layer, "d_" + n, s.norms["%d.%s" % (i, n)].data_ptr())
            layer.layer_output_scale = 1.0
            layer.d_key_cache, layer.d_value_cache = s.rings[i, 0].data_ptr(), s.rings[i, 1].data_ptr()
            layer.attention = s.config
            s.layers.append(layer)
    if kind == "head" or case.get("head"):
        s.logits = f32(t, case["vocab"])
    if kind == "head":
        k = case["k"]
        s.ids, s.values = torch.empty(t, k, dtype=torch.int32, device="cuda:0"), f32(t, k)
        s.probabilities = torch.zeros(t, k, dtype=torch.float64, device="cuda:0")
        s.tokens, s.kept = (torch.empty(t, dtype=torch.int32, device="cuda:0") for _ in range(2))
        s.seed = torch.tensor([SEED_RNG + seed], dtype=torch.int32, device="cuda:0")
        s.rng = torch.empty_like(s.seed)
        s.sampling = H.resolveGenerationSamplingOptions(topK=k)
    torch.cuda.synchronize()
    return s


def run(s):
    case, kind, t = s.case, s.case["kind"], s.case["tokens"]
    q = s.stream.cuda_stream
    if kind == "runner":
        return H.matMulQuantizedHipResidentMulti(list(s.weights.values()), s.x, case["hidden"], t)
    if kind == "proj":
        ws, outs = list(s.weights.values()), list(s.out.values())
        H.matmul_multi_device([w.handle for w in ws], s.inputs["x"].data_ptr(), ws[0].inputSize, t,
                              [o.data_ptr() for o in outs], [o.numel() for o in outs], q)
        return s.out
    if kind == "ffn":
        H.matmul_geglu_device(s.weights["ffn_gate"].handle, s.weights["ffn_up"].handle, s.inputs["x"].data_ptr(),
                              case["hidden"], t, s.mid.data_ptr(), case["ffn"], q)
        H.matmul_multi_device([s.weights["ffn_down"].handle], s.mid.data_ptr(), case["ffn"], t, [s.out.data_ptr()],
                              [s.out.numel()], q)
        return {"hidden": s.mid, "out": s.out}
    if kind == "attention":
        x, keys, values = s.inputs, s.rings[0, 0], s.rings[0, 1]
        H.attention_prep_device(s.config, x["q"].data_ptr(), x["k"].data_ptr(), x["v"].data_ptr(),
                                s.norms["0.attn_q_norm"].data_ptr(), s.norms["0.attn_k_norm"].data_ptr(),
                                s.position.data_ptr(), s.q.data_ptr(), keys.data_ptr(), values.data_ptr(), q, t)
        H.gqa_attention_device(s.config, s.q.data_ptr(), keys.data_ptr(), values.data_ptr(), s.position.data_ptr(),
                               s.out.data_ptr(), q, t)
        return {"out": s.out, "rings": s.rings}
    with torch.cuda.stream(s.stream):
        if kind == "head":
            s.rng.copy_(s.seed)  # the request's generator
            x = s.inputs["x"]
        else:
            s.hidden.copy_(s.inputs["x"])  # the embedding rows
            x = s.normed
    if kind == "layers":
        H.decode_layers_device(s.layers, s.hidden.data_ptr(), s.position.data_ptr(),
                               s.norms["output_norm"].data_ptr(), s.normed.data_ptr(), q, t)
    if kind == "head" or case["head"]:
        H.matmul_multi_device([s.weights["head"].handle], x.data_ptr(), case["hidden"], t, [s.logits.data_ptr()],
                              [s.logits.numel()], q)
    if kind == "layers":
        out = {"hidden": s.hidden, "normed": s.normed, "rings": s.rings}
        return dict(out, logits=s.logits) if case["head"] else out
    k = case["k"]
    H.assertHipOk(H.lib().hp_hip_topk_device(s.logits.data_ptr(), t, case["vocab"], k, 0.0, s.ids.data_ptr(),
                                             s.values.data_ptr(), q), "topk")
    H.sample_device(s.ids.data_ptr(), s.values.data_ptr(), t, k, k, s.sampling, s.rng.data_ptr(),
                    s.tokens.data_ptr(), s.probabilities.data_ptr(), s.kept.data_ptr(), q)
    return {"logits": s.logits, "ids": s.ids, "values": s.values, "probabilities": s.probabilities,
            "tokens": s.tokens, "kept": s.kept}


# ---- what a pass needs ---------------------------------------------------------------------------------------

_BLOCK_BYTES = {"Q4_K": 144, "Q6_K": 210}


def _attention_work(case):
    """Bytes and operations of one layer's attention: the ring slots its tokens see, read once."""
    t, p = case["tokens"], case["position"]
    limit = min(case["capacity"], case["window"] or case["capacity"])
    last = p + t - 1
    seen = min(limit, last + 1)
    start = last + 1 - seen
    keys = sum(max(0, p + i + 1 - start) for i in range(t))
    return 2 * seen * case["kv_heads"] * 512, 4 * 256 * case["heads"] * keys


def work(case):
    kind, t = case["kind"], case["tokens"]
    size, ops = 0, 0
    for label, wt, rows, k in _tensors(case, 0):
        size += rows * (k // 256) * _BLOCK_BYTES[wt]
        ops += 2 * rows * k * t
    if kind in ("proj", "runner"):
        ws = _tensors(case, 0)
        size += 4 * t * (ws[0][3] + sum(w[2] for w in ws))
    elif kind == "ffn":
        size += 4 * t * (2 * case["hidden"] + 2 * case["ffn"])
    elif kind == "head":
        size += 4 * t * (case["hidden"] + case["vocab"])
    elif kind == "attention":
        b, f = _attention_work(case)
        size += b + 4 * 256 * t * (2 * case["heads"] + 2 * case["kv_heads"])
        ops += f
    else:
        b, f = _attention_work(case)
        size += case["layers"] * b + 4 * t * (3 * case["hidden"] + (case["vocab"] if case["head"] else 0))
        ops += case["layers"] * f
    return {"bytes": size, "flops": ops}


def tolerance(case):
    """Four times what the same pass through this framework's other kernels (another order of the f32 sums) differed
    by, or, for attention and layers, what it differed from exact() by."""
    kind, t = case["kind"], case["tokens"]
    if kind in ("runner", "head") or (kind in ("proj", "ffn") and t < 64):
        return "exact"  # stated so by the entry points: the reference's own f32 order
    if kind == "proj":
        return {"rel": 6e-7, "max": 4e-6}
    if kind == "ffn":  # an f16 step of gelu, and the Q8_K steps of down's input that follow from it
        return {"rel": 5e-4, "max": 2e-2}
    if kind == "attention":  # f16 output rows
        return {"rel": 8e-4, "max": 4e-3}
    # Q8_K steps that fall the other way, carried through the layers after them: 0.002-0.011 over three layers (over
    # all 42 a last-bit change of the input moves the logits by 0.09, so there this asks for the same order of sums)
    return {"rel": 2.5e-2, "max": 0.9}


# ---- the same in 64 bits -------------------------------------------------------------------------------------

def _dequantized(kind, blocks, k):
    """f64 [rows][k] of GGUF blocks."""
    rows = blocks.shape[0]
    b = blocks.view(rows * (k // 256), -1)
    half = lambda at: b[:, at:at + 2].contiguous().view(torch.float16).double()  # noqa: E731
    if kind == "Q4_K":
        s = b[:, 4:16].long()
        sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)], 1)
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1)
        qs = b[:, 16:].view(-1, 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], 2).view(-1, 8, 32).double()
        w = (half(0) * sc)[:, :, None] * q - (half(2) * mn)[:, :, None]
    else:
        ql, qh = b[:, :128].view(-1, 2, 2, 32), b[:, 128:192].view(-1, 2, 1, 32)
        lo = torch.cat([ql & 15, ql >> 4], 2)
        hi = torch.cat([qh & 3, (qh >> 2) & 3, (qh >> 4) & 3, qh >> 6], 2)
        q = (lo | (hi << 4)).view(-1, 16, 16).double() - 32
        w = (half(208) * b[:, 192:208].view(torch.int8).double())[:, :, None] * q
    return w.reshape(rows, k)


def _q8_k(x):
    """The Q8_K values of x's rows (the path's definition: 8-bit quants of every 256 inputs, in f32), as f64."""
    v = x.float().reshape(x.shape[0], -1, 256)
    mag = v.abs()
    top = mag.amax(2, keepdim=True)
    at = torch.where(mag == top, torch.arange(256, device=v.device), 256).amin(2, keepdim=True)
    peak = v.gather(2, at)
    inv = (-127.0 / torch.where(top == 0, torch.ones_like(peak), peak).double()).float()
    p = (inv * v).double()
    q = (torch.sign(p) * torch.floor(p.abs() + 0.5)).clamp(-128, 127)
    out = torch.where(top == 0, torch.zeros_like(q), q * (1.0 / inv.double()).float().double())
    return out.reshape(x.shape)


def _project(case, seed, tensor, x):
    """x [tokens][k] through one weight tensor, f64 [tokens][rows]."""
    label, kind, rows, k = tensor
    blocks = _blocks(seed, label, kind, rows, k, case["weights"])
    xq, step = _q8_k(x), max(1, (1 << 27) // k)
    return torch.cat([xq @ _dequantized(kind, blocks[r:r + step], k).T for r in range(0, rows, step)], 1)


def _rms(x, w):
    y = x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPSILON)
    return y if w is None else y * w.double()


def _half64(x):
    return x.clamp(-65504, 65504).half().double()


def _gelu(x):
    """The path's gelu: of the f16 value of its input, rounded to f16; 0 or the input itself past +-10."""
    h = _half64(x.float().double())
    y = 0.5 * h * (1 + torch.tanh(math.sqrt(2 / math.pi) * h * (1 + 0.044715 * h * h)))
    return torch.where(x <= -10, torch.zeros_like(x), torch.where(x >= 10, x, _half64(y)))


def _rope(x, position):
    """ropeNeox over 256 dims: the angle of a pair is the previous one times the step, kept in 32 bits."""
    theta = np.arange(position, position + x.shape[0], dtype=np.float64)
    step, angles = FREQ_BASE ** (-2.0 / 256), []
    for _ in range(128):
        angles.append(theta)
        theta = (theta * step).astype(np.float32).astype(np.float64)
    a = torch.from_numpy(np.stack(angles, 1)).to(x.device)[:, None, :]
    x0, x1 = x[..., :128], x[..., 128:]
    return torch.cat([x0 * a.cos() - x1 * a.sin(), x0 * a.sin() + x1 * a.cos()], -1)


def _attend(case, q, k, v, q_norm, k_norm, ring):
    """Head norms, RoPE and append ([tokens][heads][256] in, ring [2][kv heads][capacity][256] f64 updated in
    place), then the attention of every token up to its own position inside the last token's window."""
    t, p, cap = case["tokens"], case["position"], case["capacity"]
    q, k, v = _rope(_rms(q, q_norm), p), _rope(_rms(k, k_norm), p), _rms(v, None)
    slots = torch.arange(p, p + t, device=q.device) % cap
    ring[0][:, slots], ring[1][:, slots] = k.transpose(0, 1), v.transpose(0, 1)
    seen = min(cap, case["window"] or cap, p + t)
    keys = torch.arange(p + t - seen, p + t, device=q.device)
    kk, vv = _half64(ring[0][:, keys % cap]), _half64(ring[1][:, keys % cap])
    groups = case["heads"] // case["kv_heads"]
    hidden = keys[None, :] > torch.arange(p, p + t, device=q.device)[:, None]
    out = []
    for h in range(case["heads"]):
        scores = _half64(q[:, h]) @ kk[h // groups].T
        out.append(torch.softmax(scores.masked_fill(hidden, -math.inf), 1) @ vv[h // groups])
    return torch.stack(out, 1)


def exact(case, seed):
    kind, t = case["kind"], case["tokens"]
    if kind == "layers" and case["layers"] > 4:
        return None  # a Q8_K step that falls the other way early moves everything after it
    x = {n: v.double() for n, v in _inputs(case, seed).items()}
    ws = {w[0]: w for w in _tensors(case, seed)}
    if kind in ("proj", "runner"):
        out = {n: _project(case, seed, w, x["x"]) for n, w in ws.items()}
        return [v.reshape(-1) for v in out.values()] if kind == "runner" else out
    if kind == "head":
        return {"logits": _project(case, seed, ws["head"], x["x"]), "ids": None, "values": None,
                "probabilities": None, "tokens": None, "kept": None}

    def ffn(y, prefix=""):
        gate, up = (_project(case, seed, ws[prefix + n], y) for n in ("ffn_gate", "ffn_up"))
        mid = _gelu(gate) * up
        return mid, _project(case, seed, ws[prefix + "ffn_down"], mid)

    if kind == "ffn":
        mid, out = ffn(x["x"])
        return {"hidden": mid, "out": out}
    norms, rings = _norm_weights(case, seed), _rings(case, seed).double()
    if kind == "attention":
        out = _attend(case, x["q"], x["k"], x["v"], norms["0.attn_q_norm"], norms["0.attn_k_norm"], rings[0])
        return {"out": out, "rings": rings}
    y = x["x"]
    for i in range(case["layers"]):
        n = lambda name: norms["%d.%s" % (i, name)]  # noqa: E731
        z = _rms(y, n("attn_norm"))
        q, k, v = (_project(case, seed, ws["%d.%s" % (i, w)], z).view(t, -1, 256)
                   for w in ("attn_q", "attn_k", "attn_v"))
        a = _half64(_attend(case, q, k, v, n("attn_q_norm"), n("attn_k_norm"), rings[i])).view(t, -1)
        y = y + _rms(_project(case, seed, ws["%d.attn_output" % i], a), n("post_attention_norm"))
        y = y + _rms(ffn(_rms(y, n("ffn_norm")), "%d." % i)[1], n("post_ffw_norm"))
    return {"hidden": y, "normed": _rms(y, norms["output_norm"]), "rings": rings}
