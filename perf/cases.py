"""The work that users of the PLaMo-3 0.8B token loop have it do, as measurable cases.

Kernel cases go through the C ABI's kernel entry points (include/plamo_hip.h) at the
projection and attention shapes of the model, a few layers in turn as a step or a prompt
passes through them: each layer has weights (or a KV cache) of its own, more than the
memory-side cache holds in all, so that they come from memory as they do in the model.
Whole-model cases go through Runtime and Batch on a synthetic model directory.
"""
import ctypes
import json
import math
import os
import sys

import numpy as np
import torch

_ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(_ROOT, "plamo3-0.8b-runtime_amd"))

import plamo_hip  # noqa: E402
from plamo_hip import native, synth  # noqa: E402

HIDDEN, HEADS, DIM, INTER, VOCAB, LAYERS, WINDOW = 1536, 16, 128, 6144, 107520, 16, 2048
SCALE = 1.0 / math.sqrt(DIM)
# projection -> (output features, input features, layers of a kernel case)
SHAPES = {"qkv": (2304, 1536, 16), "o": (1536, 2048, 16), "gate_up": (12288, 1536, 4), "down": (1536, 6144, 8),
          "head": (VOCAB, 1536, 1)}
P12 = 0.7686  # bytes of a .p12 tensor over its BF16 bytes, for N(0, 0.02) weights
PARAMS = LAYERS * sum(SHAPES[s][0] * SHAPES[s][1] for s in ("qkv", "o", "gate_up", "down"))
HEAD = VOCAB * HIDDEN


def listed():
    return [
        # one projection of a greedy decode step: the smallest launch that a token waits for
        {"name": "step_qkv", "kind": "linear", "shape": "qkv", "rows": 1, "packed": False},
        # the same for four translated segments at once, on the smaller weight file
        {"name": "step_down_p12_rows4", "kind": "linear", "shape": "down", "rows": 4, "packed": True},
        # a full forward() call of 16 tokens, or the last few words of a prompt
        {"name": "prompt16_o", "kind": "gemm", "shape": "o", "tokens": 16},
        # a sentence, with its template around it
        {"name": "prompt77_gate_up", "kind": "gemm", "shape": "gate_up", "tokens": 77},
        # a paragraph
        {"name": "prompt300_down", "kind": "gemm", "shape": "down", "tokens": 300},
        # a document: one full prefill chunk
        {"name": "prompt2048_gate_up", "kind": "gemm", "shape": "gate_up", "tokens": 2048},
        # the sliding-window layers at a paragraph that comes after a long text
        {"name": "attend_local_333", "kind": "attend", "full": False, "tokens": 333, "p0": 3001, "layers": 14},
        # the global layers at the second chunk of a document
        {"name": "attend_global_2048", "kind": "attend", "full": True, "tokens": 2048, "p0": 2048, "layers": 2},
        # the sliding-window layers of a decode step early in a translation
        {"name": "step_attend_local", "kind": "step", "full": False, "rows": 1, "pos": 343, "layers": 14},
        # the global layers of a decode step deep in a long document, two sequences
        {"name": "step_attend_global_long", "kind": "step", "full": True, "rows": 2, "pos": 20011, "layers": 2},
        # a sentence scored: its prompt, then the steps of a known translation, plain weights
        {"name": "sentence", "kind": "sequence", "prompt": 61, "steps": 16},
        # four paragraphs side by side on .p12 weights: their prompts, then batch steps
        {"name": "paragraphs_p12", "kind": "lanes", "prompt": 301, "spread": 87, "steps": 8},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng):
    kind = rng.choice(["linear", "gemm", "gemm", "gemm", "attend", "attend", "step", "sequence", "lanes"])
    if kind == "linear":
        return {"kind": kind, "shape": rng.choice(["qkv", "o", "gate_up", "down", "head"]), "rows": rng.randint(1, 4),
                "packed": rng.random() < 0.5}
    if kind == "gemm":
        return {"kind": kind, "shape": rng.choice(["qkv", "o", "gate_up", "down"]), "tokens": _log(rng, 2, 2048)}
    if kind == "attend":
        full, tokens = rng.random() < 0.5, _log(rng, 2, 2048)
        p0 = 0 if rng.random() < 0.3 else _log(rng, 16, 4096 if full else 16384)
        return {"kind": kind, "full": full, "tokens": tokens, "p0": p0, "layers": 2 if full else 6}
    if kind == "step":
        full = rng.random() < 0.5
        return {"kind": kind, "full": full, "rows": rng.randint(1, 4), "pos": _log(rng, 1, 30000),
                "layers": 2 if full else 14}
    if kind == "sequence":
        return {"kind": kind, "prompt": _log(rng, 2, 512), "steps": rng.randint(2, 16)}
    prompt = _log(rng, 16, 301)
    return {"kind": kind, "prompt": prompt, "spread": rng.randint(0, prompt // 4), "steps": rng.randint(2, 8)}


# ------------------------------------------------------------------------------ inputs
def _gen(seed):
    return torch.Generator("cuda").manual_seed(int(seed) * 7919 + 17)


def _randn(g, *shape, std=1.0):
    return (torch.randn(*shape, generator=g, device="cuda") * std).to(torch.bfloat16)


def _weights(g, shape):
    m, n, layers = SHAPES[shape]
    return [_randn(g, m, n, std=0.02) for _ in range(layers)]


def _rows(g, shape, rows):
    """Activation rows of a projection: normed rows, attention outputs, or SwiGLU activations."""
    n = SHAPES[shape][1]
    if shape == "o":
        return _randn(g, rows, n, std=0.3)
    if shape == "down":
        a, b = _randn(g, rows, n, std=0.8).float(), _randn(g, rows, n, std=0.8).float()
        return (torch.nn.functional.silu(a) * b).to(torch.bfloat16)
    return _randn(g, rows, n)


def _model():
    """The synthetic checkpoint, made once."""
    return synth.ensure_model()


def _tokens(seed, n):
    return np.random.default_rng([11, int(seed)]).integers(1024, VOCAB, n).tolist()


def _lane_lengths(case):
    return [max(1, case["prompt"] - i * case["spread"]) for i in range(4)]


def _rope(rows, full, context=0):
    """The framework's RoPE table (BF16 cos | sin << 16) -> int32 [rows][64] on the GPU."""
    freqs = synth.frequencies()[1 if full else 0]
    out = np.empty((rows, 64), dtype=np.uint32)
    native.call(native.load().plamo_rope_table, (ctypes.c_double * 64)(*freqs), rows, 1 if full else 0,
                out.ctypes.data)
    return torch.from_numpy(out.view(np.int32)).cuda()


def _capacity(case):
    """Cache slots of a layer: the context (here the next 1,024 tokens), or the sliding
    window and one prefill chunk."""
    last = case["p0"] + case["tokens"] if case["kind"] == "attend" else case["pos"] + 1
    context = -(-last // 1024) * 1024
    return context if case["full"] else min(context, 2 * WINDOW)


def _inputs(case, seed):
    """The tensors of a kernel case, from the seed alone."""
    g, s = _gen(seed), {}
    if case["kind"] in ("linear", "gemm"):
        rows = case["rows"] if case["kind"] == "linear" else case["tokens"]
        s["x"], s["w"] = _rows(g, case["shape"], rows), _weights(g, case["shape"])
    elif case["kind"] == "attend":
        cap = _capacity(case)
        # queries and keys leave a unit RMS norm; values are a projection's outputs
        s["q"] = [_randn(g, case["tokens"], HEADS, DIM) for _ in range(case["layers"])]
        s["k"] = [_randn(g, cap, DIM) for _ in range(case["layers"])]
        s["v"] = [_randn(g, cap, DIM, std=0.8) for _ in range(case["layers"])]
    else:
        cap, rows = _capacity(case), case["rows"]
        s["qkv"] = [_randn(g, rows, 18 * DIM, std=0.8).float() for _ in range(case["layers"])]
        s["gain"] = [_randn(g, 2, DIM, std=0.05) for _ in range(case["layers"])]
        s["k"] = [_randn(g, rows, cap, DIM) for _ in range(case["layers"])]
        s["v"] = [_randn(g, rows, cap, DIM, std=0.8) for _ in range(case["layers"])]
    return s


def _positions(case):
    """Sequences side by side stand at slightly different positions."""
    return [max(0, case["pos"] - 37 * q) for q in range(case["rows"])]


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("sequence", "lanes"):
        directory, sha = _model()
        if kind == "sequence":
            toks = _tokens(seed, case["prompt"] + case["steps"])
            rt = plamo_hip.Runtime(directory, len(toks) + 8, source_sha256=sha)
            return {"kind": kind, "rt": rt, "prompt": toks[:case["prompt"]], "forced": toks[case["prompt"]:]}
        lengths = _lane_lengths(case)
        toks = [_tokens(1000 * seed + i, n + case["steps"]) for i, n in enumerate(lengths)]
        rt = plamo_hip.Runtime(directory, max(lengths) + case["steps"] + 8, packed=True, source_sha256=sha)
        return {"kind": kind, "rt": rt, "batch": plamo_hip.Batch(rt),
                "prompts": [t[:n] for t, n in zip(toks, lengths)],
                "forced": [[t[n + k] for t, n in zip(toks, lengths)] for k in range(case["steps"])]}
    s = _inputs(case, seed)
    s.update(kind=kind, lib=native.load(), case=dict(case))
    if kind == "linear":
        m, n, _ = SHAPES[case["shape"]]
        s["x"] = s["x"].float()  # the entry point takes FP32 rows that hold BF16 values
        if case["packed"]:
            s["w"] = [tuple(torch.from_numpy(a).cuda() for a in (payload, table.view(np.int32)))
                      for payload, table in (native.pack_tensor(w.view(torch.int16).cpu().numpy().view(np.uint16))
                                             for w in s["w"])]
        else:
            s["w"] = [(w, None) for w in s["w"]]
        # the LM head's outputs are BF16 logits, the others' FP32 rows
        out = torch.bfloat16 if case["shape"] == "head" else torch.float32
        s["y"] = [torch.empty(case["rows"], m, dtype=out, device="cuda") for _ in s["w"]]
    elif kind == "gemm":
        cols = INTER if case["shape"] == "gate_up" else SHAPES[case["shape"]][0]
        s["y"] = [torch.empty(case["tokens"], cols, dtype=torch.bfloat16, device="cuda") for _ in s["w"]]
    elif kind == "attend":
        s["rope"] = _rope(WINDOW + 16, False)
        s["y"] = [torch.empty(case["tokens"], HEADS * DIM, dtype=torch.bfloat16, device="cuda") for _ in s["q"]]
    else:
        s["rope"] = _rope(WINDOW + 16, False)
        s["grope"] = _rope(_capacity(case), True) if case["full"] else s["rope"]
        s["pos"] = native.i32(_positions(case))
        s["y"] = [torch.empty(case["rows"], HEADS * DIM, dtype=torch.bfloat16, device="cuda") for _ in s["qkv"]]
    return s


# --------------------------------------------------------------------------------- run
def run(s):
    kind = s["kind"]
    if kind == "sequence":
        rt = s["rt"]
        rt.reset()
        rt.prefill(s["prompt"])
        for t in s["forced"]:
            rt.forward([t])
        return {"logits": rt.logits(), "hidden": rt.hidden()}
    if kind == "lanes":
        b = s["batch"]
        b.reset()
        b.prefill(s["prompts"])
        for tokens in s["forced"]:
            b.step(tokens)
        # a lane's logits arrive as BF16 bits
        return {"logits": [(b.logit_bits(i).astype(np.uint32) << 16).view(np.float32) for i in range(4)],
                "hidden": [b.hidden(i) for i in range(4)]}
    lib, case, stream = s["lib"], s["case"], torch.cuda.current_stream().cuda_stream
    rc = 0
    if kind == "linear":
        m, n, _ = SHAPES[case["shape"]]
        mode = 2 if case["shape"] == "head" else 0
        for (w, table), y in zip(s["w"], s["y"]):
            rc |= lib.plamo_kernel_linear(w.data_ptr(), table.data_ptr() if table is not None else 0,
                                          s["x"].data_ptr(), y.data_ptr(), n, m, case["rows"], mode, stream)
    elif kind == "gemm":
        m, n, _ = SHAPES[case["shape"]]
        mode = 3 if case["shape"] == "gate_up" else 1
        for w, y in zip(s["w"], s["y"]):
            rc |= lib.plamo_kernel_gemm(w.data_ptr(), 0, s["x"].data_ptr(), y.data_ptr(), n, m, case["tokens"], mode,
                                        stream)
    elif kind == "attend":
        for q, k, v, y in zip(s["q"], s["k"], s["v"], s["y"]):
            rc |= lib.plamo_kernel_attention_prefill(q.data_ptr(), k.data_ptr(), v.data_ptr(), k.shape[0], case["p0"],
                                                     case["tokens"], 1 if case["full"] else 0, s["rope"].data_ptr(),
                                                     y.data_ptr(), stream)
    else:
        for qkv, gain, k, v, y in zip(s["qkv"], s["gain"], s["k"], s["v"], s["y"]):
            rc |= lib.plamo_kernel_attention_decode(qkv.data_ptr(), gain[0].data_ptr(), gain[1].data_ptr(),
                                                    k.data_ptr(), v.data_ptr(), k.shape[1], s["pos"], case["rows"],
                                                    1 if case["full"] else 0, s["rope"].data_ptr(),
                                                    s["grope"].data_ptr(), y.data_ptr(), stream)
    if rc:
        raise RuntimeError("kernel entry point failed: %d" % rc)
    if kind == "step":  # the step writes its key and value into the caches
        return {"out": s["y"], "keys": s["k"], "values": s["v"]}
    return s["y"]


# -------------------------------------------------------------------------------- work
def _pairs(tokens, p0, full):
    """(query, visible key) pairs of `tokens` queries from position p0."""
    n = np.arange(p0 + 1, p0 + tokens + 1, dtype=np.int64)
    return int((n if full else np.minimum(n, WINDOW)).sum())


def work(case):
    kind = case["kind"]
    if kind in ("linear", "gemm"):
        m, n, layers = SHAPES[case["shape"]]
        rows = case["rows"] if kind == "linear" else case["tokens"]
        cols = INTER if kind == "gemm" and case["shape"] == "gate_up" else m
        element = 4 if kind == "linear" and case["shape"] != "head" else 2
        per = m * n * 2 * (P12 if case.get("packed") else 1) + rows * cols * element
        return {"bytes": layers * per + rows * n * (4 if kind == "linear" else 2), "flops": 2 * layers * rows * m * n}
    if kind == "attend":
        t, p0, full = case["tokens"], case["p0"], case["full"]
        keys = p0 + t if full else min(p0 + t, WINDOW - 1 + t)
        return {"bytes": case["layers"] * (2 * t * HEADS * DIM * 2 + keys * DIM * 4),
                "flops": case["layers"] * 4 * HEADS * DIM * _pairs(t, p0, full)}
    if kind == "step":
        pairs = sum(_pairs(1, p, case["full"]) for p in _positions(case))
        return {"bytes": case["layers"] * (pairs * DIM * 4 + case["rows"] * (18 * DIM * 4 + HEADS * DIM * 2 + DIM * 4)),
                "flops": case["layers"] * 4 * HEADS * DIM * pairs}
    lanes = [case["prompt"]] if kind == "sequence" else _lane_lengths(case)
    ratio, steps = 1 if kind == "sequence" else P12, case["steps"]
    total, flops = 0.0, 0.0
    for n in lanes:  # every prompt passes over the layers' weights once, and the head's
        total += (PARAMS + HEAD) * 2 * ratio
        flops += 2 * PARAMS * (n + steps) + 2 * HEAD * (steps + 1)
        flops += 4 * HEADS * DIM * (14 * _pairs(n + steps, 0, False) + 2 * _pairs(n + steps, 0, True))
    total += steps * (PARAMS + HEAD) * 2 * ratio  # and a step's rows share one pass
    total += sum(LAYERS * DIM * 4 * (n + k) for n in lanes for k in range(steps))
    return {"bytes": total, "flops": flops}


def tolerance(case):
    kind = case["kind"]
    if kind in ("sequence", "lanes"):
        return {"rel": 7e-2}  # sixteen layers of BF16 rounding (1.7e-2 from 64 bits)
    if kind == "gemm" and case["shape"] == "gate_up":
        return {"rel": 1.4e-2}  # the gate, the up, the SiLU and the result rounded to BF16 (3.6e-3)
    if kind == "step":
        # queries and keys rounded four times before the scores, which the global layers'
        # RoPE scales by 2.4 (2.9e-3 local, 6.6e-3 global)
        return {"rel": 2.6e-2 if case["full"] else 1.2e-2}
    if kind == "attend" and not case["full"]:
        return {"rel": 1.2e-2}  # the keys rounded as they turn (3e-3)
    return {"rel": 7e-3}  # one BF16 rounding of each result (1.7e-3)


# ------------------------------------------------------------------------------- exact
def _table64(table):
    t = table.long() & 0xFFFFFFFF
    both = torch.stack([(t & 0xFFFF) << 16, t & 0xFFFF0000], 0)
    both = torch.where(both >= 2 ** 31, both - 2 ** 32, both).to(torch.int32).view(torch.float32).double()
    return both[0], both[1]


def _rotate(x, c, s):
    """Rotate-half RoPE of x [..., 128] with c, s [..., 64]."""
    a, b = x[..., :64], x[..., 64:]
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def _rms(x):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-6)


def _softmax_pv(q, k, v, visible):
    """q [T][16][128], k and v [keys][128], visible [T][keys] -> [T][2048]."""
    out = []
    for i in range(0, q.shape[0], 64):
        s = (q[i:i + 64].reshape(-1, DIM) @ k.T).reshape(-1, HEADS, k.shape[0]) * SCALE
        s = s.masked_fill(~visible[i:i + 64][:, None, :], -math.inf)
        p = torch.softmax(s, -1)
        out.append((p.reshape(-1, k.shape[0]) @ v).reshape(-1, HEADS * DIM))
    return torch.cat(out)


def _visible(pos, first, count, full):
    key = torch.arange(first, first + count, device="cuda")[None]
    ok = key <= pos[:, None]
    return ok if full else ok & (key > pos[:, None] - WINDOW)


def _exact_attend(case, s):
    cap, p0, t, full = _capacity(case), case["p0"], case["tokens"], case["full"]
    c, sn = _table64(_rope(WINDOW + 16, False))
    got = []
    for q, k, v in zip(s["q"], s["k"], s["v"]):
        out, step = [], t if full else 16  # local keys turn with each 16-token chunk's base
        for i in range(0, t, step):
            n = min(step, t - i)
            pos = torch.arange(p0 + i, p0 + i + n, device="cuda")
            first = 0 if full else max(0, p0 + i - (WINDOW - 1))
            at = torch.arange(first, p0 + i + n, device="cuda")
            kk, vv = k[at % cap].double(), v[at % cap].double()
            if not full:
                kk = _rotate(kk, c[at - first], sn[at - first])
            out.append(_softmax_pv(q[i:i + n].double(), kk, vv, _visible(pos, first, len(at), full)))
        got.append(torch.cat(out))
    return got


def _exact_step(case, s):
    cap, full = _capacity(case), case["full"]
    c, sn = _table64(_rope(cap, True) if full else _rope(WINDOW + 16, False))
    got = {"out": [], "keys": [], "values": []}
    for qkv, gain, keys, values in zip(s["qkv"], s["gain"], s["k"], s["v"]):
        keys, values, out = keys.double(), values.double(), []
        for row, pos in enumerate(_positions(case)):
            x, g = qkv[row].double(), gain.double() + 1.0
            base = 0 if full else max(0, pos - (WINDOW - 1))
            q = _rotate(_rms(x[:HEADS * DIM].reshape(HEADS, DIM)) * g[0], c[pos - base], sn[pos - base])
            k = _rms(x[HEADS * DIM:17 * DIM]) * g[1]
            keys[row, pos % cap] = _rotate(k, c[pos], sn[pos]) if full else k
            values[row, pos % cap] = x[17 * DIM:]
            at = torch.arange(base, pos + 1, device="cuda")
            kk = keys[row, at % cap]
            if not full:
                kk = _rotate(kk, c[at - base], sn[at - base])
            seen = torch.ones(1, len(at), dtype=torch.bool, device="cuda")
            out.append(_softmax_pv(q[None], kk, values[row, at % cap], seen))
        got["out"].append(torch.cat(out))
        got["keys"].append(keys)
        got["values"].append(values)
    return got


def _exact_model(tokens):
    """Logits and final hidden row of each token list's last token, in 64 bits throughout."""
    directory, _ = _model()
    path = os.path.join(directory, "model.safetensors")
    with open(path, "rb") as f:
        n = int.from_bytes(f.read(8), "little")
        header = json.loads(f.read(n))
    data = np.memmap(path, dtype=np.uint8, mode="r", offset=8 + n)

    def load(name):
        a, b = header[name]["data_offsets"]
        raw = torch.from_numpy(np.array(data[a:b]).view(np.int16)).cuda()
        return raw.view(torch.bfloat16).reshape(header[name]["shape"]).double()

    with open(os.path.join(directory, "config-mlx.json")) as f:
        freqs = json.load(f)["plamo_rope_inv_freq"]
    embed = load("model.embed_tokens.weight")
    rows = [embed[torch.tensor(t, device="cuda")] for t in tokens]
    del embed
    for i in range(LAYERS):
        p, full = f"model.layers.layers.{i}.", i % 8 == 7
        w = {s: load(p + s + ".weight") for s in (
            "mixer.qkv_proj", "mixer.o_proj", "mixer.q_norm", "mixer.k_norm", "mlp.gate_up_proj", "mlp.down_proj",
            "pre_mixer_norm", "post_mixer_norm", "pre_mlp_norm", "post_mlp_norm")}
        f = torch.tensor(freqs["full" if full else "local"], dtype=torch.float64, device="cuda")
        scale = 1.5545177444479562 if full else 1.0
        for j, x in enumerate(rows):
            pos = torch.arange(len(x), device="cuda")
            angle = pos.double()[:, None] * f
            c, s = torch.cos(angle) * scale, torch.sin(angle) * scale
            y = (_rms(x) * (w["pre_mixer_norm"] + 1.0)) @ w["mixer.qkv_proj"].T
            q = _rms(y[:, :HEADS * DIM].reshape(-1, HEADS, DIM)) * (w["mixer.q_norm"] + 1.0)
            k = _rms(y[:, HEADS * DIM:17 * DIM]) * (w["mixer.k_norm"] + 1.0)
            a = _softmax_pv(_rotate(q, c[:, None], s[:, None]), _rotate(k, c, s), y[:, 17 * DIM:],
                            _visible(pos, 0, len(x), full))
            x = x + _rms(a @ w["mixer.o_proj"].T) * (w["post_mixer_norm"] + 0.2)
            u = (_rms(x) * (w["pre_mlp_norm"] + 1.0)) @ w["mlp.gate_up_proj"].T
            a = torch.nn.functional.silu(u[:, :INTER]) * u[:, INTER:]
            rows[j] = x + _rms(a @ w["mlp.down_proj"].T) * (w["post_mlp_norm"] + 5.0 ** -1.5)
    last = torch.stack([x[-1] for x in rows])
    hidden = _rms(last) * (load("model.norm.weight") + 1.0)
    return hidden @ load("lm_head.weight").T, hidden


def exact(case, seed):
    kind = case["kind"]
    if kind == "sequence":
        logits, hidden = _exact_model([_tokens(seed, case["prompt"] + case["steps"])])
        return {"logits": logits[0], "hidden": hidden[0]}
    if kind == "lanes":
        logits, hidden = _exact_model([_tokens(1000 * seed + i, n + case["steps"])
                                       for i, n in enumerate(_lane_lengths(case))])
        return {"logits": list(logits), "hidden": list(hidden)}
    s = _inputs(case, seed)
    if kind == "attend":
        return _exact_attend(case, s)
    if kind == "step":
        return _exact_step(case, s)
    x, got = s["x"].double(), []
    for w in s["w"]:
        y = torch.cat([x @ part.double().T for part in w.split(16384)], -1)
        got.append(torch.nn.functional.silu(y[:, :INTER]) * y[:, INTER:]
                   if kind == "gemm" and case["shape"] == "gate_up" else y)
    return got
