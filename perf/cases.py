"""The work whose speed is measured: what a program that runs Llama-3.2-1B
shaped GGUF models with this package has it do, through the public API
(sqhip.Llama3_2 / ModelContext and sqhip.ops).

Whole calls take prompts of 32 to 2048 tokens through `forward` and windows of
text through `score` (a batched prefill, then one decode step per token).
Operator calls are the ones a program with its own layer loop makes: the
quantized projections, attention, normalization.  Sizes are those of the 1B
model (width 2048, FFN 8192, 32 query and 8 KV heads of 64, vocabulary 128256)
and of the small models of the tests, with odd lengths between them.
"""
from __future__ import annotations

import math
import os
import sys
import tempfile

import numpy as np
import torch

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(REPO, "squirrel-rs_amd")
if PKG not in sys.path:
    sys.path.insert(0, PKG)

import sqhip  # noqa: E402
from sqhip import ops  # noqa: E402

DIM, FFN, HEADS, KV_HEADS, HEAD_DIM, VOCAB = 2048, 8192, 32, 8, 64, 128256
KV_DIM = KV_HEADS * HEAD_DIM
EPS = 1e-5
WTYPE = {"Q8_0": sqhip.SQ_Q8_0, "Q4_0": sqhip.SQ_Q4_0}
BLOCK_BYTES = {"Q8_0": 34, "Q4_0": 18}  # one block of 32 weights


def listed():
    return [
        # one token through an attention output projection: the smallest call
        # of a program that decodes operator by operator
        {"name": "linear_q8_1_row", "op": "linear", "wtype": "Q8_0", "m": 1, "k": DIM, "rows": DIM},
        # the stacked gate and up rows for a prompt of odd length
        {"name": "linear_q4_131_rows", "op": "linear", "wtype": "Q4_0", "m": 131, "k": DIM, "rows": 2 * FFN},
        # the FFN down projection of a 2048-token prompt: the longest K
        {"name": "linear_q8_2048_rows", "op": "linear", "wtype": "Q8_0", "m": 2048, "k": FFN, "rows": DIM},
        # q, k and v of a short chat turn, its activations quantized once
        {"name": "qkv_q8_32_rows", "op": "linear_shared", "wtype": "Q8_0", "m": 32, "k": DIM, "rows": DIM,
         "rows2": KV_DIM, "rows3": KV_DIM},
        # one decoded token's attention over a long context
        {"name": "sdpa_decode_4096", "op": "sdpa", "seq_q": 1, "seq_k": 4096, "heads": HEADS, "kv_heads": KV_HEADS},
        # a prompt's causal attention
        {"name": "sdpa_prompt_1500", "op": "sdpa", "seq_q": 1500, "seq_k": 1500, "heads": HEADS,
         "kv_heads": KV_HEADS},
        # the norm before each projection, a few hundred prompt rows
        {"name": "rms_norm_500_rows", "op": "rms_norm", "m": 500, "dim": DIM},
        # prompts to logits, four of the 1B model's layers (every layer runs
        # the same kernels at the same widths): a chat turn, a paragraph of
        # odd length, a document
        {"name": "prompt_q8_32", "op": "prompt", "wtype": "Q8_0", "layers": 4, "n": 32},
        {"name": "prompt_q4_301", "op": "prompt", "wtype": "Q4_0", "layers": 4, "n": 301},
        {"name": "prompt_q8_2048", "op": "prompt", "wtype": "Q8_0", "layers": 4, "n": 2048},
        # one window of the perplexity harness at its default sizes on the
        # whole 1B model: a 256-token prefill, then 255 decode steps
        {"name": "score_q8_512", "op": "score", "wtype": "Q8_0", "layers": 16, "n": 512, "burn": 256},
        # decode behind a 4096-token context, the whole 1B model
        {"name": "score_q8_long", "op": "score", "wtype": "Q8_0", "layers": 16, "n": 4096 + 128, "burn": 4096},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    op = rng.choice(["linear", "linear", "linear_shared", "sdpa", "sdpa", "rms_norm", "prompt", "prompt", "prompt",
                     "score", "score"])
    wtype = rng.choice(["Q8_0", "Q4_0"])
    if op in ("linear", "linear_shared"):
        m = _log_int(rng, 1, 2048)
        if op == "linear":
            # a projection of the model, or any shape of its range
            k, rows = rng.choice([(DIM, DIM), (DIM, KV_DIM), (DIM, FFN), (FFN, DIM), (DIM, DIM + 2 * KV_DIM),
                                  (32 * _log_int(rng, 4, 256), _log_int(rng, 64, 8192))])
            return {"op": op, "wtype": wtype, "m": m, "k": k, "rows": rows}
        rows, rows2, rows3 = rng.choice([(DIM, KV_DIM, KV_DIM), (512, 128, 128), (FFN, FFN, 0), (1024, 1024, 0)])
        return {"op": op, "wtype": wtype, "m": m, "k": rng.choice([DIM, DIM, 512]), "rows": rows, "rows2": rows2,
                "rows3": rows3}
    if op == "sdpa":
        heads, kv = rng.choice([(HEADS, KV_HEADS), (HEADS, KV_HEADS), (8, 2), (4, 2), (16, 16)])
        # one token behind a context, a whole prompt, a further turn of a chat
        kind = rng.choice(["decode", "prompt", "turn"])
        if kind == "decode":
            seq_q, seq_k = 1, _log_int(rng, 16, 8192)
        elif kind == "prompt":
            seq_q = seq_k = _log_int(rng, 2, 2048)
        else:
            seq_q = _log_int(rng, 2, 512)
            seq_k = seq_q + _log_int(rng, 16, 3584)
        return {"op": op, "seq_q": seq_q, "seq_k": seq_k, "heads": heads, "kv_heads": kv}
    if op == "rms_norm":
        return {"op": op, "m": _log_int(rng, 1, 4096), "dim": rng.choice([DIM, DIM, 512, 256, 1000])}
    if op == "prompt":
        return {"op": op, "wtype": wtype, "layers": 4, "n": _log_int(rng, 2, 2048)}
    if rng.random() < 0.5:
        n = _log_int(rng, 40, 512)
        burn = max(1, n // 2)
    else:
        burn = _log_int(rng, 256, 4096)
        n = burn + _log_int(rng, 16, 128)
    return {"op": "score", "wtype": wtype, "layers": 16, "n": n, "burn": burn}


class Buffer:
    """A torch tensor's memory as sqhip.ops takes it."""

    def __init__(self, t):
        self.ptr, self.shape, self.size = t.data_ptr(), tuple(t.shape), t.numel()


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _normal(g, *shape, std=1.0):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32) * std


def _weight_blocks(g, wtype, rows, k):
    """rows x k weights ~ N(0, 0.02) as GGUF blocks (host memory)."""
    w = _normal(g, rows, k, std=0.02).view(rows * k // 32, 32)
    if wtype == "Q8_0":
        d = (w.abs().amax(1) / 127.0).half()
        q = torch.clamp(torch.round(w / d.float()[:, None]), -127, 127).to(torch.int8)
        out = np.zeros(len(w), ops.BLOCK_Q8_0)
    else:
        top = torch.gather(w, 1, w.abs().argmax(1, keepdim=True))[:, 0]
        d = (top / -8.0).half()
        q = torch.clamp(torch.round(w / d.float()[:, None]) + 8, 0, 15).to(torch.uint8)
        q = q[:, :16] | (q[:, 16:] << 4)
        out = np.zeros(len(w), ops.BLOCK_Q4_0)
    out["d"] = d.cpu().numpy().view(np.uint16)
    out["qs"] = q.cpu().numpy()
    return out


_models = {}


def _model(wtype, layers):
    """The random-init 1B model with `layers` layers, loaded once as a program does."""
    key = (wtype, layers)
    if key not in _models:
        with tempfile.TemporaryDirectory() as d:
            path = sqhip.write_synthetic_gguf(os.path.join(d, "model.gguf"), wtype, seed=0, n_layers=layers)
            _models[key] = sqhip.Llama3_2(path)
    return _models[key]


def _rows_of(case):
    return [r for r in (case["rows"], case.get("rows2", 0), case.get("rows3", 0)) if r]


def prepare(case, seed):
    op = case["op"]
    state = {"op": op}
    if op in ("linear", "linear_shared"):
        g = _generator(seed)
        m, k = case["m"], case["k"]
        state["x"] = _normal(g, m, k)
        state["weights"] = [ops.Weight(WTYPE[case["wtype"]], _weight_blocks(g, case["wtype"], r, k), r, k)
                            for r in _rows_of(case)]
        state["outs"] = [torch.empty(m, r, device="cuda") for r in _rows_of(case)]
    elif op == "sdpa":
        g = _generator(seed)
        state["heads"], state["kv_heads"] = case["heads"], case["kv_heads"]
        state["q"] = _normal(g, case["seq_q"], case["heads"] * HEAD_DIM)
        state["k"] = _normal(g, case["seq_k"], case["kv_heads"] * HEAD_DIM)
        state["v"] = _normal(g, case["seq_k"], case["kv_heads"] * HEAD_DIM)
        state["out"] = torch.empty_like(state["q"])
    elif op == "rms_norm":
        g = _generator(seed)
        state["x"] = _normal(g, case["m"], case["dim"])
        state["w"] = 1.0 + _normal(g, case["dim"], std=0.1)
        state["out"] = torch.empty_like(state["x"])
    else:
        model = _model(case["wtype"], case["layers"])
        state["ids"] = np.random.default_rng(seed).integers(0, VOCAB, case["n"]).astype(np.uint32)
        state["ctx"] = model.new_context(case["n"])
        state["burn"] = case.get("burn", 0)
    return state


def run(state):
    op = state["op"]
    if op == "linear":
        ops.linear(Buffer(state["x"]), state["weights"][0], Buffer(state["outs"][0]))
        return state["outs"][0]
    if op == "linear_shared":
        ops.linear_shared(Buffer(state["x"]), state["weights"], [Buffer(o) for o in state["outs"]])
        return state["outs"]
    if op == "sdpa":
        ops.sdpa_cached(Buffer(state["q"]), Buffer(state["k"]), Buffer(state["v"]), Buffer(state["out"]),
                        state["heads"], state["kv_heads"], HEAD_DIM)
        return state["out"]
    if op == "rms_norm":
        ops.rms_norm(Buffer(state["x"]), Buffer(state["w"]), Buffer(state["out"]), EPS)
        return state["out"]
    ctx = state["ctx"]
    if op == "prompt":
        ctx.reset_cache()
        ctx.forward(state["ids"])
        return ctx.logits()
    return ctx.score(state["ids"], state["burn"])


def _layer_params():
    return DIM * (DIM + 2 * KV_DIM) + DIM * DIM + 3 * DIM * FFN


def _pass_work(wtype, layers, n, past):
    """One forward of n tokens behind `past` cached positions: every matrix
    once, the norms, n embedding rows, the cached K and V read and n rows of
    each written, one row of logits written."""
    per_weight = BLOCK_BYTES[wtype] / 32
    pairs = n * past + n * (n + 1) / 2
    nbytes = ((layers * _layer_params() + VOCAB * DIM + n * DIM) * per_weight + (2 * layers + 1) * DIM * 4
              + 2 * layers * KV_DIM * 4 * (past + n) + VOCAB * 4)
    flops = 2.0 * n * layers * _layer_params() + 2.0 * VOCAB * DIM + 4.0 * layers * pairs * HEADS * HEAD_DIM
    return nbytes, flops


def work(case):
    op = case["op"]
    if op in ("linear", "linear_shared"):
        m, k, rows = case["m"], case["k"], sum(_rows_of(case))
        return {"bytes": 4 * m * k + rows * k * BLOCK_BYTES[case["wtype"]] / 32 + 4 * m * rows,
                "flops": 2.0 * m * k * rows}
    if op == "sdpa":
        sq, sk, h, kv = case["seq_q"], case["seq_k"], case["heads"], case["kv_heads"]
        pairs = sq * (sk - sq) + sq * (sq + 1) / 2
        return {"bytes": 4 * HEAD_DIM * (2 * sq * h + 2 * sk * kv), "flops": 4.0 * HEAD_DIM * h * pairs}
    if op == "rms_norm":
        n = case["m"] * case["dim"]
        return {"bytes": 4 * (2 * n + case["dim"]), "flops": 4.0 * n}
    if op == "prompt":
        nbytes, flops = _pass_work(case["wtype"], case["layers"], case["n"], 0)
        return {"bytes": nbytes, "flops": flops}
    nbytes, flops = _pass_work(case["wtype"], case["layers"], case["burn"], 0)
    for past in range(case["burn"], case["n"] - 1):
        b, f = _pass_work(case["wtype"], case["layers"], 1, past)
        nbytes, flops = nbytes + b, flops + f
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """Single operators sum f32 terms: about four times their distance from
    the 64-bit result.  Whole calls quantize their activations to 8 bits at
    every site, so a last-bit difference in one layer moves quantized values
    by whole steps downstream: two correct orders of summation (the f32 and
    the split-f16 attention) leave the logits of four layers 1.1e-2 to 1.7e-2
    apart, and a window's log-probabilities (on the two decode paths, too) up
    to 3.9e-3."""
    op = case["op"]
    if op in ("linear", "linear_shared"):
        return {"rel": 2e-6, "max": 1e-4}
    if op == "sdpa":
        return {"rel": 2e-6, "max": 2e-4}
    if op == "rms_norm":
        return {"rel": 5e-7, "max": 4e-6}
    if op == "prompt":
        return {"rel": 0.03, "max": 0.3}
    return {"rel": 0.016, "max": 0.064}


def _exact_linear(x, wtype, rows, blocks):
    """x quantized to Q8_0 as the format defines it, then 64-bit sums."""
    m, k = x.shape
    xb = x.cpu().numpy().reshape(m * k // 32, 32)
    scale = np.abs(xb).max(1) / np.float32(127.0)
    with np.errstate(divide="ignore"):
        inv = np.where(scale > 0, np.float32(1.0) / scale, np.float32(0.0)).astype(np.float32)
    v = xb * inv[:, None]
    q = np.clip(np.trunc(v + np.copysign(np.float32(0.5), v)), -127, 127)
    # (v + 0.5 rounds up to 1 for the value just below a half)
    q = np.where(np.abs(v) < 0.5, 0.0, q)
    a = (q.astype(np.float64) * scale.astype(np.float16).astype(np.float64)[:, None]).reshape(m, k)
    d = blocks["d"].view(np.float16).astype(np.float64)[:, None]
    qs = blocks["qs"]
    if wtype == "Q4_0":
        qs = np.concatenate([qs & 15, qs >> 4], axis=1).astype(np.int8) - np.int8(8)
    w = torch.from_numpy(qs.astype(np.float64) * d).view(rows, k).cuda()
    return torch.from_numpy(a).cuda() @ w.t().contiguous()


def exact(case, seed):
    op = case["op"]
    g = _generator(seed)
    if op in ("linear", "linear_shared"):
        x = _normal(g, case["m"], case["k"])
        got = [_exact_linear(x, case["wtype"], r, _weight_blocks(g, case["wtype"], r, case["k"]))
               for r in _rows_of(case)]
        return got if op == "linear_shared" else got[0]
    if op == "sdpa":
        sq, sk, h, kv = case["seq_q"], case["seq_k"], case["heads"], case["kv_heads"]
        q = _normal(g, sq, h * HEAD_DIM).double().view(sq, h, HEAD_DIM)
        k = _normal(g, sk, kv * HEAD_DIM).double().view(sk, kv, HEAD_DIM)
        v = _normal(g, sk, kv * HEAD_DIM).double().view(sk, kv, HEAD_DIM)
        hidden = torch.arange(sk, device="cuda")[None, :] > torch.arange(sq, device="cuda")[:, None] + (sk - sq)
        out = torch.empty_like(q)
        for i in range(h):
            j = i // (h // kv)
            s = (q[:, i].contiguous() @ k[:, j].t().contiguous()) / math.sqrt(HEAD_DIM)
            p = torch.softmax(s.masked_fill(hidden, -math.inf), dim=1)
            out[:, i] = p @ v[:, j].contiguous()
        return out.view(sq, h * HEAD_DIM)
    if op == "rms_norm":
        x = _normal(g, case["m"], case["dim"]).double()
        w = (1.0 + _normal(g, case["dim"], std=0.1)).double()
        return x * w / torch.sqrt((x * x).mean(1, keepdim=True) + EPS)
    # Whole calls have no 64-bit value to be near: the 8-bit quantization of
    # the activations turns last-bit differences into whole steps.
    return None
