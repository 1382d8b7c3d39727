"""The calls whose speed this repository is measured by, at sizes that its users meet.

Model widths are the 4B-class hybrid decoder's (EngineConfig's defaults: hidden 2560, ffn 9216, 16 query / 4 kv
heads of 256, 32 delta-net value heads of 128 on 16 key heads, vocab 151936).  The kinds of case:

step        one decode step of the whole 32-block decoder as a serving loop that picks tokens itself makes it: the
            tokens and positions go in, one graph replay, the logits are there when the engine's stream is drained.
prompt      a new batch of prompts through a delta-net block, an attention block and the vocabulary projection: reset,
            chunked prefill of every prompt, the last tokens' logits.  Two blocks, because 32 blocks of random weights
            and int8 activations amplify a last-bit difference past any useful tolerance.
ffn         the SwiGLU block of a prompt chunk through the C ABI's prefill calls, the residual added by the last GEMM.
chunk_attn  causal attention of a prompt chunk over an INT8 cache that holds the earlier chunks.
scan        the gated delta rule over a prompt chunk, the heads' state updated in place.
attn        INT8 decode attention of a batch of sequences, one query token each.
vocab       the reference-signature arithmetic (GGUF bytes in place, fp32 activations): one token's projection.
"""
from __future__ import annotations

import math
import sys
from pathlib import Path

import numpy as np
import torch

_PKG = str(Path(__file__).resolve().parents[1] / "echo-core_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from echohip.engine import B_LOGITS, Engine, EngineConfig  # noqa: E402
from echohip.lib import Q4_K, Q8_0, load  # noqa: E402

HIDDEN, FFN, VOCAB = 2560, 9216, 151936
HEAD_DIM = 256
KEY_HEADS, VALUE_HEADS, STATE_DIM = 16, 32, 128
FORMATS = {"q8_0": Q8_0, "q4_K": Q4_K}


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # one user's chat, a few hundred tokens in: the smallest step, where launches count most
        {"name": "step_1", "kind": "step", "batch": 1, "min_ctx": 500, "max_ctx": 500, "pieces": 2},
        # a serving batch of ragged conversations
        {"name": "step_8", "kind": "step", "batch": 8, "min_ctx": 128, "max_ctx": 4096, "pieces": 2},
        # one short question: a prompt below a chunk
        {"name": "prompt_1x130", "kind": "prompt", "prompts": 1, "min_len": 130, "max_len": 130},
        # a batch of ragged prompts, several chunks each
        {"name": "prompt_4", "kind": "prompt", "prompts": 4, "min_len": 300, "max_len": 4096},
        # a short prompt's rows, a ragged pass's, and two whole chunks in one pass
        {"name": "ffn_q8_40", "kind": "ffn", "fmt": "q8_0", "rows": 40, "hidden": HIDDEN, "ffn": FFN},
        {"name": "ffn_q8_1024", "kind": "ffn", "fmt": "q8_0", "rows": 1024, "hidden": HIDDEN, "ffn": FFN},
        {"name": "ffn_q4_387", "kind": "ffn", "fmt": "q4_K", "rows": 387, "hidden": HIDDEN, "ffn": FFN},
        # the eighth chunk of a 4096-token prompt
        {"name": "chunk_attn_512", "kind": "chunk_attn", "rows": 512, "pos0": 3584, "heads": 16, "kv": 4},
        # a prompt of two chunks' length in one call
        {"name": "scan_1000", "kind": "scan", "rows": 1000, "seqs": 1},
        # one long document, and a ragged batch
        {"name": "attn_32768", "kind": "attn", "seqs": 1, "min_ctx": 32768, "max_ctx": 32768, "heads": 16, "kv": 4},
        {"name": "attn_8", "kind": "attn", "seqs": 8, "min_ctx": 128, "max_ctx": 4096, "heads": 16, "kv": 4},
        # the vocabulary projection of a program built against the reference's headers
        {"name": "vocab_q4", "kind": "vocab", "fmt": "q4_K", "rows": VOCAB, "cols": HIDDEN},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("step", "prompt", "ffn", "ffn", "ffn", "chunk_attn", "chunk_attn", "scan", "attn", "vocab"))
    if kind == "step":
        lo = _log(rng, 64, 2048)
        return {"kind": kind, "batch": rng.randint(1, 8), "min_ctx": lo, "max_ctx": _log(rng, lo, 4096),
                "pieces": rng.choice((1, 2, 2))}
    if kind == "prompt":
        lo = _log(rng, 16, 1024)
        return {"kind": kind, "prompts": rng.randint(1, 4), "min_len": lo, "max_len": _log(rng, lo, 3000)}
    if kind == "ffn":
        hidden, ffn = rng.choice(((2560, 9216), (2560, 9216), (2048, 6144), (1024, 4096)))
        return {"kind": kind, "fmt": rng.choice(("q8_0", "q8_0", "q4_K")), "rows": _log(rng, 17, 1024),
                "hidden": hidden, "ffn": ffn}
    if kind == "chunk_attn":
        heads, kv = rng.choice(((16, 4), (16, 4), (16, 8), (8, 8)))
        return {"kind": kind, "rows": _log(rng, 17, 512), "pos0": rng.randint(0, 3584), "heads": heads, "kv": kv}
    if kind == "scan":
        return {"kind": kind, "rows": _log(rng, 128, 1024), "seqs": rng.randint(1, 2)}
    if kind == "attn":
        heads, kv = rng.choice(((16, 4), (16, 4), (16, 8), (8, 8)))
        lo = _log(rng, 64, 2048)
        return {"kind": kind, "seqs": rng.randint(1, 16), "min_ctx": lo, "max_ctx": _log(rng, lo, 4096),
                "heads": heads, "kv": kv}
    return {"kind": kind, "fmt": rng.choice(("q8_0", "q4_K")), "rows": _log(rng, 1024, 100000),
            "cols": rng.choice((2560, 2560, 4096, 9216))}


def _lengths(n, lo, hi):
    """n lengths from lo to hi, evenly spread over the range: the same for every seed."""
    return [lo + (hi - lo) * i // max(1, n - 1) for i in range(n)]


# ---------------------------------------------------------------- inputs
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 7919 + 17)


def _randn(g, *shape):
    return torch.randn(shape, generator=g, device="cuda")


def _gguf(fmt, rows, cols, g):
    """GGUF bytes [rows][blocks][bytes] of a weight matrix of about 0.02 standard deviation."""
    if fmt == Q8_0:
        n = cols // 32
        out = torch.empty((rows, n, 34), dtype=torch.uint8, device="cuda")
        d = (_randn(g, rows, n).abs() * (0.02 / 73.0)).half()
        out[:, :, :2] = d.view(torch.uint8).view(rows, n, 2)
        q = torch.randint(-127, 128, (rows, n, 32), generator=g, device="cuda", dtype=torch.int8)
        out[:, :, 2:] = q.view(torch.uint8)
        return out
    n = cols // 256
    out = torch.empty((rows, n, 144), dtype=torch.uint8, device="cuda")
    d = (0.5 + torch.rand((rows, n, 1), generator=g, device="cuda")) * (0.02 / 150.0)
    out[:, :, :2] = d.half().view(torch.uint8)
    out[:, :, 2:4] = (7.5 * d).half().view(torch.uint8)
    # six-bit scales and mins and the nibbles are uniform, as their packed bytes then are
    out[:, :, 4:] = torch.randint(0, 256, (rows, n, 140), generator=g, device="cuda", dtype=torch.int32).to(torch.uint8)
    return out


def _tiled(hip, fmt, rows, cols, g):
    raw = _gguf(fmt, rows, cols, g)
    tiled = torch.empty(hip.tiled_bytes(fmt, rows, cols), dtype=torch.uint8, device="cuda")
    hip.repack(fmt, raw, tiled, rows, cols)
    return tiled


def _cache(g, positions, kv):
    """INT8 keys and values of N(0, 1) rows with their scales, one per (position, kv head)."""
    parts = []
    for _ in range(2):
        x = _randn(g, positions, kv, HEAD_DIM)
        d = x.abs().amax(-1) / 127.0
        parts.append(((x / d[:, :, None]).round().to(torch.int8), d))
    (keys, ks), (vals, vs) = parts
    return keys, vals, ks, vs


class _Device:
    """A buffer of the engine as a torch tensor; the tensor keeps the engine."""

    def __init__(self, engine, which, shape):
        at, _ = engine.buffer(which)
        self.engine = engine
        self.__cuda_array_interface__ = {"shape": shape, "typestr": "<f4", "data": (at, False), "version": 3,
                                         "strides": None}


def _logits(engine):
    return torch.as_tensor(_Device(engine, B_LOGITS, (engine.cfg.max_batch, engine.cfg.vocab)), device="cuda")


def prepare(case, seed):
    kind = case["kind"]
    if kind == "step":
        return _prepare_step(case, seed)
    if kind == "prompt":
        lens = _lengths(case["prompts"], case["min_len"], case["max_len"])
        engine = Engine(EngineConfig(n_layers=2, attn_interval=2, max_batch=len(lens), max_ctx=max(lens) + 64))
        engine.init_random(seed)
        rng = np.random.default_rng(seed)
        return {"kind": kind, "engine": engine, "logits": _logits(engine),
                "jobs": [(i, rng.integers(0, VOCAB, n).astype(np.int32), 0) for i, n in enumerate(lens)]}
    hip, g = load(), _gen(seed)
    hip.device_init(torch.cuda.current_device())
    s = dict(case, hip=hip)
    if kind == "ffn":
        fmt, m, h, f = FORMATS[case["fmt"]], case["rows"], case["hidden"], case["ffn"]
        s.update(fmt=fmt, w=1.0 + 0.1 * _randn(g, h), x=_randn(g, m, h), gate_up=_tiled(hip, fmt, 2 * f, h, g),
                 down=_tiled(hip, fmt, h, f, g), gu=torch.empty((m, 2 * f), device="cuda"),
                 y=torch.empty((m, h), device="cuda"), n=torch.empty((m, h), device="cuda"),
                 p=torch.empty((m, f), device="cuda"),
                 act_h=torch.empty(hip.gemm_act_bytes(fmt, m, h), dtype=torch.uint8, device="cuda"),
                 act_f=torch.empty(hip.gemm_act_bytes(fmt, m, f), dtype=torch.uint8, device="cuda"))
    elif kind == "chunk_attn":
        m, heads = case["rows"], case["heads"]
        s["end"] = case["pos0"] + m
        s["q"] = _randn(g, m, heads * HEAD_DIM)
        s["cache"] = _cache(g, s["end"], case["kv"])
        s["out"] = torch.empty_like(s["q"])
        s["ws"] = torch.empty(max(16, hip.attn_prefill_ws_bytes(m, heads, s["end"])), dtype=torch.uint8, device="cuda")
    elif kind == "scan":
        m, n = case["rows"], case["seqs"]
        unit = torch.nn.functional.normalize
        s.update(state=0.02 * _randn(g, n, VALUE_HEADS, STATE_DIM, STATE_DIM),
                 q=unit(_randn(g, m, n, KEY_HEADS, STATE_DIM), dim=-1),
                 k=unit(_randn(g, m, n, KEY_HEADS, STATE_DIM), dim=-1), v=_randn(g, m, n, VALUE_HEADS, STATE_DIM),
                 decay=torch.sigmoid(2 + 0.5 * _randn(g, m, n, VALUE_HEADS)),
                 beta=torch.sigmoid(_randn(g, m, n, VALUE_HEADS)),
                 out=torch.empty((m, n, VALUE_HEADS, STATE_DIM), device="cuda"),
                 ws=torch.empty(hip.deltanet_chunked_ws_bytes(m, n, VALUE_HEADS), dtype=torch.uint8, device="cuda"))
    elif kind == "attn":
        n, heads, kv = case["seqs"], case["heads"], case["kv"]
        s["q"] = _randn(g, n, heads * HEAD_DIM)
        s["cache"] = _cache(g, n * case["max_ctx"], kv)
        s["ctx"] = torch.tensor(_lengths(n, case["min_ctx"], case["max_ctx"]), dtype=torch.int32, device="cuda")
        s["out"] = torch.empty_like(s["q"])
        s["ws"] = torch.empty(hip.attn_ws_bytes(n, heads, HEAD_DIM, case["max_ctx"]), dtype=torch.uint8, device="cuda")
    else:
        fmt = FORMATS[case["fmt"]]
        s.update(fmt=fmt, weights=_gguf(fmt, case["rows"], case["cols"], g), x=_randn(g, case["cols"]),
                 y=torch.empty(case["rows"], device="cuda"))
    return s


STEPS = 64  # positions that a step state's passes walk over before they start again


def _prepare_step(case, seed):
    lens = _lengths(case["batch"], case["min_ctx"], case["max_ctx"])
    engine = Engine(EngineConfig(max_batch=len(lens), max_ctx=max(lens) + STEPS + 1))
    engine.init_random(seed)
    engine.set_act_pieces(case["pieces"])
    rng = np.random.default_rng(seed)
    engine.prefill_batch([(i, rng.integers(0, VOCAB, n).astype(np.int32), 0) for i, n in enumerate(lens)])
    return {"kind": "step", "engine": engine, "logits": _logits(engine), "lens": np.array(lens, np.int32),
            "tokens": rng.integers(0, VOCAB, (STEPS, len(lens))).astype(np.int32), "at": 0}


# ---------------------------------------------------------------- one pass
def run(s):
    kind = s["kind"]
    if kind == "step":
        i = s["at"] % STEPS
        s["at"] += 1
        s["engine"].set_inputs(s["tokens"][i], s["lens"] + i)
        s["engine"].step()
        s["engine"].sync()  # the program reads the logits now, on its own stream
        return s["logits"]
    if kind == "prompt":
        s["engine"].reset()
        s["engine"].prefill_batch(s["jobs"])
        return s["logits"]
    hip = s["hip"]
    if kind == "ffn":
        fmt, m, h, f = s["fmt"], s["rows"], s["hidden"], s["ffn"]
        if fmt == Q8_0:
            hip.rmsnorm_rows_gemm_act(s["x"], s["w"], s["act_h"], m, h)
        else:
            hip.rmsnorm_rows(s["x"], s["w"], s["n"], m, h)
            hip.gemm_quantize_act(fmt, s["n"], s["act_h"], m, h)
        hip.gemm(fmt, s["gate_up"], s["act_h"], s["gu"], m, 2 * f, h)
        if fmt == Q8_0:
            hip.swiglu_rows_gemm_act(s["gu"], s["act_f"], m, f)
        else:
            hip.swiglu_rows(s["gu"], s["p"], m, f)
            hip.gemm_quantize_act(fmt, s["p"], s["act_f"], m, f)
        s["y"].copy_(s["x"])
        hip.gemm(fmt, s["down"], s["act_f"], s["y"], m, h, f, accumulate=True)
        return [s["gu"], s["y"]]
    if kind == "chunk_attn":
        hip.attn_prefill(s["q"], *s["cache"], s["out"], s["rows"], s["pos0"], s["heads"], s["kv"], HEAD_DIM, s["end"],
                         ws=s["ws"])
        return s["out"]
    if kind == "scan":
        hip.deltanet_chunked(s["state"], s["q"], s["k"], s["v"], s["decay"], s["beta"], s["out"], s["rows"], s["seqs"],
                             VALUE_HEADS, KEY_HEADS, STATE_DIM, STATE_DIM, s["ws"])
        return [s["out"], s["state"]]
    if kind == "attn":
        hip.attn_decode(s["q"], *s["cache"], s["out"], s["ctx"], s["seqs"], s["max_ctx"] * s["kv"] * HEAD_DIM,
                        s["heads"], s["kv"], HEAD_DIM, s["max_ctx"], s["ws"])
        return s["out"]
    s["y"].zero_()  # the call adds to y, as the reference's does
    hip.matvec_gguf_f32(s["fmt"], s["weights"], s["x"], s["y"], s["rows"], s["cols"])
    return s["y"]


# ---------------------------------------------------------------- what a pass cannot do without
def _row_bytes(fmt, cols):
    return cols // 32 * 34 if fmt == Q8_0 else cols // 256 * 144


def _model(delta, attn):
    """Matrix elements of a stack of so many delta-net and attention blocks, without the head."""
    cfg = EngineConfig()
    n = (delta + attn) * 3 * HIDDEN * FFN + attn * (cfg.nin_attn * HIDDEN + HIDDEN * cfg.n_heads * cfg.head_dim)
    return n + delta * (cfg.nin_delta * HIDDEN + HIDDEN * cfg.ssm_inner)


def work(case):
    kind = case["kind"]
    state = VALUE_HEADS * STATE_DIM * STATE_DIM
    if kind == "step":
        lens = _lengths(case["batch"], case["min_ctx"], case["max_ctx"])
        b, delta, attn = len(lens), 24, 8
        n = _model(delta, attn) + VOCAB * HIDDEN
        moved = n // 32 * 34 + delta * b * 2 * 4 * state + attn * sum(lens) * 4 * (2 * HEAD_DIM + 8) + 4 * b * VOCAB
        return {"bytes": moved, "flops": 2 * n * b + delta * b * 7 * state + attn * sum(lens) * 4 * 16 * HEAD_DIM}
    if kind == "prompt":
        lens = _lengths(case["prompts"], case["min_len"], case["max_len"])
        t, n, head = sum(lens), _model(1, 1), VOCAB * HIDDEN
        return {"bytes": (n + head) // 32 * 34 + 4 * len(lens) * VOCAB,
                "flops": 2 * n * t + 2 * head * len(lens) + t * 7 * state
                + sum(x * x / 2 for x in lens) * 4 * 16 * HEAD_DIM}
    if kind == "ffn":
        fmt, m, h, f = FORMATS[case["fmt"]], case["rows"], case["hidden"], case["ffn"]
        return {"bytes": 2 * f * _row_bytes(fmt, h) + h * _row_bytes(fmt, f) + 4 * m * (2 * h + 2 * f),
                "flops": 2 * m * 3 * h * f}
    if kind == "chunk_attn":
        m, p, heads, kv = case["rows"], case["pos0"], case["heads"], case["kv"]
        return {"bytes": (p + m) * kv * (2 * HEAD_DIM + 8) + 8 * m * heads * HEAD_DIM,
                "flops": 4 * HEAD_DIM * heads * (m * p + m * (m + 1) / 2)}
    if kind == "scan":
        m, n = case["rows"], case["seqs"]
        row = 2 * KEY_HEADS * STATE_DIM + 2 * VALUE_HEADS * STATE_DIM + 2 * VALUE_HEADS
        return {"bytes": 4 * n * (m * row + 2 * state), "flops": 7 * state * m * n}
    if kind == "attn":
        lens, heads, kv = _lengths(case["seqs"], case["min_ctx"], case["max_ctx"]), case["heads"], case["kv"]
        return {"bytes": sum(lens) * kv * (2 * HEAD_DIM + 8) + 8 * len(lens) * heads * HEAD_DIM,
                "flops": 4 * HEAD_DIM * heads * sum(lens)}
    rows, cols = case["rows"], case["cols"]
    return {"bytes": rows * _row_bytes(FORMATS[case["fmt"]], cols) + 4 * (rows + cols), "flops": 2 * rows * cols}


def tolerance(case):
    # Each is about four times what was measured between two orders of the same arithmetic.
    return {
        "step": {"rel": 0.03, "max": 0.3},
        "prompt": {"rel": 0.03, "max": 0.3},
        "ffn": {"rel": 1e-3, "max": 0.05},
        "chunk_attn": {"rel": 4e-6},
        "scan": {"rel": 4e-6},
        "attn": {"rel": 2e-6},
        "vocab": {"rel": 1e-6},
    }[case["kind"]]


# ---------------------------------------------------------------- the same in 64 bits
def _dequant(fmt, raw):
    """float64 [rows][cols] of GGUF bytes [rows][blocks][bytes], in the reference's element order."""
    rows, n = raw.shape[:2]
    half = lambda b: b.contiguous().view(torch.float16).double()  # noqa: E731
    if fmt == Q8_0:
        return (half(raw[:, :, :2]) * raw[:, :, 2:].contiguous().view(torch.int8).double()).reshape(rows, n * 32)
    s = raw[:, :, 4:16].int()
    lo, hi = s[:, :, :4], s[:, :, 4:8]
    sc = torch.cat((lo & 63, (s[:, :, 8:] & 15) | ((lo >> 6) << 4)), -1).double()
    mn = torch.cat((hi & 63, (s[:, :, 8:] >> 4) | ((hi >> 6) << 4)), -1).double()
    nib = raw[:, :, 16:].reshape(rows, n, 8, 16)
    sub = torch.stack((nib & 15, nib >> 4), -2).double()  # [rows][n][sub-block][run][16]
    w = sub * (half(raw[:, :, :2]) * sc)[..., None, None] - (half(raw[:, :, 2:4]) * mn)[..., None, None]
    # sub-block 2h + j: its run r is elements 64h + 32r + 16j .. +15
    return w.reshape(rows, n, 4, 2, 2, 16).transpose(3, 4).reshape(rows, n * 256)


def _quantized(fmt, x):
    """float64 values of the rows after the reference's per-32 int8 quantizer (Q4_K: per sub-block), whose own
    arithmetic is 32-bit."""
    m, k = x.shape
    if fmt == Q8_0:
        b = x.float().view(m, k // 32, 32)
    else:
        b = x.float().view(m, k // 64, 2, 2, 16).transpose(2, 3).reshape(m, k // 32, 32)
    amax = b.abs().amax(-1, keepdim=True)
    scale = torch.where(amax > 0, amax / 127.0, torch.ones_like(amax))
    q = (b * (1.0 / scale)).round().clamp(-128, 127).double() * scale.double()
    return (q if fmt == Q8_0 else q.view(m, k // 64, 2, 2, 16).transpose(2, 3)).reshape(m, k)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("step", "prompt"):
        return None  # a whole stack: every block's int8 activations round on the values before them
    g = _gen(seed)
    if kind == "ffn":
        fmt, m, h, f = FORMATS[case["fmt"]], case["rows"], case["hidden"], case["ffn"]
        w, x = 1.0 + 0.1 * _randn(g, h), _randn(g, m, h)
        gate_up = _gguf(fmt, 2 * f, h, g)
        n = x.double() * torch.rsqrt(x.double().square().mean(-1, keepdim=True) + 1e-6) * w.double()
        # the second product's int8 activations round on the first one's values
        return [_quantized(fmt, n) @ _dequant(fmt, gate_up).T, None]
    if kind == "chunk_attn":
        m, p, heads, kv = case["rows"], case["pos0"], case["heads"], case["kv"]
        q = _randn(g, m, heads * HEAD_DIM).double().view(m, heads, HEAD_DIM)
        keys, vals, ks, vs = _cache(g, p + m, kv)
        hidden = torch.arange(p + m, device="cuda")[None, :] > p + torch.arange(m, device="cuda")[:, None]
        out = torch.empty_like(q)
        for h in range(heads):
            j = h % kv
            score = q[:, h] @ (keys[:, j].double() * ks[:, j, None].double()).T / math.sqrt(HEAD_DIM)
            soft = torch.softmax(score.masked_fill(hidden, -math.inf), -1)
            out[:, h] = soft @ (vals[:, j].double() * vs[:, j, None].double())
        return out.reshape(m, heads * HEAD_DIM)
    if kind == "scan":
        m, n = case["rows"], case["seqs"]
        unit = torch.nn.functional.normalize
        state = (0.02 * _randn(g, n, VALUE_HEADS, STATE_DIM, STATE_DIM)).double()
        q = unit(_randn(g, m, n, KEY_HEADS, STATE_DIM), dim=-1).double()
        k = unit(_randn(g, m, n, KEY_HEADS, STATE_DIM), dim=-1).double()
        v = _randn(g, m, n, VALUE_HEADS, STATE_DIM).double()
        decay = torch.sigmoid(2 + 0.5 * _randn(g, m, n, VALUE_HEADS)).double()[..., None, None]
        beta = torch.sigmoid(_randn(g, m, n, VALUE_HEADS)).double()[..., None]
        q, k = (t.repeat_interleave(VALUE_HEADS // KEY_HEADS, 2)[..., None, :] for t in (q, k))
        out = torch.empty((m, n, VALUE_HEADS, STATE_DIM), dtype=torch.float64, device="cuda")
        for t in range(m):
            state = state * decay[t]
            delta = (v[t] - (state * k[t]).sum(-1)) * beta[t]
            state = state + delta[..., None] * k[t]
            out[t] = (state * q[t]).sum(-1) / math.sqrt(STATE_DIM)
        return [out, state]
    if kind == "attn":
        n, heads, kv, top = case["seqs"], case["heads"], case["kv"], case["max_ctx"]
        q = _randn(g, n, heads * HEAD_DIM).double().view(n, heads, HEAD_DIM)
        keys, vals, ks, vs = _cache(g, n * top, kv)
        out = torch.empty_like(q)
        for i, ctx in enumerate(_lengths(n, case["min_ctx"], top)):
            at = slice(i * top, i * top + ctx)
            for h in range(heads):
                j = h % kv
                score = (keys[at, j].double() * ks[at, j, None].double()) @ q[i, h] / math.sqrt(HEAD_DIM)
                out[i, h] = torch.softmax(score, 0) @ (vals[at, j].double() * vs[at, j, None].double())
        return out.reshape(n, heads * HEAD_DIM)
    fmt = FORMATS[case["fmt"]]
    weights, x = _gguf(fmt, case["rows"], case["cols"], g), _randn(g, case["cols"]).double()
    return torch.cat([_dequant(fmt, part) @ x for part in weights.split(16384)])
