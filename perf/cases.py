"""The work that users of this package have it do, as cases that can be timed and compared.

A case is a dict of plain values; ``prepare`` makes its inputs and resident weights from a seed, ``run`` makes one pass
through the public entry points (``NativeHipBackend``, ``HipModel`` and the device-pointer calls of the C ABI), ``work``
says what a pass cannot do without and ``tolerance`` how far another correct implementation may be off.

Four kinds of work:

  gemv     one product on a resident matrix, host vectors in and out: what an engine calls that keeps its activations on
           the host (``gemv_q1_g128_cached``, ``gemv_tq2_g128_cached``, ``gemv_cached_batch``, ``gemm_cached``)
  proj     the projections of a layer on device buffers (QKV, gate || up, down; ``oxb_hip_gemv_dev`` up to eight
           activation rows, ``oxb_hip_gemm_dev`` beyond): an engine that keeps its activations on the GPU
  prefill  ``HipModel.prefill``: a prompt, or a further chunk of one, into a sequence's cache; logits of its last token
  decode   ``HipModel.forward``: single positions of every sequence of a batch, logits to the host-side sampler
"""
from __future__ import annotations

import math

import numpy as np
import torch

from oxibonsai_amd import Q1, TQ2, NativeHipBackend, _lib
from oxibonsai_amd.model import KV_F16, KV_FP8_E4M3, KV_I8, HipModel

FORMATS = {"q1": Q1, "tq2": TQ2}
BLOCK_BYTES = {"q1": 18, "tq2": 34}
KV_TYPES = {"f16": KV_F16, "i8": KV_I8, "fp8": KV_FP8_E4M3}

#: The model shapes of the package's own benchmark: 8B with one-bit weights, 1.7B with ternary ones.
SHAPE_8B = dict(fmt="q1", layers=36, h=4096, inter=12288, nq=32, nkv=8, hd=128, vocab=151936)
SHAPE_1P7B = dict(fmt="tq2", layers=28, h=2048, inter=6144, nq=16, nkv=8, hd=128, vocab=151936)
#: How a model's attention is set up where a case says nothing else: fp16 rows, contiguous cache, every key visible.
PLAIN_CACHE = dict(kv="f16", window=0, sinks=0, page=0)


def listed():
    return [
        # The smallest call: one vector through the K (or V) rows of a 1.7B layer, host to host.  Latency is everything.
        dict(name="gemv_host_kv_rows", kind="gemv", fmt="tq2", n=1024, k=2048, m=1),
        # A batched product between host buffers with a ragged number of rows, as a per-layer prefill makes it.
        dict(name="gemm_host_ragged", kind="gemv", fmt="q1", n=4096, k=4096, m=77),
        # The projections of one decoded token: the package's headline GEMV set.
        dict(name="proj_one_token", kind="proj", fmt="q1", h=4096, qkv=6144, inter=12288, m=1),
        # The same for the eight sequences that share one pass over the weights.
        dict(name="proj_eight_tokens", kind="proj", fmt="q1", h=4096, qkv=6144, inter=12288, m=8),
        # The projections of a prompt chunk, ternary weights.
        dict(name="proj_prompt_512", kind="proj", fmt="tq2", h=2560, qkv=5120, inter=9728, m=512),
        # A short chat turn in front of a small model.
        dict(name="prefill_short", kind="prefill", **SHAPE_1P7B, **PLAIN_CACHE, max_seq=4096, start=0, m=23),
        # A long prompt at once: the largest case.
        dict(name="prefill_2048", kind="prefill", **SHAPE_8B, **PLAIN_CACHE, max_seq=4096, start=0, m=2048),
        # A follow-up message behind several thousand cached positions, one-byte cache rows.
        dict(name="prefill_follow_up", kind="prefill", **SHAPE_8B, **dict(PLAIN_CACHE, kv="i8"), max_seq=8192, start=6000, m=301),
        # A single user's decode loop, small model, a few hundred positions in.
        dict(name="decode_small_model", kind="decode", **SHAPE_1P7B, **PLAIN_CACHE, max_seq=4096, batch=1, ctx=700, steps=4),
        # A handful of sequences (an odd number) on the larger model.
        dict(name="decode_six_sequences", kind="decode", **SHAPE_8B, **PLAIN_CACHE, max_seq=4096, batch=6, ctx=2048, steps=2),
        # A full serving batch with the INT8 cache.
        dict(name="decode_32_sequences", kind="decode", **SHAPE_8B, **dict(PLAIN_CACHE, kv="i8"), max_seq=2304, batch=32, ctx=2048, steps=1),
        # One long document: FP8 rows in pages.
        dict(name="decode_long_context", kind="decode", **SHAPE_8B, **dict(PLAIN_CACHE, kv="fp8", page=16), max_seq=32768, batch=1, ctx=32000, steps=2),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _blocks(rng, lo, hi):
    """A multiple of 128 between lo and hi."""
    return 128 * max(1, round(_log_int(rng, lo, hi) / 128))


def draw(rng):
    kind = rng.choice(["gemv", "proj", "prefill", "prefill", "decode", "decode"])
    fmt = rng.choice(["q1", "tq2"])
    if kind == "gemv":
        return dict(kind=kind, fmt=fmt, n=_log_int(rng, 256, 32768), k=_blocks(rng, 512, 12288), m=_log_int(rng, 1, 128))
    if kind == "proj":
        h = _blocks(rng, 1024, 4096)
        return dict(kind=kind, fmt=fmt, h=h, qkv=_log_int(rng, h, 2 * h), inter=_blocks(rng, 2 * h, 3.5 * h), m=_log_int(rng, 1, 1024))
    h, hd = _blocks(rng, 1024, 4096), rng.choice([64, 128, 128])
    nkv, group = rng.choice([4, 8, 8]), rng.choice([2, 4])
    case = dict(kind=kind, fmt=fmt, layers=rng.randint(8, 28), h=h, inter=_blocks(rng, 2.5 * h, 3.25 * h), nq=nkv * group, nkv=nkv, hd=hd,
                vocab=_log_int(rng, 32000, 152000), kv=rng.choice(["f16", "f16", "i8", "fp8"]), window=0, sinks=0,
                page=rng.choice([0, 0, 16, 128]))
    if rng.random() < 0.2:
        case.update(window=_log_int(rng, 256, 4096), sinks=rng.randint(0, 8))
    if kind == "prefill":
        start, m = rng.choice([0, 0, _log_int(rng, 16, 8000)]), _log_int(rng, 5, 1500)
        return dict(case, max_seq=start + m + 256, start=start, m=m)
    batch = _log_int(rng, 1, 48)
    ctx = _log_int(rng, 16, min(16000, 64000 // batch))
    return dict(case, max_seq=ctx + 300, batch=batch, ctx=ctx, steps=1 if batch > 8 else 2)


# ---- inputs ---------------------------------------------------------------------------------------------------------
_TRITS = np.array([sum(((v // 3**i) % 3) << (2 * i) for i in range(4)) for v in range(81)], dtype=np.uint8)


def _weight(g, fmt, n, k):
    """Blocks of an n x k matrix in the file formats' byte order: balanced signs / trits, fp16 scales.  The scale keeps
    the size of what passes through, as trained weights do: about 1 / sqrt(k) for each weight."""
    nb = n * (k // 128)
    d = (g.random(nb, dtype=np.float32) + np.float32(0.5)) * np.float32((1.0 if fmt == "q1" else 1.22) / math.sqrt(k))
    d = d.astype(np.float16).view(np.uint8).reshape(nb, 2)
    out = np.empty((nb, BLOCK_BYTES[fmt]), dtype=np.uint8)
    if fmt == "q1":
        out[:, :2] = d
        out[:, 2:] = np.frombuffer(g.bytes(nb * 16), dtype=np.uint8).reshape(nb, 16)
    else:
        out[:, :32] = _TRITS[np.frombuffer(g.bytes(nb * 64), dtype=np.uint16) % 81].reshape(nb, 32)
        out[:, 32:] = d
    return out.reshape(-1)


def _norm(g, n):
    return (1.0 + 0.02 * g.standard_normal(n, dtype=np.float32)).astype(np.float16).astype(np.float32)


def _rows(g, m, h):
    """Embedding rows, stored as fp16 in a checkpoint and widened."""
    return g.standard_normal((m, h), dtype=np.float32).astype(np.float16).astype(np.float32)


class _State:
    """What a program keeps between calls; the device memory goes with the object."""

    def __init__(self, case):
        self.case, self.be = case, NativeHipBackend(0)
        self.handles, self.model = [], None

    def upload(self, g, n, k):
        b = _weight(g, self.case["fmt"], n, k)
        up = self.be.upload_weights_raw if self.case["fmt"] == "q1" else self.be.upload_weights_ternary
        self.handles.append(up(b, n, k))
        return self.handles[-1]

    def __del__(self):
        if self.model is not None:
            self.model.close()
        for h in self.handles:
            self.be.free_weights(h)


def _make_model(state, g, c, batch):
    qd, kd, h, inter = c["nq"] * c["hd"], c["nkv"] * c["hd"], c["h"], c["inter"]
    shapes = dict(q=(qd, h), k=(kd, h), v=(kd, h), o=(h, qd), gate=(inter, h), up=(inter, h), down=(h, inter))
    # three layers' worth of random blocks; every layer of the model gets a copy of its own on the device
    blocks = [{n: _weight(g, c["fmt"], *s) for n, s in shapes.items()} for _ in range(min(3, c["layers"]))]
    layers = [dict(blocks[i % len(blocks)], attn_norm=_norm(g, h), ffn_norm=_norm(g, h), q_norm=_norm(g, c["hd"]), k_norm=_norm(g, c["hd"]))
              for i in range(c["layers"])]
    cfg = dict(fmt=FORMATS[c["fmt"]], n_layers=c["layers"], h=h, inter=inter, nq=c["nq"], nkv=c["nkv"], hd=c["hd"], vocab=c["vocab"],
               max_seq=c["max_seq"], eps=1e-6, rope_theta=1e6)
    m = state.model = HipModel(state.be, cfg, {"layers": layers, "final_norm": _norm(g, h), "lm_head": _weight(g, c["fmt"], c["vocab"], h)}, batch=batch)
    if c["kv"] != "f16" or c["window"] or c["page"]:
        pages = batch * -(-c["max_seq"] // c["page"]) if c["page"] else 0
        m.set_attention(KV_TYPES[c["kv"]], c["window"], c["sinks"], c["page"], pages)
    return m


def _fill(m, g, c, n):
    """n positions of every sequence's cache, written by the prefill of prompts in chunks of at most 2048 tokens that are
    drawn from a vocabulary of 1024 embedding rows."""
    table = _rows(g, 1024, c["h"])
    for seq in range(m.batch):
        for p in range(0, n, 2048):
            m.prefill(table[g.integers(0, len(table), min(2048, n - p))], p, seq=seq, want_logits=False)


def prepare(case, seed):
    g, s, kind = np.random.default_rng(seed), _State(case), case["kind"]
    if kind == "gemv":
        s.w = s.upload(g, case["n"], case["k"])
        s.x = g.standard_normal((case["m"], case["k"]), dtype=np.float32)
    elif kind == "proj":
        h, inter, m = case["h"], case["inter"], case["m"]
        s.calls = []
        for n, k in ((case["qkv"], h), (2 * inter, h), (h, inter)):
            x = torch.from_numpy(g.standard_normal((m, k), dtype=np.float32)).cuda()
            s.calls.append((s.upload(g, n, k), x, torch.zeros((m, n), device="cuda"), n, k))
        lib = _lib.lib()
        s.product = lib.oxb_hip_gemv_dev if m <= 8 else lib.oxb_hip_gemm_dev
        torch.cuda.synchronize()     # the library's stream is its own
    elif kind == "prefill":
        m = _make_model(s, g, case, 1)
        _fill(m, g, case, case["start"])
        s.rows = _rows(g, case["m"], case["h"])
    else:
        m = _make_model(s, g, case, case["batch"])
        _fill(m, g, case, case["ctx"])
        s.rows = [_rows(g, case["batch"], case["h"]) for _ in range(case["steps"])]
    return s


def run(s):
    c = s.case
    if c["kind"] == "gemv":
        if c["m"] == 1:
            f = s.be.gemv_q1_g128_cached if c["fmt"] == "q1" else s.be.gemv_tq2_g128_cached
            return f(s.w, s.x[0], c["n"], c["k"])
        if c["m"] <= 8:
            return s.be.gemv_cached_batch(s.w, s.x, c["n"], c["k"])
        return s.be.gemm_cached(s.w, s.x, c["m"], c["n"], c["k"])
    if c["kind"] == "proj":
        for w, x, y, n, k in s.calls:
            args = (n, k, c["m"]) if c["m"] <= 8 else (c["m"], n, k)
            if s.product(int(w), x.data_ptr(), y.data_ptr(), *args):
                raise RuntimeError(_lib.last_error())
        return [y for _, _, y, _, _ in s.calls]
    if c["kind"] == "prefill":
        logits, token = s.model.prefill(s.rows, c["start"])
        return {"logits": logits, "chosen": logits[token]}
    out = []
    for i, rows in enumerate(s.rows):      # the tokens of a known continuation: every step's input is fixed
        logits, tokens = s.model.forward(rows, c["ctx"] + i)
        out.append({"logits": logits, "chosen": logits[np.arange(c["batch"]), tokens]})
    return out


# ---- what a pass costs at least --------------------------------------------------------------------------------------
def _visible(c, pos):
    """Keys that the query at position pos sees."""
    return pos + 1 if not c["window"] else min(pos + 1, c["window"])


def _seen_by_any(c, first, last):
    """Keys that at least one of the queries at first .. last sees."""
    n = _visible(c, first) + last - first
    return min(last + 1, n)


def work(case):
    c = case
    if c["kind"] == "gemv":
        return {"bytes": c["n"] * (c["k"] // 128) * BLOCK_BYTES[c["fmt"]] + 4 * c["m"] * (c["k"] + c["n"]), "flops": 2 * c["m"] * c["n"] * c["k"]}
    if c["kind"] == "proj":
        t = [work(dict(kind="gemv", fmt=c["fmt"], n=n, k=k, m=c["m"])) for n, k in ((c["qkv"], c["h"]), (2 * c["inter"], c["h"]), (c["h"], c["inter"]))]
        return {key: sum(w[key] for w in t) for key in ("bytes", "flops")}
    qd, kd = c["nq"] * c["hd"], c["nkv"] * c["hd"]
    layer, head = (qd + 2 * kd) * c["h"] + qd * c["h"] + 3 * c["h"] * c["inter"], c["vocab"] * c["h"]
    per_weight = BLOCK_BYTES[c["fmt"]] / 128
    row = 2 * c["nkv"] * (2 * c["hd"] if c["kv"] == "f16" else c["hd"] + 4)    # K and V of one position in one layer
    if c["kind"] == "prefill":
        first, last = c["start"], c["start"] + c["m"] - 1
        pairs = sum(_visible(c, p) for p in range(first, last + 1))
        return {"bytes": (c["layers"] * layer + head) * per_weight + 4 * c["m"] * c["h"] + 4 * c["vocab"] + c["layers"] * row * _seen_by_any(c, first, last),
                "flops": 2 * c["m"] * c["layers"] * layer + 2 * head + 4 * c["layers"] * qd * pairs}
    B, total = c["batch"], {"bytes": 0, "flops": 0}
    for i in range(c["steps"]):
        seen = _visible(c, c["ctx"] + i)
        total["bytes"] += (c["layers"] * layer + head) * per_weight + 4 * B * (c["h"] + c["vocab"]) + B * c["layers"] * row * seen
        total["flops"] += 2 * B * (c["layers"] * layer + head) + 4 * B * c["layers"] * qd * seen
    return total


def tolerance(case):
    c = case
    if c["kind"] in ("gemv", "proj"):
        # up to eight rows the products are exact in fp32; beyond, activations are rounded to fp16 (2^-11)
        return {"rel": 1e-5, "max": 1e-4} if c["m"] <= 8 else {"rel": 1e-3, "max": 1e-2}
    # fp16 activations or cache rows through all layers: a few thousandths of the logits' size.  A one-byte cache adds rows
    # whose codes fall on the other side of a rounding boundary: one step of a code is 1 % (INT8) to 6 % (FP8) of a value.
    return {"rel": 5e-3, "max": 5e-2} if c["kv"] == "f16" else {"rel": 2e-2, "max": 0.2}
