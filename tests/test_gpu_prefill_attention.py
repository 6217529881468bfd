"""The prefill's attention kernel on its own (oxb_hip_model_prefill_attention), against softmax(q K^T / sqrt(hd)) V in
float64 over the cache rows that the device stored.

What the kernel rounds, element by element of the output: every probability to fp16 (2^-11 of it), every V value of a
quantised cache twice (the row scale to fp16, the product to fp16), and the scores to fp32 accuracy (q enters as fp16 hi +
lo, 2^-22 of it; sums of hd products).  With sum(p |v|) for one output element, p the float64 probabilities,

    |out - want| <= (2^-11 + 2 * 2^-11 [quantised] + 2^-15) sum(p |v|) + n_keys 2^-25 max|v| / sum

where the last term covers probabilities below fp16's smallest normal number (a quantum of 2^-24, sum: in units of the
largest probability)."""
import ctypes as C

import numpy as np
import pytest

from helpers import Q1, TQ2
from oracle import oracle
from oxibonsai_amd import _lib, synth
from oxibonsai_amd.backend import _check
from oxibonsai_amd.model import KV_F16, KV_FP8_E4M3, KV_I8, HipModel

pytestmark = pytest.mark.gpu


def _model(backend, nq, nkv, hd, max_seq, q_norm=None, seed=1, batch=1):
    h = 128
    cfg = dict(fmt=Q1, n_layers=2, h=h, inter=256, nq=nq, nkv=nkv, hd=hd, vocab=32, max_seq=max_seq, eps=1e-6, rope_theta=1e6)
    w = synth.make_model(cfg, seed)
    if q_norm is not None:
        for layer in w["layers"]:
            layer["q_norm"], layer["k_norm"] = np.full(hd, q_norm, np.float32), np.ones(hd, np.float32)
    return HipModel(backend, cfg, w, batch=batch), w


def _attend(gpu, layer, seq, qkv, pos):
    cfg = gpu.cfg
    qkv = np.ascontiguousarray(qkv, dtype=np.float32)
    out = np.full((qkv.shape[0], cfg["nq"] * cfg["hd"]), np.nan, dtype=np.float32)
    _check(_lib.lib().oxb_hip_model_prefill_attention(gpu.id, layer, seq, qkv.ctypes.data_as(_lib.f32p), qkv.shape[0], pos, out.ctypes.data_as(_lib.f32p)))
    return out.reshape(qkv.shape[0], cfg["nq"], cfg["hd"])


def _rows(gpu, layer, head, n, seq):
    """The device's own cache rows as float64 values."""
    mode = gpu.attention().kv_dtype
    k, v, ks, vs = gpu.read_kv(layer, head, 0, n, seq)
    if mode == KV_F16:
        return k.astype(np.float64), v.astype(np.float64)
    val = (lambda c: c.view(np.int8).astype(np.float64)) if mode == KV_I8 else (lambda c: oracle.fp8_decode(np.arange(256, dtype=np.uint8)).astype(np.float64)[c])
    return val(k) * ks[:, None].astype(np.float64), val(v) * vs[:, None].astype(np.float64)


def _queries(cfg, w, layer, qkv, cos, sin):
    """Q in float64: per-head RMSNorm, rotation of the pairs (d, d + hd/2), log2 e / sqrt(hd)."""
    M, nq, hd = qkv.shape[0], cfg["nq"], cfg["hd"]
    q = qkv[:, :nq * hd].astype(np.float64).reshape(M, nq, hd)
    q = q / np.sqrt((q * q).mean(-1, keepdims=True) + cfg["eps"]) * w["layers"][layer]["q_norm"].astype(np.float64)
    a, b = q[..., :hd // 2], q[..., hd // 2:]
    c, s = cos[:, None, :].astype(np.float64), sin[:, None, :].astype(np.float64)
    return np.concatenate([a * c - b * s, a * s + b * c], axis=-1) * (np.log2(np.e) / np.sqrt(hd))


def _visible(pos, n, window, sinks):
    key, qp = np.arange(n)[None, :], pos[:, None]
    return (key <= qp) & ((window == 0) | (key < sinks) | (qp - key < max(window - sinks, 0)))


# (queries, first position, q heads, kv heads, head_dim, cache, window, sinks, page size): what the launcher makes of them is
# noted as runs of keys x blocks per run (all with one query tile per wave).
CASES = [
    (7, 0, 2, 1, 128, KV_F16, 0, 0, 0),           # a single block, whose rows the launch stores itself, as in the next seven
    (32, 0, 8, 2, 128, KV_I8, 0, 0, 0),           # the longest of head_dim 128: two workgroups of a kv head
    (17, 0, 3, 3, 128, KV_F16, 0, 0, 0),          # one head per workgroup, three kv heads
    (31, 0, 5, 1, 128, KV_FP8_E4M3, 9, 2, 16),    # five workgroups of one kv head, windowed, paged
    (64, 0, 8, 2, 64, KV_F16, 0, 0, 64),          # the longest of head_dim 64, paged
    (50, 0, 4, 1, 32, KV_I8, 0, 0, 0),
    (32, 0, 2, 1, 256, KV_FP8_E4M3, 0, 0, 0),     # the longest of head_dim 256
    (1, 0, 4, 2, 64, KV_I8, 0, 0, 0),
    (33, 0, 4, 2, 128, KV_I8, 0, 0, 0),           # one row more than the launch stores: 1 x 2
    (130, 0, 8, 2, 64, KV_F16, 0, 0, 0),          # 1 x 3
    (5, 1200, 1, 1, 128, KV_F16, 0, 0, 0),        # 13 x 3: an odd number (13 x 5 x 1) of rows of sums
    (7, 1500, 3, 3, 128, KV_F16, 0, 0, 16),       # 12 x 4, paged
    (49, 3001, 2, 2, 64, KV_F16, 0, 0, 32),       # 12 x 4, the last workgroup one query, paged
    (48, 3001, 4, 2, 128, KV_F16, 0, 0, 0),       # 16 x 6
    (64, 4000, 4, 2, 128, KV_F16, 0, 0, 0),       # 16 x 8
    (331, 768, 4, 2, 128, KV_I8, 0, 0, 0),        # 7 x 5
    (331, 768, 4, 2, 128, KV_FP8_E4M3, 0, 0, 16),
    (33, 2900, 4, 1, 32, KV_I8, 0, 0, 64),        # 12 x 4: half a wave fetches all pieces of a block
    (100, 3000, 4, 1, 32, KV_FP8_E4M3, 0, 0, 0),  # 10 x 5
    (3, 2300, 5, 1, 128, KV_I8, 0, 0, 128),       # five heads: one per workgroup
    (21, 1000, 2, 1, 256, KV_F16, 0, 0, 0),       # 16 x 2
    (17, 900, 2, 2, 256, KV_I8, 0, 0, 16),        # 15 x 2
    (90, 2100, 8, 2, 64, KV_F16, 700, 5, 0),      # a window: 5 x 3, runs that some queries see nothing of
    (50, 2500, 4, 2, 128, KV_I8, 1200, 70, 16),   # 11 x 4, sinks across a block's edge, paged
    (40, 2500, 4, 2, 64, KV_FP8_E4M3, 64, 64, 32),  # nothing visible but the sinks
]


@pytest.mark.parametrize("M,start,nq,nkv,hd,mode,window,sinks,page", CASES)
def test_prefill_attention_matches_float64(backend, M, start, nq, nkv, hd, mode, window, sinks, page):
    max_seq, layer, seq = start + M + 9, 1, 1
    gpu, w = _model(backend, nq, nkv, hd, max_seq, batch=2)
    g = np.random.default_rng([M, start, hd, mode])
    try:
        if mode != KV_F16 or window or page:
            gpu.set_attention(mode, window, sinks, page, 2 * -(-max_seq // page) if page else 0)
        ang = g.uniform(0, 2 * np.pi, (max_seq, hd // 2)).astype(np.float32)
        cos, sin = np.cos(ang), np.sin(ang)
        gpu.set_rope_rows(0, cos, sin)
        qkv = g.standard_normal((start + M, (nq + 2 * nkv) * hd)).astype(np.float32)
        if start:
            gpu.kv_reserve(0, 17)                 # (another sequence's pages in between)
            _attend(gpu, layer, seq, qkv[:start], 0)
        got = _attend(gpu, layer, seq, qkv[start:], start)
        n = start + M
        q = _queries(gpu.cfg, w, layer, qkv[start:], cos[start:n], sin[start:n])
        vis = _visible(np.arange(start, n), n, window, sinks)
        worst = 0.0
        for kvh in range(nkv):
            K, V = _rows(gpu, layer, kvh, n, seq)
            for hh in range(nq // nkv):
                s = np.where(vis, q[:, kvh * (nq // nkv) + hh] @ K.T, -np.inf)
                p = np.exp2(s - s.max(1, keepdims=True))
                total = p.sum(1, keepdims=True)
                want, size = p @ V / total, p @ np.abs(V) / total
                bound = ((3 if mode != KV_F16 else 1) * 2.0**-11 + 2.0**-15) * size + n * 2.0**-25 * np.abs(V).max() / total
                worst = max(worst, float((np.abs(got[:, kvh * (nq // nkv) + hh] - want) / bound).max()))
        assert worst <= 1.0, worst
    finally:
        gpu.close()


# Two query tiles per wave and two walkers per workgroup, as (queries, first position, q heads, kv heads, cache, window,
# sinks, page size), noted as before with blocks of 64 keys.
WALKED = [
    (1000, 3000, 28, 4, KV_F16, 0, 0, 0),         # 1 x 63: the second walker has no last block; seven heads, one per workgroup
    (960, 2000, 28, 4, KV_F16, 2000, 70, 32),     # 1 x 38, sinks across a block's edge, paged
    (1000, 1000, 24, 8, KV_FP8_E4M3, 1000, 70, 16),  # 1 x 22
    (1000, 6000, 8, 2, KV_I8, 0, 0, 0),           # 4 x 28, four heads per workgroup: 1000 ends inside the last one's first tile
    (960, 4000, 8, 2, KV_I8, 4000, 70, 64),       # 4 x 17, odd runs, some of them empty
    (200, 6000, 24, 8, KV_I8, 0, 0, 0),           # 5 x 20, the last run 17
]


@pytest.mark.parametrize("M,start,nq,nkv,mode,window,sinks,page", WALKED)
def test_two_walkers_match_float64(backend, M, start, nq, nkv, mode, window, sinks, page):
    max_seq, layer, seq, hd = start + M, 1, 1, 128
    gpu, w = _model(backend, nq, nkv, hd, max_seq, batch=2)
    g = np.random.default_rng([M, start, mode])
    try:
        if mode != KV_F16 or window or page:
            gpu.set_attention(mode, window, sinks, page, 2 * -(-max_seq // page) if page else 0)
        ang = g.uniform(0, 2 * np.pi, (max_seq, hd // 2)).astype(np.float32)
        cos, sin = np.cos(ang), np.sin(ang)
        gpu.set_rope_rows(0, cos, sin)
        qkv = g.standard_normal((max_seq, (nq + 2 * nkv) * hd), dtype=np.float32)
        _attend(gpu, layer, seq, qkv[:start], 0)
        got = _attend(gpu, layer, seq, qkv[start:], start)
        t = np.unique(np.r_[0, 1, 15:M:31, M - 17, M - 2, M - 1])
        q = _queries(gpu.cfg, w, layer, qkv[start + t], cos[start + t], sin[start + t])
        vis = _visible(start + t, max_seq, window, sinks)
        worst = 0.0
        for kvh in (0, nkv - 1):
            K, V = _rows(gpu, layer, kvh, max_seq, seq)
            for hh in range(nq // nkv):
                head = kvh * (nq // nkv) + hh
                s = np.where(vis, q[:, head] @ K.T, -np.inf)
                p = np.exp2(s - s.max(1, keepdims=True))
                total = p.sum(1, keepdims=True)
                want, size = p @ V / total, p @ np.abs(V) / total
                bound = ((3 if mode != KV_F16 else 1) * 2.0**-11 + 2.0**-15) * size + max_seq * 2.0**-25 * np.abs(V).max() / total
                worst = max(worst, float((np.abs(got[t, head] - want) / bound).max()))
        assert worst <= 1.0, worst
    finally:
        gpu.close()


@pytest.mark.parametrize("mode", [KV_F16, KV_I8, KV_FP8_E4M3])
@pytest.mark.parametrize("hd,n", [(128, 32), (64, 64), (32, 64), (256, 32), (128, 1)])
def test_a_short_prompt_stores_the_rows_that_a_longer_one_does(backend, hd, n, mode):
    # n tokens: the attention launch works the new rows out; one more than it takes: a launch of their own does.
    gpu, _ = _model(backend, 12, 3, hd, 80, batch=2)
    try:
        if mode != KV_F16:
            gpu.set_attention(mode, 0, 0, 16, 2 * 5)
        x = np.random.default_rng([hd, n, mode]).standard_normal((65 if hd < 128 else 33, 18 * hd)).astype(np.float32)
        _attend(gpu, 1, 0, x[:n], 0)
        _attend(gpu, 1, 1, x, 0)
        for head in range(3):
            for a, b in zip(gpu.read_kv(1, head, 0, n, 0), gpu.read_kv(1, head, 0, n, 1)):
                assert np.array_equal(a.view(np.uint8), b.view(np.uint8))
    finally:
        gpu.close()


@pytest.mark.parametrize("shape", ["spread", "sink", "far sink", "late peak"])
@pytest.mark.parametrize("M", [16, 64])
def test_prefill_attention_weights_are_relative_to_the_row_maximum(backend, M, shape):
    # Against float64 the kernel is as good as probabilities rounded to fp16 relative to the row's own maximum, over their
    # unrounded sum: the largest weight is exactly 1, which an attention sink (one key 12 or 17 above 16 000 others) lives on.
    # The comparison allows a quarter more, and 3e-6 for sums of 16 000 fp32 terms.
    nq, nkv, hd, n = 4, 2, 128, 16000 + M
    c = {"spread": 3.0, "sink": 12.0 / 11.2, "far sink": 17.0 / 11.2, "late peak": 6.0 / 11.2}[shape]
    gpu, w = _model(backend, nq, nkv, hd, n, q_norm=c)
    g = np.random.default_rng([M, len(shape)])
    try:
        gpu.set_rope_rows(0, np.ones((n, hd // 2), np.float32), np.zeros((n, hd // 2), np.float32))
        x = g.standard_normal((n, nq + 2 * nkv, hd)).astype(np.float32)
        if shape != "spread":
            u = g.standard_normal(hd)
            u /= np.linalg.norm(u)
            k = x[:, nq:nq + nkv]
            k -= (k @ u)[..., None] * u
            k[9000 if shape == "late peak" else 0] = u * 11.0
            x[:, :nq] = 11.0 * u + 0.12 * x[:, :nq]
        qkv = x.reshape(n, -1)
        _attend(gpu, 0, 0, qkv[:16000], 0)
        got = _attend(gpu, 0, 0, qkv[16000:], 16000)
        q = _queries(gpu.cfg, w, 0, qkv[16000:], np.ones((M, hd // 2)), np.zeros((M, hd // 2)))
        vis = _visible(np.arange(16000, n), n, 0, 0)
        err = ref = size = 0.0
        for h in range(nq):
            K, V = _rows(gpu, 0, h // (nq // nkv), n, 0)
            s = np.where(vis, q[:, h] @ K.T, -np.inf)
            p = np.exp2(s - s.max(1, keepdims=True))
            want = p @ V / p.sum(1, keepdims=True)
            rounded = p.astype(np.float16).astype(np.float64) @ V / p.sum(1, keepdims=True)
            err += ((got[:, h] - want)**2).sum()
            ref += ((rounded - want)**2).sum()
            size += (want**2).sum()
        err, ref = np.sqrt(err / size), np.sqrt(ref / size)
        print(f"{shape}, {M} queries: {err:.2e} off float64, weights rounded against the maximum {ref:.2e}")
        assert err <= 1.25 * ref + 3e-6, (err, ref)
    finally:
        gpu.close()


@pytest.mark.parametrize("fmt", [Q1, TQ2])
def test_steps_behind_value_rows_larger_than_the_model_makes(backend, fmt):
    # Rows that the caller stores may be larger than anything the model's own value rows and norms can make, the outputs of the
    # attention with them.  Nine sequences and prompts (fp16 products) against a single sequence's steps (fp32): 1e-2, as for any prefill.
    cfg = dict(fmt=fmt, n_layers=2, h=512, inter=512, nq=4, nkv=2, hd=128, vocab=96, max_seq=64, eps=1e-6, rope_theta=1e6)
    w = synth.make_model(cfg, 12)
    g = np.random.default_rng(3)
    qkv = g.standard_normal((20, 8 * 128)).astype(np.float32)
    qkv[:, 6 * 128:] *= 1e4
    rows = g.standard_normal((9, 512)).astype(np.float32)
    one, nine = HipModel(backend, cfg, w), HipModel(backend, cfg, w, batch=9)
    try:
        nine.forward(rows, 0)           # a captured step that is in use already
        for seq in range(9):
            for layer in range(2):
                _attend(nine, layer, seq, qkv, 0)
        for layer in range(2):
            _attend(one, layer, 0, qkv, 0)
        got = nine.forward(rows, 20)[0]
        want = np.stack([one.forward(r, 20)[0][0] for r in rows])
        assert np.all(np.abs(got - want) <= 1e-2 * np.maximum(1.0, np.abs(want)))
        for i, r in enumerate(rows):
            last = one.forward(r, 20 + i)[0][0]
        got = one.prefill(rows, 20)[0]
        assert np.all(np.abs(got - last) <= 1e-2 * np.maximum(1.0, np.abs(last)))
    finally:
        one.close()
        nine.close()
