"""GPU parity of the batched prefill pipeline (prefill GEMMs on the matrix cores, causal attention, KV store)
against the CPU oracle's token-by-token forward, through the C ABI.

The oracle is run with K/V rounded through f16 like the GPU cache.  The prefill projections round their
activations to fp16, so logits are held to 1e-2 under the reference's gate form
(abs < tol or |a-b| / max(|a|, |b|, 1e-3) < tol, metal_prefill_ternary_parity_tests.rs:294-308, which the
reference applies to its own batched-prefill-vs-sequential comparison at :254-311); greedy tokens must agree
wherever the oracle's top-2 margin exceeds that tolerance.  Decode steps that follow a prefill read the
cache the prefill wrote, which checks the stored keys and values."""
import numpy as np
import pytest

from helpers import Q1, TQ2, gemm_plan, parity_violations
from oracle import oracle
from oxibonsai_amd import GpuError, synth
from oxibonsai_amd.model import HipModel

pytestmark = pytest.mark.gpu
PREFILL_TOL = 1e-2

TINY = dict(n_layers=2, h=128, inter=256, nq=4, nkv=2, hd=32, vocab=32, max_seq=64, eps=1e-6, rope_theta=1e6)
SMALL = dict(n_layers=3, h=512, inter=1536, nq=8, nkv=2, hd=64, vocab=1000, max_seq=400, eps=1e-6, rope_theta=1e6)
MID = dict(n_layers=2, h=512, inter=1024, nq=8, nkv=4, hd=128, vocab=512, max_seq=700, eps=1e-6, rope_theta=1e6)
WIDE = dict(n_layers=1, h=256, inter=512, nq=2, nkv=2, hd=256, vocab=64, max_seq=96, eps=1e-6, rope_theta=1e4)
# groups of four and eight q heads per kv head: the attention workgroup shares K and V between its waves
G4_HD32 = dict(n_layers=2, h=128, inter=256, nq=4, nkv=1, hd=32, vocab=64, max_seq=200, eps=1e-6, rope_theta=1e4)
G4_HD256 = dict(n_layers=1, h=1024, inter=512, nq=4, nkv=1, hd=256, vocab=64, max_seq=96, eps=1e-6, rope_theta=1e6)
G8_HD128 = dict(n_layers=1, h=1024, inter=512, nq=8, nkv=1, hd=128, vocab=64, max_seq=160, eps=1e-6, rope_theta=1e6)
# an FFN wide enough (392 gate tiles x 7 token tiles of 80) for the gate || up GEMM to take three row tiles per wave, gate
# and up tiles in different waves; 392 = 65 x 6 + 2 and 500 = 6 x 80 + 20: the last workgroups are partly empty
LONG_FFN = dict(n_layers=1, h=256, inter=6272, nq=4, nkv=2, hd=64, vocab=64, max_seq=520, eps=1e-6, rope_theta=1e6)


def _rows(seed, n, h):
    return synth.embedding_rows(seed, [(7 * i + 3) % 211 for i in range(n)], h) * 50.0   # O(1) activations


def _oracle_logits(cpu, rows, pos0=0):
    out = None
    for i, r in enumerate(rows):
        last = i == len(rows) - 1
        out = cpu.forward(r, pos0 + i, want_logits=last)
    return out


def _check(got, want, tok):
    assert parity_violations(got, want, PREFILL_TOL) == 0, f"max abs {np.max(np.abs(got - want)):.3e}"
    top2 = np.sort(want)[-2:]
    if top2[1] - top2[0] > 2 * PREFILL_TOL * max(1.0, abs(top2[1])):
        assert tok == oracle.argmax_first(want)
    assert tok == int(np.argmax(got))


@pytest.mark.parametrize("fmt", [TQ2, Q1])
@pytest.mark.parametrize("cfg,n", [(TINY, 8), (TINY, 17), (TINY, 33), (SMALL, 130), (MID, 70), (WIDE, 40),
                                   (G4_HD32, 97), (G4_HD32, 32), (G4_HD256, 50), (G8_HD128, 100), (SMALL, 1), (SMALL, 65),
                                   (LONG_FFN, 500)])
def test_prefill_matches_sequential_oracle(backend, fmt, cfg, n):
    cfg = dict(cfg, fmt=fmt)
    w = synth.make_model(cfg, 100 + n)
    cpu = oracle.OracleModel(cfg, w, kv_f16=True)
    gpu = HipModel(backend, cfg, w, batch=1)
    try:
        rows = _rows(5, n, cfg["h"])
        got, tok = gpu.prefill(rows)
        _check(got, _oracle_logits(cpu, rows), tok)
        # decode continues on the cache the prefill wrote
        for step in range(3):
            r = _rows(6 + step, 1, cfg["h"])[0]
            want = cpu.forward(r, n + step)
            g, t = gpu.forward(r, n + step)
            _check(g[0], want, int(t[0]))
    finally:
        gpu.close()


# (format, hidden, inter, q heads, kv heads, head_dim, tokens; the gate || up product's form: narrow kernel, row tiles, token
# tiles; K slices of the down product, whose sums the next layer's pack adds): the forms of the SwiGLU product ...
SWIGLU_FORMS = [(fmt, 640, 384, 4, 2, 64, m, (1, 2, -(-m // 16)), None) for fmt in (Q1, TQ2) for m in (9, 19, 34, 49, 67, 82, 97)]
SWIGLU_FORMS += [(fmt, 256, 4224, 4, 2, 64, m, (1, 4, -(-m // 16)), None) for fmt in (Q1, TQ2) for m in (19, 34, 49)]
SWIGLU_FORMS += [(fmt, 256, inter, 4, 2, 64, m, form, None) for fmt in (Q1, TQ2) for m, inter, form in
                 ((115, 384, (0, 2, 4)), (67, 8320, (0, 2, 5)), (82, 8320, (0, 3, 4)), (129, 8320, (0, 3, 5)))]
SWIGLU_FORMS += [(Q1, 640, 8320, 4, 2, 64, 1, (1, 6, 1), None), (Q1, 256, 8320, 4, 2, 64, 19, (1, 6, 2), None), (Q1, 256, 10496, 4, 2, 64, 500, (0, 3, 8), None),
                 (TQ2, 256, 12416, 4, 2, 64, 250, (0, 2, 8), None), (TQ2, 256, 11008, 4, 2, 64, 161, (0, 3, 8), None)]
# ... and the packs that add a residual product's K slices: up to 64 rows one to four items per thread, beyond two or four
# rows per workgroup with rows of up to 4096, 8192 and 12288 values
SUM_PACKS = [(Q1, 1024, 4096, 16, 4, 128, 40, None, 4), (TQ2, 4096, 4096, 4, 2, 64, 64, None, 2), (Q1, 4352, 4608, 4, 2, 64, 40, None, 3),
             (Q1, 1024, 4096, 16, 4, 128, 100, None, 4), (TQ2, 4096, 4096, 4, 2, 64, 130, None, 4), (TQ2, 4352, 4608, 4, 2, 64, 66, None, 3),
             (Q1, 8320, 3072, 4, 2, 64, 66, None, 3), (TQ2, 1024, 4096, 16, 4, 128, 520, None, 4), (TQ2, 4352, 4608, 4, 2, 64, 600, None, 3),
             (TQ2, 10240, 9216, 4, 2, 64, 600, None, 3)]


@pytest.mark.parametrize("fmt,h,inter,nq,nkv,hd,n,form,slices", SWIGLU_FORMS + SUM_PACKS)
def test_prefill_rows_match_the_oracle(backend, fmt, h, inter, nq, nkv, hd, n, form, slices):
    """Every token's K and V rows of the second layer - behind all products of the first one - and the last token's logits.
    About six roundings of activations to fp16 (2^-11 / sqrt 3 in the root mean square each) lie in front of a row, and one
    of the row itself: 7e-4; three times that is allowed for any single row."""
    narrow, rt, _, ct, _, _ = gemm_plan(fmt, n, 2 * inter, h, swiglu=True)
    assert form in (None, (narrow, rt, ct))
    assert slices in (None, gemm_plan(fmt, n, h, inter, sum_later=True)[4])
    cfg = dict(fmt=fmt, n_layers=2, h=h, inter=inter, nq=nq, nkv=nkv, hd=hd, vocab=64, max_seq=n + 4, eps=1e-6, rope_theta=1e6)
    w = synth.make_model(cfg, 300 + n)
    rows = _rows(21, n, h)
    cpu = oracle.OracleModel(cfg, w, kv_f16=True, simd=True)
    want = cpu.forward_batch(rows, 0)
    gpu = HipModel(backend, cfg, w)
    try:
        got, tok = gpu.prefill(rows)
        worst = 0.0
        for head in range(nkv):
            for a, b in zip(gpu.read_kv(1, head, 0, n)[:2], cpu.cache_rows(1, head, 0, n)):
                d = a.astype(np.float64) - b
                worst = max(worst, float(np.sqrt(np.mean(d * d, axis=1) / np.mean(b.astype(np.float64) ** 2, axis=1)).max()))
        print(f"worst row {worst:.2e}, logits {np.max(np.abs(got - want)):.2e} off, largest {np.max(np.abs(want)):.2e}")
        assert worst <= 2.1e-3, worst
        _check(got, want, tok)
    finally:
        gpu.close()


@pytest.mark.parametrize("cfg,n", [(SMALL, 23), (SMALL, 130), (LONG_FFN, 500)])
def test_prefill_of_ternary_ffn_scales_above_and_below_a_doubled_weight(backend, cfg, n):
    # gate and up with scales up to 2^15 .. 2^16, which do not enter the products twice as large, and with half of each, which do; the
    # norm weights in front of them take the factor off again.  Powers of two all along: the same bits.
    cfg, logits = dict(cfg, fmt=TQ2), []
    rows = _rows(9, n, cfg["h"])
    for top in (14, 15):
        w = synth.make_model(cfg, 77)
        for ly in w["layers"]:
            d = [ly[name].reshape(-1, 34)[:, 32:].copy().view(np.float16) for name in ("gate", "up")]
            up = top - int(np.floor(np.log2(max(np.abs(v).max() for v in d).astype(np.float64))))
            for name, v in zip(("gate", "up"), d):
                ly[name].reshape(-1, 34)[:, 32:] = np.ldexp(v.astype(np.float32), up).astype(np.float16).view(np.uint8)
            ly["ffn_norm"] = np.ldexp(ly["ffn_norm"], -up).astype(np.float32)
        gpu = HipModel(backend, cfg, w, batch=1)
        try:
            logits.append(gpu.prefill(rows)[0].copy())
        finally:
            gpu.close()
    assert np.all(np.isfinite(logits[0])) and np.array_equal(*logits)


def test_chunked_prefill_equals_one_prefill(backend):
    # the reference's chunked 4 + 4 = 8 test (metal_prefill_ternary_parity_tests.rs:427-473), at tile-crossing sizes
    cfg = dict(SMALL, fmt=TQ2)
    w = synth.make_model(cfg, 77)
    rows = _rows(8, 150, cfg["h"])
    a = HipModel(backend, cfg, w)
    b = HipModel(backend, cfg, w)
    try:
        whole, tok_w = a.prefill(rows)
        b.prefill(rows[:49], want_logits=False)
        b.prefill(rows[49:128], pos_start=49, want_logits=False)
        parts, tok_p = b.prefill(rows[128:], pos_start=128)
        # same arithmetic per token row; only the attention's key-block boundaries move with the chunking
        assert parity_violations(parts, whole, 1e-3) == 0
        cpu = oracle.OracleModel(cfg, w, kv_f16=True)
        _check(parts, _oracle_logits(cpu, rows), tok_p)
    finally:
        a.close()
        b.close()


def test_prefill_then_long_greedy_decode_tracks_oracle(backend):
    cfg = dict(SMALL, fmt=Q1)
    w = synth.make_model(cfg, 55)
    cpu = oracle.OracleModel(cfg, w, kv_f16=True)
    gpu = HipModel(backend, cfg, w)
    try:
        n = 40
        rows = _rows(9, n, cfg["h"])
        got, tok = gpu.prefill(rows)
        want = _oracle_logits(cpu, rows)
        _check(got, want, tok)
        agree = decided = 0
        for step in range(64):      # free-running: the GPU's token feeds both sides
            r = synth.embedding_rows(9, [tok], cfg["h"])[0] * 50.0
            want = cpu.forward(r, n + step)
            g, t = gpu.forward(r, n + step)
            assert parity_violations(g[0], want, PREFILL_TOL) == 0
            top2 = np.sort(want)[-2:]
            if top2[1] - top2[0] > 2 * PREFILL_TOL * max(1.0, abs(top2[1])):
                decided += 1
                agree += int(t[0] == oracle.argmax_first(want))
            tok = int(t[0])
        assert agree == decided and decided > 32
    finally:
        gpu.close()


def test_prefill_into_one_sequence_of_a_batch(backend):
    cfg = dict(TINY, fmt=TQ2)
    w = synth.make_model(cfg, 3)
    gpu = HipModel(backend, cfg, w, batch=2)
    solo = HipModel(backend, cfg, w, batch=1)
    try:
        rows0, rows1 = _rows(1, 20, cfg["h"]), _rows(2, 20, cfg["h"])
        l0, _ = gpu.prefill(rows0, seq=0)
        l1, _ = gpu.prefill(rows1, seq=1)
        s0, _ = solo.prefill(rows0)
        assert np.array_equal(l0, s0)
        s1, _ = solo.prefill(rows1)
        assert np.array_equal(l1, s1)
        # one batched decode step over both caches
        step = np.stack([_rows(3, 1, cfg["h"])[0], _rows(4, 1, cfg["h"])[0]])
        got, _ = gpu.forward(step, [20, 20])
        solo.prefill(rows0)
        w0, _ = solo.forward(step[0], 20)
        assert parity_violations(got[0], w0[0], 1e-3) == 0
    finally:
        gpu.close()
        solo.close()


def test_prefill_validation(backend):
    cfg = dict(TINY, fmt=Q1)
    gpu = HipModel(backend, cfg, synth.make_model(cfg, 4))
    try:
        rows = _rows(1, 10, cfg["h"])
        with pytest.raises(GpuError) as e:
            gpu.prefill(rows, pos_start=60)          # 60 + 10 > max_seq 64
        assert e.value.kind == "InvalidArgument"
        with pytest.raises(GpuError) as e:
            gpu.prefill(rows, seq=1)
        assert e.value.kind == "InvalidArgument"
        with pytest.raises(GpuError) as e:
            gpu.prefill(rows[:0])
        assert e.value.kind == "InvalidArgument"
    finally:
        gpu.close()


def _scaled(fmt, blocks, k, rows, by, block=slice(None)):
    """Some rows of a matrix `by` times as large (or one block of 128 weights of each)."""
    b = np.array(blocks, copy=True).reshape(-1, k // 128, 18 if fmt == Q1 else 34)
    at = 0 if fmt == Q1 else 32
    d = b[rows, block, at:at + 2].copy().view(np.float16)
    b[rows, block, at:at + 2] = (d * np.float16(by)).view(np.uint8)
    return b.reshape(-1)


def _louder(fmt, blocks, k, row, by):
    """One row of a matrix `by` times as large."""
    return _scaled(fmt, blocks, k, [row], by)


def _second_layer_errors(backend, cfg, w, rows, ctx, batch):
    """K and V rows of layer 1 behind `ctx` tokens against the oracle's: relative error of each.  The rows from ctx on are the rest of the
    prompt, or (batch > 1) one further position of each sequence."""
    n = 1 if batch > 1 else len(rows) - ctx
    cpu = oracle.OracleModel(cfg, w, kv_f16=True, simd=True)
    gpu = HipModel(backend, cfg, w, batch=batch)
    err = []
    try:
        for seq in range(batch):
            if ctx:
                gpu.prefill(rows[:ctx], 0, seq=seq, want_logits=False)
        if batch > 1:
            gpu.forward(rows[ctx:], ctx)
        else:
            gpu.prefill(rows[ctx:], ctx)
        if ctx:
            cpu.forward_batch(rows[:ctx], 0, want_logits=False)
        for seq in range(batch):
            cpu.forward_batch(rows[ctx + seq:ctx + seq + n], ctx, want_logits=False)
            for head in range(cfg["nkv"]):
                for a, b in zip(gpu.read_kv(1, head, ctx, n, seq=seq)[:2], cpu.cache_rows(1, head, ctx, n)):
                    d = a.astype(np.float64) - b
                    err += list(np.sqrt(np.mean(d * d, axis=1) / np.mean(b.astype(np.float64) ** 2, axis=1)))
    finally:
        gpu.close()
    print(f"median row {np.median(err):.2e}, worst {max(err):.2e}")
    return np.array(err)


# tokens in front, tokens (of each of `batch` sequences a single one where batch > 1), head_dim, size of the hidden rows
HANDED_ON = [(0, 1, 1, 64, 1.0), (0, 17, 1, 32, 1.0), (0, 130, 1, 128, 1e-4), (0, 33, 1, 256, 1e3), (1600, 21, 1, 128, 1.0), (1600, 50, 1, 64, 1.0),
             (60, 1, 9, 128, 1.0), (300, 1, 17, 64, 1e3), (300, 1, 10, 128, 1e-4)]


@pytest.mark.parametrize("fmt", [Q1, TQ2])
@pytest.mark.parametrize("loud", [1, 6, 16])
@pytest.mark.parametrize("ctx,n,batch,hd,size", HANDED_ON)
def test_operands_handed_on_keep_their_precision(backend, fmt, ctx, n, batch, hd, size, loud):
    """The attention and the SwiGLU product leave the next product's fp16 operand under a power of two that comes from bounds,
    not from the values: with weight rows up to as much louder than the rest as is handed on (and about as much as is not: the scales
    differ by themselves) and a norm weight forty times (which meets zeros), which push the bounds above what is met, and rows of very
    different size.  The rows of the second layer have seven fp16 roundings behind them (7e-4, as in the test above): twice that for the
    median row (of nkv heads' K and V, n tokens or `batch` sequences).  A single row may also see its attention scores, of size up to
    sqrt(hd) between normalised vectors, off by the 4e-4 of two roundings of q and k.
    inter = 9 blocks: three blocks of the operand are padding."""
    nq = 1024 // hd
    cfg = dict(fmt=fmt, n_layers=2, h=512, inter=1152, nq=nq, nkv=nq // 4, hd=hd, vocab=64, max_seq=ctx + n + 8, eps=1e-6, rope_theta=1e6)
    w = synth.make_model(cfg, 900 + ctx + n)
    for lw in w["layers"]:
        lw["gate"], lw["up"] = _louder(fmt, lw["gate"], 512, 3, loud), _louder(fmt, lw["up"], 512, 700, loud)
        lw["v"] = _louder(fmt, lw["v"], 512, 1, loud)
        lw["ffn_norm"] = lw["ffn_norm"].copy()
        lw["ffn_norm"][7] = 40.0
    w["layers"][0]["attn_norm"] = w["layers"][0]["attn_norm"].copy()
    w["layers"][0]["attn_norm"][7] = 40.0
    rows = _rows(31, ctx + n * batch, 512) * np.float32(size)
    rows[:, 7] = 0.0
    err = _second_layer_errors(backend, cfg, w, rows, ctx, batch)
    assert np.median(err) <= 1.4e-3 and max(err) <= 3 * (7e-4 + 4e-4 * np.sqrt(hd))


# What is uneven: a gate row `loud` times the rest beside an up row as much quieter; or a gate row alone, whose output the down projection
# takes as much quieter (its block of 128), so that the other outputs are what counts
@pytest.mark.parametrize("fmt", [Q1, TQ2])
@pytest.mark.parametrize("ctx,n,batch,hd", [(0, 130, 1, 64), (0, 17, 1, 128), (60, 1, 9, 128)])
@pytest.mark.parametrize("loud", [256, 2048])
@pytest.mark.parametrize("what", ["gate and up", "gate and down"])
def test_uneven_rows_leave_the_other_outputs_their_precision(backend, fmt, ctx, n, batch, hd, loud, what):
    """SwiGLU outputs keep fp16's eleven bits however much louder than the rest one row of gate or up is: seven fp16 roundings lie in
    front of the second layer's rows (7e-4), twice that for the median row."""
    nq = 1024 // hd
    cfg = dict(fmt=fmt, n_layers=2, h=512, inter=1152, nq=nq, nkv=nq // 4, hd=hd, vocab=64, max_seq=ctx + n + 8, eps=1e-6, rope_theta=1e6)
    w = synth.make_model(cfg, 77 + loud)
    for lw in w["layers"]:
        lw["gate"] = _scaled(fmt, lw["gate"], 512, [3], loud)
        if what == "gate and up":
            lw["up"] = _scaled(fmt, lw["up"], 512, [3], 1 / loud)
        else:
            lw["down"] = _scaled(fmt, lw["down"], 1152, slice(None), 1 / loud, block=0)
    err = _second_layer_errors(backend, cfg, w, _rows(31, ctx + n * batch, 512), ctx, batch)
    assert np.median(err) <= 1.4e-3


# One residual of 1e18 where the FFN's norm weight is 20: the sum of the squares in front of the division by the root mean square is
# beyond fp32's range, the normalised activations are not.  Rows of 1e-22 with an eps to match and norm weights of 0.01: their squares are 0.
@pytest.mark.parametrize("fmt", [Q1, TQ2])
@pytest.mark.parametrize("n,batch", [(1, 1), (21, 1), (70, 1), (1, 9)])
@pytest.mark.parametrize("case", ["loud", "quiet"])
def test_swiglu_outputs_of_rows_at_the_ends_of_the_range(backend, fmt, n, batch, case):
    """The logits have a few fp16 roundings of the FFN's values behind them, 2^-12 of each at most: 1e-3 of the row."""
    cfg = dict(fmt=fmt, n_layers=1, h=512, inter=1152, nq=8, nkv=2, hd=64, vocab=96, max_seq=n + 8, eps=1e-6 if case == "loud" else 2e-38, rope_theta=1e6)
    w = synth.make_model(cfg, 5)
    lw, rows = w["layers"][0], _rows(17, n * batch, 512)
    if case == "loud":
        rows[:, 5] = 1e18
        lw["ffn_norm"] = lw["ffn_norm"].copy()
        lw["ffn_norm"][5] = 20.0
        w["final_norm"] = w["final_norm"].copy()
        w["final_norm"][5] = 0.0           # the logits are those of the other 511 values
    else:
        rows *= np.float32(1e-22)
        lw["ffn_norm"] = lw["ffn_norm"] * np.float32(0.01)
        lw["o"] = _scaled(fmt, lw["o"], 512, slice(None), 0.0)
    cpu = oracle.OracleModel(cfg, w, kv_f16=True)
    gpu = HipModel(backend, cfg, w, batch=batch)
    try:
        got = gpu.forward(rows, 0)[0] if batch > 1 else gpu.prefill(rows, 0)[0][None]
        for b in range(batch):
            want = cpu.forward(rows[b], 0) if batch > 1 else _oracle_logits(cpu, rows)
            err = np.sqrt(np.mean((got[b].astype(np.float64) - want) ** 2) / np.mean(want.astype(np.float64) ** 2))
            print(f"{err:.2e}")
            assert err <= 1e-3
    finally:
        gpu.close()


# What is uneven: a value row `loud` times the rest, whose outputs the O projection takes as much quieter; or a norm weight in front of
# Q || K || V that meets zeros
@pytest.mark.parametrize("fmt", [Q1, TQ2])
@pytest.mark.parametrize("ctx,n,batch,hd", [(0, 130, 1, 64), (0, 17, 1, 128), (1600, 40, 1, 128), (60, 1, 9, 128)])
@pytest.mark.parametrize("what", ["value row", "norm weight", "both"])
def test_uneven_value_rows_leave_the_attention_its_precision(backend, fmt, ctx, n, batch, hd, what):
    """The same for the attention's outputs in front of the O projection; the FFN is silent, so that they are what the second layer's
    rows are made of."""
    nq, loud = 1024 // hd, 2048
    cfg = dict(fmt=fmt, n_layers=2, h=512, inter=512, nq=nq, nkv=nq // 4, hd=hd, vocab=64, max_seq=ctx + n + 8, eps=1e-6, rope_theta=1e6)
    w = synth.make_model(cfg, 78)
    rows = _rows(32, ctx + n * batch, 512)
    for lw in w["layers"]:
        lw["down"] = _scaled(fmt, lw["down"], 512, slice(None), 0.0)
        if what != "norm weight":
            lw["v"] = _scaled(fmt, lw["v"], 512, [3], loud)
            lw["o"] = _scaled(fmt, lw["o"], 1024, slice(None), 1 / loud, block=slice(0, 4 * hd // 128))   # its four q heads
        if what != "value row":
            lw["attn_norm"] = lw["attn_norm"].copy()
            lw["attn_norm"][7] = 2.0 ** 24
    if what != "value row":
        rows[:, 7] = 0.0
        for lw in w["layers"]:
            lw["o"] = _scaled(fmt, lw["o"], 1024, [7], 0.0)
    err = _second_layer_errors(backend, cfg, w, rows, ctx, batch)
    assert np.median(err) <= 1.4e-3


@pytest.mark.parametrize("fmt", [Q1, TQ2])
@pytest.mark.parametrize("n,batch", [(40, 1), (1, 9)])
def test_quieter_value_rows_in_place_of_loud_ones(backend, fmt, n, batch):
    """Q || K || V of a live model is replaced by one whose value rows are 2^24 times as quiet: what the old ones could reach says nothing
    about the new ones' precision."""
    cfg = dict(fmt=fmt, n_layers=2, h=512, inter=512, nq=8, nkv=2, hd=128, vocab=64, max_seq=n + 8, eps=1e-14, rope_theta=1e6)
    w = synth.make_model(cfg, 79)
    for lw in w["layers"]:
        lw["down"] = _scaled(fmt, lw["down"], 512, slice(None), 0.0)
    quiet = {**w, "layers": [{**lw, "v": _scaled(fmt, lw["v"], 512, slice(None), 1 / 4096)} for lw in w["layers"]]}
    loud = {**w, "layers": [{**lw, "v": _scaled(fmt, lw["v"], 512, slice(None), 4096)} for lw in w["layers"]]}
    rows = _rows(33, n * batch, 512) * np.float32(1e-5)
    cpu = oracle.OracleModel(cfg, quiet, kv_f16=True, simd=True)
    gpu = HipModel(backend, cfg, loud, batch=batch)
    try:
        up = backend.upload_weights_raw if fmt == Q1 else backend.upload_weights_ternary
        run = (lambda: gpu.forward(rows, 0)) if batch > 1 else (lambda: gpu.prefill(rows, 0))
        run()
        for i, lw in enumerate(quiet["layers"]):
            up(np.concatenate([lw["q"], lw["k"], lw["v"]]), 1536, 512, handle_id=gpu._ids[i].qkv)
        run()
        err = []
        for seq in range(batch):
            cpu.forward_batch(rows[seq:seq + n], 0, want_logits=False)
            for head in range(2):
                for a, b in zip(gpu.read_kv(1, head, 0, n, seq=seq)[:2], cpu.cache_rows(1, head, 0, n)):
                    err += list(np.sqrt(np.mean((a.astype(np.float64) - b) ** 2, axis=1) / np.mean(b.astype(np.float64) ** 2, axis=1)))
        print(f"median row {np.median(err):.2e}, worst {max(err):.2e}")
        assert np.median(err) <= 1.4e-3
    finally:
        gpu.close()


def _free_bytes():
    import ctypes as C
    from oxibonsai_amd import _lib
    free, total = C.c_size_t(0), C.c_size_t(0)
    assert _lib.lib().oxb_hip_device_info(None, 0, C.byref(free), C.byref(total)) == 0
    return free.value


def test_buffers_that_a_prefill_has_no_use_for(backend):
    """Where SwiGLU outputs and attention outputs go to the next product's operand their fp32 rows take no memory: 2048 tokens x (24576 +
    1024) values, 210 MB.  What a prefill allocates is the operand in fp16 (with a quarter to spare), the projections and smaller things.
    A layer that is uneven all of a sudden gets its rows."""
    cfg = dict(fmt=Q1, n_layers=2, h=128, inter=24576, nq=8, nkv=2, hd=128, vocab=64, max_seq=2100, eps=1e-6, rope_theta=1e6)
    w = synth.make_model(cfg, 6)
    uneven = {**w, "layers": [dict(w["layers"][0], gate=_scaled(Q1, w["layers"][0]["gate"], 128, [9], 64),
                                   v=_scaled(Q1, w["layers"][0]["v"], 128, [9], 64)), w["layers"][1]]}
    rows = _rows(7, 2048, 128)
    gpu, other = HipModel(backend, cfg, w), HipModel(backend, cfg, uneven)
    try:
        before = _free_bytes()
        gpu.prefill(rows)
        used = before - _free_bytes()
        print(f"{used / 2**20:.0f} MiB")
        assert used <= 2048 * (1.25 * 2 * (24576 + 1024) + 4 * (1536 + 128)) + (32 << 20)   # (sums of K slices and what rounding up adds)
        lw = uneven["layers"][0]
        backend.upload_weights_raw(np.concatenate([lw["gate"], lw["up"]]), 2 * 24576, 128, handle_id=gpu._ids[0].gate_up)
        backend.upload_weights_raw(np.concatenate([lw["q"], lw["k"], lw["v"]]), 1536, 128, handle_id=gpu._ids[0].qkv)
        assert np.array_equal(gpu.prefill(rows)[0], other.prefill(rows)[0])
    finally:
        gpu.close()
        other.close()
