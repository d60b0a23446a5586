"""Row-major INT8 GEMM tiles at both sides of their size rule, against exact integer products."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from gpu_util import assert_bits_equal, dev, empty, host, runtime

pytestmark = pytest.mark.gpu
F32 = np.float32


@pytest.fixture(scope="module")
def rt():
    r = runtime()
    yield r
    r.close()


@pytest.mark.parametrize("m,n,k", [
    (2048, 2048, 128),    # 128 x 128 tiles, one round, two 64-byte stages
    (1999, 2017, 256),    # ... ragged rows and columns
    (1999, 2081, 256),    # five rounds of 64 x 64 tiles against two: 64 x 64, ragged
    (65, 32000, 128),     # 128 x 128, the second row half of every tile nearly empty
    (2048, 2560, 384),    # just below the rule: 64 x 64 tiles
    (1100, 2048, 128),    # three rounds against one: 64 x 64
    (333, 9000, 1152),    # 128 x 128, one ragged round
    (64, 64, 128),
])
def test_gemm_tile_sizes(rt, m, n, k):
    """INT32 sums, the dequantized product and the product added to a residual equal the
    definition (exact integers; float64 scale product rounded once, one float32
    multiplication, one addition)."""
    rng = np.random.default_rng(m + n + k)
    a = rng.integers(-127, 128, (m, k)).astype(np.int8)
    w = rng.integers(-127, 128, (n, k)).astype(np.int8)
    s_a, s_w = rng.uniform(1e-3, 1e-1, m), rng.uniform(1e-4, 1e-2, n).astype(F32)
    res = rng.standard_normal((m, n)).astype(F32)
    want = (a.astype(F32) @ w.astype(F32).T).astype(np.int64)   # |sum| <= 127^2 k < 2^24 for k <= 1040
    if k > 1040:
        want = a.astype(np.float64) @ w.astype(np.float64).T
    want = want.astype(np.int32)
    da, dw = dev(a), dev(w)
    acc = empty((m, n), np.int32)
    rt.call("tl_gemm_i8", da, dw, m, n, k, acc)
    assert np.array_equal(host(acc), want)
    y = empty((m, n), F32)
    rt.call("tl_gemm_i8_dequant", da, dev(s_a), dw, dev(s_w), m, n, k, None, y)
    deq = want.astype(F32) * (s_a[:, None] * s_w.astype(np.float64)[None, :]).astype(F32)
    assert_bits_equal(host(y), deq, "dequantized")
    rt.call("tl_gemm_i8_dequant", da, dev(s_a), dw, dev(s_w), m, n, k, dev(res), y)
    assert_bits_equal(host(y), res + deq, "with residual")


def _large_tiles(m, n):
    """The size rule of the row-major tiles: 128 x 128 where 64 x 64 ones need at
    least four rounds of the 256 CUs, and three for each round of theirs."""
    r64, r128 = (-(-(-(-n // t) * -(-m // t)) // 256) for t in (64, 128))
    return r64 >= 4 and r64 >= 3 * r128


@pytest.mark.parametrize("B,vocab,large", [
    (33, 2048, False), (40, 32000, False), (129, 24000, False),   # 1, 2 and 5 rounds (5 against 2)
    (65, 32000, True), (90, 32000, True),                         # 4 rounds against 1
    (129, 32000, True),                                           # 6 against 2, one row in the second row tile
])
def test_many_row_lm_head_ties(B, vocab, large):
    """The LM head over more than 32 rows takes the argmax in its tiles: with
    every head row repeated once in the same 32 columns and once far away, equal
    logits resolve to the lowest id, in 64 x 64 and in 128 x 128 tiles."""
    assert _large_tiles(B, vocab) == large
    from lpta.engine import Engine
    cfg = dict(oracle.SMALL_CFG, n_layers=1, vocab=vocab)
    m = oracle.synthetic_model(cfg, seed=B)
    half = vocab // 2
    for src, dst in ((slice(0, half, 2), slice(1, half, 2)), (slice(0, half), slice(half, vocab))):
        m.lm_w[dst] = m.lm_w[src]
        m.lm_s[dst] = m.lm_s[src]
    eng = Engine(cfg, max_seqs=B).load_model(m)
    rng = np.random.default_rng(1)
    toks = rng.integers(0, vocab, B).astype(np.int32)
    got = eng.decode_batch(toks, np.zeros(B, np.int32), 2)
    assert (got < half).all() and (got % 2 == 0).all()
    # one by one: the batch-1 head
    for b in (0, B // 2, B - 1):
        one = eng.decode_batch(toks[b:b + 1], np.zeros(1, np.int32), 2)
        assert_bits_equal(one[0], got[b], f"sequence {b}")
    eng.close()
