"""GPU parity between the 32-row tile and the large tiles: batches and prompts of 33 to 300 rows, and the context
bounds of the batched attention."""
from __future__ import annotations

import os

import numpy as np
import pytest

import oracle
from gpu_util import assert_bits_equal, dev, host

pytestmark = pytest.mark.gpu
F32 = np.float32


def _fill(eng, cfg, seq, n, rng, kc, vc):
    for layer in range(cfg["n_layers"]):
        for g in range(cfg["n_kv_heads"]):
            kc[layer, g, :n] = np.clip(np.rint(rng.standard_normal((n, 64)) * 25), -127, 127)
            vc[layer, g, :n] = np.clip(np.rint(rng.standard_normal((n, 64)) * 25), -127, 127)
            eng.kv_write(seq, layer, g, 0, kc[layer, g, :n], vc[layer, g, :n])


@pytest.mark.parametrize("B,top", [(33, 505), (64, 1017), (90, 300), (128, 70), (129, 90), (3, 510)])
def test_decode_batch_rows_and_context_bounds(B, top):
    """Batches past 32 rows (32 x 32 tiles of several row tiles, their last
    one partial; LM-head argmax keys of 64-column tiles) with ragged contexts up
    to `top` cached rows, so that a second call of the same batch crosses the
    bound of 512 or 1024 keys (another captured step, another wavefront count
    of the grouped attention): ids and appended K/V rows equal the oracle's."""
    from lpta.engine import Engine
    cfg = dict(oracle.TINYLLAMA_CFG, n_layers=1, vocab=512)
    m = oracle.synthetic_model(cfg, seed=70 + B)
    eng = Engine(m.cfg, max_seqs=B).load_model(m)
    rng = np.random.default_rng(B)
    start = rng.integers(max(1, top - 60), top + 1, B).astype(np.int32)
    start[0], start[-1] = top, 1
    toks = rng.integers(0, cfg["vocab"], B).astype(np.int32)
    caches = []
    for b in range(B):
        kc, vc = m.new_cache()
        _fill(eng, cfg, b, int(start[b]), rng, kc, vc)
        caches.append((kc, vc))
    oracle.lib().or_set_threads(max(1, min(16, len(os.sched_getaffinity(0)))))
    orc = oracle.Oracle(m)
    pos, tok = start.copy(), toks
    for steps in (3, 5):   # one eager step and replays; the second call ends past the bound for top = 505, 1017, 510
        got = eng.decode_batch(tok, pos, steps)
        for s in range(steps):
            x = np.stack([orc.embed(int(t)) for t in tok]).astype(F32)
            orc.decode_rows(0, pos, x, caches)
            tok, _ = orc.lm_head_rows(x)
            tok = np.asarray(tok, np.int32)
            assert_bits_equal(np.asarray(got[:, s], np.int32), tok, f"ids of step {s}")
            pos = pos + 1
    for b in (0, 1, 31, 32, B // 2, B - 1):
        if b >= B:
            continue
        kc, vc = caches[b]
        n = int(pos[b])
        for g in range(cfg["n_kv_heads"]):
            k, v = eng.kv_read(b, 0, g, 0, n)
            assert_bits_equal(k, kc[0, g, :n], f"K seq {b} head {g}")
            assert_bits_equal(v, vc[0, g, :n], f"V seq {b} head {g}")
    eng.close()


def test_decode_batch_sizes_alternate_on_one_engine():
    """Captured batch steps stay valid when the split-K scratch moves: on one
    engine, batches of 4, 40 (split-K projections: this intermediate width has no packed
    form), 60 and a scored prompt of 63 tokens, each needing more scratch than
    the one before, and then 4 and 40 again give the oracle's ids."""
    from lpta.engine import Engine
    cfg = dict(oracle.SMALL_CFG)
    m = oracle.synthetic_model(cfg, seed=91)
    eng = Engine(m.cfg, max_seqs=60).load_model(m)
    orc = oracle.Oracle(m)
    rng = np.random.default_rng(91)
    toks = rng.integers(0, cfg["vocab"], 60).astype(np.int32)
    steps = 4   # an eager one and three replays
    caches = [m.new_cache() for _ in range(60)]
    want, tok = [], toks
    for p in range(steps):   # sequences of a batch are independent: the first B of 60
        x = np.stack([orc.embed(int(t)) for t in tok]).astype(F32)
        for layer in range(cfg["n_layers"]):
            orc.decode_rows(layer, np.full(60, p, np.int32), x, caches)
        tok, _ = orc.lm_head_rows(x)
        tok = np.asarray(tok, np.int32)
        want.append(tok)
    want = np.stack(want, 1)
    logits = dev(np.zeros((63, cfg["vocab"]), F32))
    for b in (4, 40, 60, None, 4, 40, 60):
        if b is None:
            eng.rt.call("tl_prefill_logits", 0, rng.integers(0, cfg["vocab"], 63).astype(np.int32), 63, logits)
            continue
        got = eng.decode_batch(toks[:b], np.zeros(b, np.int32), steps)
        assert_bits_equal(np.asarray(got, np.int32), want[:b], f"batch of {b}")
    eng.close()


@pytest.fixture(scope="module")
def layer_eng():
    from lpta.engine import Engine
    e = Engine(dict(oracle.TINYLLAMA_CFG, n_layers=1, vocab=64), max_seqs=2)
    e.load_random(11)
    yield e
    e.close()


@pytest.mark.parametrize("rows", [32, 33, 63, 64, 65, 128, 129, 256, 257, 300, 384, 385])
def test_layer_rows_equal_single_rows(layer_eng, rows):
    """Both sides of every row count at which a projection changes kernel: the
    layer over all rows equals the single-row kernels run row after row on
    another sequence, output and cache."""
    d = oracle.TINYLLAMA_CFG["hidden"]
    x = np.random.default_rng(rows).standard_normal((rows, d)).astype(F32)
    xs = dev(x)
    layer_eng.rt.call("tl_layer_rows", 0, 0, 0, rows, xs)
    got = host(xs)
    one = dev(x)
    for r in range(rows):
        layer_eng.decode_layer(one[r], 0, r, seq=1)
    assert_bits_equal(got, host(one), f"{rows} rows")
    for g in range(4):
        for a, b in zip(layer_eng.kv_read(0, 0, g, 0, rows), layer_eng.kv_read(1, 0, g, 0, rows)):
            assert_bits_equal(a, b, f"cache head {g}")


@pytest.mark.parametrize("pos", [1, 511, 512, 700, 1023, 1024, 1535, 2046])
def test_single_row_attention_wavefront_counts(layer_eng, pos):
    """Batch-1 attention at both sides of its context bounds (4, 8 and 16
    wavefronts): two rows at pos, pos + 1 one by one equal the two rows as one
    block, which the prefill attention computes."""
    rng = np.random.default_rng(pos)
    for g in range(4):
        k, v = (np.clip(np.rint(rng.standard_normal((pos, 64)) * 25), -127, 127).astype(np.int8) for _ in range(2))
        layer_eng.kv_write(0, 0, g, 0, k, v)
        layer_eng.kv_write(1, 0, g, 0, k, v)
    x = rng.standard_normal((2, oracle.TINYLLAMA_CFG["hidden"])).astype(F32)
    both, one = dev(x), dev(x)
    layer_eng.rt.call("tl_layer_rows", 0, 0, pos, 2, both)
    for r in range(2):
        layer_eng.decode_layer(one[r], 0, pos + r, seq=1)
    assert_bits_equal(host(one), host(both), f"rows at {pos}, {pos + 1}")
    for g in range(4):
        for a, b in zip(layer_eng.kv_read(0, 0, g, pos, 2), layer_eng.kv_read(1, 0, g, pos, 2)):
            assert_bits_equal(a, b, f"cache head {g}")


@pytest.mark.parametrize("n,new", [(500, 30), (1015, 25)])
def test_decode_crosses_a_context_bound(n, new):
    """One decode call whose steps pass 512 or 1024 keys (another captured
    step from there on) writes the K/V rows that a prefill of the whole
    sequence writes, and predicts the same next token."""
    from lpta.engine import Engine
    eng = Engine(dict(oracle.TINYLLAMA_CFG, n_layers=2, vocab=4096), max_seqs=2)
    eng.load_random(3)
    prompt = np.random.default_rng(n).integers(0, 4096, n).astype(np.int32)
    first, _ = eng.prefill(prompt, seq=0)
    got, _ = eng.decode(new, seq=0)
    fed = np.concatenate([prompt, [first], got[:-1]]).astype(np.int32)
    nxt, _ = eng.prefill(fed, seq=1)
    assert nxt == got[-1]
    for layer in range(2):
        for g in range(4):
            for a, b in zip(eng.kv_read(0, layer, g, 0, fed.size), eng.kv_read(1, layer, g, 0, fed.size)):
                assert_bits_equal(a, b, f"layer {layer} head {g}")
    eng.close()


@pytest.mark.parametrize("n,off", [(2, None), (5, None), (31, None), (32, None), (33, None), (20, "TL_BATCH_O_FUSE"),
                                   (20, "TL_BATCH_KSLICE")])
def test_short_prompt_chains_layers(monkeypatch, n, off):
    """Prompts of up to 32 rows leave each layer's down projection as integer sums that the next layer's RMSNorm
    folds, and the last layer's complete (and the forms with these fusions switched off): the logits of every position, the caches of all layers and a single-layer
    call after the prompt equal the oracle's."""
    from lpta.engine import Engine
    if off:
        monkeypatch.setenv(off, "0")
    cfg = dict(oracle.TINYLLAMA_CFG, n_layers=3, vocab=512)
    m = oracle.synthetic_model(cfg, seed=500 + n)
    eng = Engine(m.cfg, max_seqs=1).load_model(m)
    orc = oracle.Oracle(m)
    rng = np.random.default_rng(n)
    toks = rng.integers(0, cfg["vocab"], n).astype(np.int32)
    kc, vc = m.new_cache()
    want = []
    for p, t in enumerate(toks):
        x = orc.embed(int(t)).astype(F32)
        for layer in range(cfg["n_layers"]):
            x = orc.decode_row(layer, p, x, kc, vc)
        want.append(np.asarray(orc.lm_head(x, want_logits=True)[2], F32))
    logits = dev(np.zeros((n, cfg["vocab"]), F32))
    for _ in range(2):   # the second call finds no sums of the first
        eng.rt.call("tl_prefill_logits", 0, toks, n, logits)
        assert_bits_equal(host(logits), np.stack(want), f"logits of {n} positions")
    for layer in range(cfg["n_layers"]):
        for g in range(cfg["n_kv_heads"]):
            k, v = eng.kv_read(0, layer, g, 0, n)
            assert_bits_equal(k, kc[layer, g, :n], f"K layer {layer} head {g}")
            assert_bits_equal(v, vc[layer, g, :n], f"V layer {layer} head {g}")
    x = rng.standard_normal((2, cfg["hidden"])).astype(F32)
    xs = dev(x)
    eng.rt.call("tl_layer_rows", 0, 1, n, 2, xs)
    rows = [orc.decode_row(1, n + r, x[r].copy(), kc, vc) for r in range(2)]
    assert_bits_equal(host(xs), np.stack(rows), "two rows through one layer")
    eng.close()
