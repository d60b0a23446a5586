"""GPU parity of the prefill kernels at the edges of their dispatch rules, against the CPU oracle."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from gpu_util import assert_bits_equal, dev, host

pytestmark = pytest.mark.gpu
F32 = np.float32


@pytest.mark.parametrize("pos0,rows,qs_lo,qs_hi", [
    (192, 64, 0.01, 0.05),      # 256 keys: the last context of 4 one-block wavefronts
    (193, 64, 1e-4, 2e-4),      # 257 keys, nearly flat scores: every probability near 127 / 257
    (448, 64, 0.002, 0.01),     # 512 keys: the last of 8 wavefronts
    (449, 64, 0.002, 0.01),     # 513 keys: 16 wavefronts
    (991, 33, 0.001, 0.05),     # 1024 keys, a one-row second tile: the last of 16
    (992, 33, 0.001, 0.05),     # 1025 keys: scores recomputed per pass, 16 wavefronts
    (760, 265, 0.001, 0.05),    # more than 256 tiles: 8 wavefronts
    (0, 1024, 0.0005, 0.02),    # 1024 tiles: 4 wavefronts, wavefronts without a block in the first tiles
    (2031, 17, 0.0005, 0.002),  # the end of the context
])
def test_attention_tile_wavefront_counts(pos0, rows, qs_lo, qs_hi):
    """tl_attention at both sides of every change of kernel or of its
    wavefront count, with score scales from nearly flat rows (probabilities of
    one or two 127ths, or all zero) to rows of a few large ones: the oracle's
    rows bit for bit."""
    cfg = dict(oracle.TINYLLAMA_CFG, n_layers=1, vocab=64)
    from lpta.engine import Engine
    eng = Engine(cfg, max_seqs=1)
    rng = np.random.default_rng(pos0 + 7 * rows)
    hkv, d = cfg["n_kv_heads"], cfg["hidden"]
    sk = rng.uniform(0.02, 0.06, (1, hkv)).astype(F32)
    sv = rng.uniform(0.02, 0.06, (1, hkv)).astype(F32)
    eng.set_kv_scales(sk, sv)
    kc = np.zeros((1, hkv, cfg["max_pos"], 64), np.int8)
    vc = np.zeros_like(kc)
    n = pos0 + rows
    for g in range(hkv):
        kc[0, g, :n] = rng.integers(-127, 128, (n, 64))
        vc[0, g, :n] = rng.integers(-127, 128, (n, 64))
        eng.kv_write(0, 0, g, 0, kc[0, g, :n], vc[0, g, :n])
    q8 = rng.integers(-127, 128, (rows, d)).astype(np.int8)
    qs = np.exp(rng.uniform(np.log(qs_lo), np.log(qs_hi), rows))
    out = dev(np.zeros((rows, d), F32))
    eng.rt.call("tl_attention", 0, 0, pos0, rows, dev(q8), dev(qs), out)
    got = host(out)
    for r in range(rows) if rows < 500 else list(range(0, rows, 13)) + [rows - 1]:
        want = oracle.attention_row(cfg, 0, pos0 + r, q8[r], qs[r], kc, vc, sk, sv)
        assert_bits_equal(got[r], want, f"row {r} (position {pos0 + r})")
    eng.close()


@pytest.mark.parametrize("pos0,rows", [(3, 40), (300, 45), (700, 40), (1100, 40), (760, 265), (0, 1024)])
def test_attention_takes_negative_row_scales(pos0, rows):
    """Each tile kernel with the caller's own row scales of both signs in one
    tile (the largest product is then the smallest score's): the oracle's rows
    bit for bit."""
    cfg = dict(oracle.TINYLLAMA_CFG, n_layers=1, vocab=64)
    from lpta.engine import Engine
    eng = Engine(cfg, max_seqs=1)
    rng = np.random.default_rng(pos0 + rows)
    hkv, d, n = cfg["n_kv_heads"], cfg["hidden"], pos0 + rows
    sk, sv = np.full((1, hkv), 0.03, F32), np.full((1, hkv), 0.05, F32)
    eng.set_kv_scales(sk, sv)
    kc = np.zeros((1, hkv, cfg["max_pos"], 64), np.int8)
    vc = np.zeros_like(kc)
    for g in range(hkv):
        kc[0, g, :n] = rng.integers(-127, 128, (n, 64))
        vc[0, g, :n] = rng.integers(-127, 128, (n, 64))
        eng.kv_write(0, 0, g, 0, kc[0, g, :n], vc[0, g, :n])
    q8 = rng.integers(-127, 128, (rows, d)).astype(np.int8)
    # products up to about 300: exponents of the wrong sign would overflow
    qs = np.exp(rng.uniform(np.log(0.001), np.log(0.5), rows)) * rng.choice([-1.0, 1.0], rows)
    qs[:2] = -0.5, 0.0
    out = dev(np.zeros((rows, d), F32))
    eng.rt.call("tl_attention", 0, 0, pos0, rows, dev(q8), dev(qs), out)
    got = host(out)
    for r in range(rows) if rows < 100 else list(range(0, rows, 13)) + [1, rows - 1]:
        want = oracle.attention_row(cfg, 0, pos0 + r, q8[r], qs[r], kc, vc, sk, sv)
        assert_bits_equal(got[r], want, f"row {r} (position {pos0 + r})")
    eng.close()
