"""tl_linear_f32 at the edges of its tiles, against 64-bit products."""
from __future__ import annotations

import numpy as np
import pytest

from gpu_util import dev, empty, host, runtime

pytestmark = pytest.mark.gpu
F32, F64 = np.float32, np.float64
EPS32 = float(np.finfo(F32).eps) / 2


@pytest.fixture(scope="module")
def rt():
    r = runtime()
    yield r
    r.close()


@pytest.mark.parametrize("m,k,n,bias,res", [
    (1, 1, 1, False, False), (33, 5, 31, True, True),          # only the last k % 8
    (32, 64, 32, False, False), (31, 63, 33, False, True),     # one chunk per wavefront, ragged everywhere
    (5, 8 * 8 * 9 + 4, 130, True, False),                      # more chunks than are in flight
    (100, 2048, 5632, False, False),                           # 3 column blocks per tile
    (640, 512, 5632, True, True),                              # 4 column blocks per tile
    (170, 2047, 2049, False, False),                           # rows of x off 16 bytes
    (257, 72, 4097, True, True),
])
def test_linear_f32_tiles(rt, m, k, n, bias, res):
    """Every column-block count, ragged rows, columns and K: within k + 3
    float32 roundings of the sum of magnitudes, the bound of any order of k
    fused multiply-adds plus bias and residual."""
    rng = np.random.default_rng(m * 31 + k * 7 + n)
    x = rng.standard_normal((m, k)).astype(F32)
    w = (rng.standard_normal((k, n)) * 0.05).astype(F32)
    b = rng.standard_normal(n).astype(F32) if bias else None
    r = rng.standard_normal((m, n)).astype(F32) if res else None
    y = empty((m, n), F32)
    rt.call("tl_linear_f32", dev(x), dev(w), None if b is None else dev(b), None if r is None else dev(r), m, n, k, y)
    want = x.astype(F64) @ w.astype(F64)
    mag = np.abs(x).astype(F64) @ np.abs(w).astype(F64)
    for extra in (b, r):
        if extra is not None:
            want, mag = want + extra, mag + np.abs(extra)
    assert (np.abs(host(y) - want) <= (k + 3) * EPS32 * mag + 1e-30).all()


def test_linear_f32_special_values(rt):
    """Denormal operands and products keep their bits, infinities and NaN
    reach the outputs their row and column meet and no other."""
    x, w = np.zeros((4, 13), F32), np.zeros((13, 40), F32)
    x[0, 3], w[3, 0] = 1e-40, 1.0
    x[2, 12] = 1e-30
    w[12, :] = 1e-12
    x[1, 5] = np.inf
    w[5, 7] = 2.0
    x[3, 1], w[1, 9] = 3e38, 3.0
    y = empty((4, 40), F32)
    rt.call("tl_linear_f32", dev(x), dev(w), None, None, 4, 40, 13, y)
    got = host(y)
    assert got[0, 0] == F32(1e-40) and got[0, 1] == 0.0
    assert (got[2] == F32(F64(x[2, 12]) * F64(w[12, 0]))).all()
    assert got[1, 7] == np.inf and np.isnan(got[1, 8])   # inf * 0
    assert got[3, 9] == np.inf and got[3, 8] == 0.0


@pytest.mark.parametrize("m,n,k", [
    (32, 1, 138_547_336),    # 31 k = 2^32 + 120: the last row's offset from its tile
    (2, 613_566_760, 8),     # 7 n = 2^32 + 24: the last row of W; 4.8 million column tiles
])
def test_linear_f32_offsets_past_32_bits(rt, m, n, k):
    """Offsets inside a tile that pass 2^32 elements: all-zero operands with a
    few small whole numbers in the first and last rows, columns and k's, whose
    products no other place may show."""
    import torch
    x = torch.zeros((m, k), device="cuda")
    w = torch.zeros((k, n), device="cuda")
    ks = [0, 3, k // 2, k - 2, k - 1]   # distinct from k = 8
    cols = sorted({0, n // 3, n - 1})
    for i, kk in enumerate(ks):
        for r in {0, m - 1}:
            x[r, kk] = 1 + i + 7 * (r > 0)
        for j, c in enumerate(cols):
            w[kk, c] = 2 + 3 * i + 11 * j
    y = torch.full((m, n), 9.0, device="cuda")
    torch.cuda.synchronize()
    rt.call("tl_linear_f32", x, w, None, None, m, n, k, y)
    for r in {0, m - 1}:
        for j, c in enumerate(cols):
            want = sum((1 + i + 7 * (r > 0)) * (2 + 3 * i + 11 * j) for i in range(len(ks)))
            assert float(y[r, c]) == want, (r, c)
            y[r, c] = 0.0
    assert int(torch.count_nonzero(y)) == 0
    del x, w, y
    torch.cuda.empty_cache()


def test_linear_f32_tiles_past_one_grid_dimension(rt):
    """8.4 million tiles of 512 threads, 2^32 threads in one dimension: an
    outer product of small whole numbers, every element compared."""
    import torch
    m, n = 16_777_300, 800   # 524291 row tiles x 9 column tiles of 96, counted as 16
    x = (torch.arange(m, device="cuda") % 251).float().reshape(m, 1)
    w = (torch.arange(n, device="cuda") % 13 + 1).float().reshape(1, n)
    y = torch.empty((m, n), device="cuda")
    torch.cuda.synchronize()
    rt.call("tl_linear_f32", x, w, None, None, m, n, 1, y)
    for i in range(0, m, 1 << 21):
        assert torch.equal(y[i:i + (1 << 21)], x[i:i + (1 << 21)] * w), i
    del x, w, y
    torch.cuda.empty_cache()
