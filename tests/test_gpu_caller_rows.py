"""Entry points that run on the caller's rows: a buffer off 16 bytes (its own route: copied, or other kernels) gives
the bits that an aligned one gives, and rows past the call's stay untouched."""
from __future__ import annotations

import numpy as np
import pytest

import oracle
from gpu_util import assert_bits_equal, host

pytestmark = pytest.mark.gpu
F32 = np.float32


@pytest.fixture(scope="module")
def eng():
    from lpta.engine import Engine
    e = Engine(dict(oracle.SMALL_CFG), max_seqs=1).load_model(oracle.synthetic_model(oracle.SMALL_CFG, seed=5))
    yield e
    e.close()


def _rows(values, shift):
    """values on the device, starting `shift` floats into a larger buffer, with guard values around them."""
    import torch
    buf = torch.full((values.size + 64,), 7.0, device="cuda")
    view = buf[32 + shift:32 + shift + values.size]
    view.copy_(torch.from_numpy(values.ravel()))
    torch.cuda.synchronize()
    return buf, view


@pytest.mark.parametrize("rows,pos0", [(1, 5), (2, 0), (33, 3), (64, 0), (70, 100)])
def test_layer_rows_in_place(eng, rows, pos0):
    d = oracle.SMALL_CFG["hidden"]
    x = np.random.default_rng(rows).standard_normal((rows, d)).astype(F32)
    rng = np.random.default_rng(1)
    for g in range(oracle.SMALL_CFG["n_kv_heads"]):
        if pos0:
            eng.kv_write(0, 1, g, 0, rng.integers(-127, 128, (pos0, 64)).astype(np.int8),
                         rng.integers(-127, 128, (pos0, 64)).astype(np.int8))
    got = []
    for shift in (0, 1, 3):
        buf, view = _rows(x, shift)
        eng.rt.call("tl_layer_rows", 0, 1, pos0, rows, view)
        got.append(host(view))
        b = host(buf)
        assert (b[:32 + shift] == 7.0).all() and (b[32 + shift + x.size:] == 7.0).all()
    assert_bits_equal(got[1], got[0], "one float off")
    assert_bits_equal(got[2], got[0], "three floats off")
    if rows == 1:
        _, view = _rows(x, 1)
        eng.decode_layer(view, 1, pos0)
        assert_bits_equal(host(view), got[0], "tl_decode_layer")


def test_lm_head_argmax_routes(eng):
    import ctypes
    import torch
    d, v = oracle.SMALL_CFG["hidden"], oracle.SMALL_CFG["vocab"]
    x = np.random.default_rng(3).standard_normal(d).astype(F32)
    got = []
    for shift in (0, 2):
        _, view = _rows(x, shift)
        for with_logits in (True, False):
            tok, lg = ctypes.c_int32(), ctypes.c_float()
            logits = torch.full((v,), np.nan, device="cuda") if with_logits else None
            eng.rt.call("tl_lm_head_argmax", view, tok, lg, logits)
            if with_logits:
                got.append(host(logits))
                assert tok.value == int(np.argmax(got[-1])) and F32(lg.value) == got[-1].max()
            else:
                assert tok.value == int(np.argmax(got[-1]))
    assert_bits_equal(got[1], got[0], "logits")
