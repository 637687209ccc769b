"""The softcap of the classifier epilogues over the magnitudes at which its form
changes (cap / 6, 0.45 cap) and beyond, for logits and cross-entropy partials,
against float64 tanh of the same fp32-exact logits.

A is diagonal and B selects one of its rows, so each logit is one exact product.
Bounds: the series are within 2^-23 of the value, the exponential form within
3e-7, and the softcapped value is rounded once more (2^-24)."""
import ctypes as C

import numpy as np
import pytest

from ane import _lib

pytestmark = pytest.mark.gpu


def _u16(a):
    return a.view(np.uint16).ctypes.data_as(C.POINTER(C.c_uint16))


def _fp(a):
    return a.ctypes.data_as(C.POINTER(C.c_float))


@pytest.mark.parametrize("top", [0.5, 2.499, 2.51, 6.74, 6.76, 14.0, 40.0, 300.0])
def test_softcap_forms(top):
    lib = _lib.load()
    M = N = K = 256
    r = np.random.default_rng(int(top * 100))
    v = (r.uniform(-top, top, M)).astype(np.float16)
    v[:4] = [0.0, np.float16(top), np.float16(-top), np.float16(1e-4)]
    a = np.zeros((M, K), np.float16)
    a[np.arange(M), np.arange(M)] = v
    b = np.ones((N, K), np.float16)
    b *= np.float16(1)
    x = a.astype(np.float64) @ b.astype(np.float64).T  # each row one value
    ref = 15.0 * np.tanh(x / 15.0)
    out = np.full((M, N), np.nan, np.float32)
    assert lib.ane_debug_gemm_epi(2, M, N, K, _u16(a), _u16(b), out.ctypes.data_as(C.c_void_p), None, None, None, 1.0,
                                  0.0, -1, 0, 0, 0) == 0, lib.ane_debug_last_error()
    assert (np.abs(out - ref) <= 4e-7 * np.abs(ref) + 1e-30).all(), np.abs((out - ref) / np.maximum(np.abs(ref), 1e-30)).max()
    # cross-entropy partials over one 256-row block: max, sum exp, the target's logit
    tgt = r.integers(0, M, N).astype(np.uint16)
    pm, ps, tl = np.zeros((1, N), np.float32), np.zeros((1, N), np.float32), np.zeros(N, np.float32)
    assert lib.ane_debug_classifier(M, N, K, _u16(a), _u16(b), tgt.ctypes.data_as(C.POINTER(C.c_uint16)), 1, M, 256, 256,
                                    8, _fp(pm), _fp(ps), _fp(tl), None, None, None, None) == 0, lib.ane_debug_last_error()
    np.testing.assert_allclose(pm[0], ref.max(0), rtol=4e-7)
    np.testing.assert_allclose(tl, ref[tgt, np.arange(N)], rtol=4e-7)
    lse = np.log(ps[0].astype(np.float64)) + pm[0]
    np.testing.assert_allclose(lse, np.log(np.exp(ref - ref.max(0)).sum(0)) + ref.max(0), rtol=0, atol=1e-5)
