"""GEMMs whose output is too small to fill the chip (gemm_thin_kernel): every
form the shape rule chooses, at the sizes where it can go wrong -- fewer
k-tiles than waves, remainders of the rings, the block counts on either side
of the rule's lines, split K -- against a float64 product.

Bounds: products of fp16 are exact in fp32; a sum of K of them in fp32, in any
order, is off by at most K 2^-24 sum |a||b|; an fp16 result by 2^-11 of itself
(2^-24 where it is subnormal) more; the epilogues' few fp32 operations by 2^-21 of
their operands."""
import ctypes as C

import numpy as np
import pytest

from ane import _lib

pytestmark = pytest.mark.gpu

STORE_H, STORE_F, RESID, SWIGLU, RELU2, SMEAR = 0, 1, 3, 4, 5, 6

# (M, N, K): 32x32 blocks with 1, 3, 12 and 36 k-tiles over 4 waves; the last
# shape of that form and the first of 32x64 (8 waves, K not a multiple of
# their round); 64x64 with two stages and with one
SHAPES = [(64, 64, 64), (64, 192, 192), (256, 768, 768), (192, 256, 2304), (512, 512, 320), (576, 512, 320),
          (512, 768, 1088), (1024, 768, 704), (1088, 1024, 256), (2112, 768, 576), (128, 16384, 64),
          (1024, 2048, 2048)]


def _u16(a):
    return a.ctypes.data_as(C.POINTER(C.c_uint16))


def _fp(a):
    return None if a is None else a.ctypes.data_as(C.POINTER(C.c_float))


def _vp(a):
    return None if a is None else a.ctypes.data_as(C.c_void_p)


def operands(m, n, k, seed):
    r = np.random.default_rng(seed)
    a = (r.standard_normal((m, k)) * 0.5).astype(np.float16)
    b = (r.standard_normal((n, k)) * 0.5).astype(np.float16)
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    return r, a, b, a64 @ b64.T, k * 2.0 ** -24 * (np.abs(a64) @ np.abs(b64).T)


def within(got, ref, bound, half=False):
    err = np.abs(got.astype(np.float64) - ref)
    lim = bound + 2.0 ** -21 * np.abs(ref) + (2.0 ** -11 * np.abs(ref) + 2.0 ** -24 if half else 0) + 1e-30
    assert np.isfinite(got).all() and (err <= lim).all(), (float((err / lim).max()), got.shape)


@pytest.mark.parametrize("m,n,k", SHAPES)
def test_stores(m, n, k):
    lib = _lib.load()
    _, a, b, ref, bound = operands(m, n, k, m + n + k)
    for epi, dt in ((STORE_F, np.float32), (STORE_H, np.float16)):
        out = np.full((m, n), np.nan, dt)
        assert lib.ane_debug_gemm(0, 0, epi, m, n, k, _u16(a.view(np.uint16)), _u16(b.view(np.uint16)), _vp(out),
                                  0, 0, 0, 0, 1) == 0, lib.ane_debug_last_error()
        within(out, ref, bound, dt == np.float16)


@pytest.mark.parametrize("m,n,k,splits", [(64, 64, 8192, 16), (256, 768, 8320, 5), (128, 192, 384, 3)])
def test_split_k(m, n, k, splits):
    lib = _lib.load()
    _, a, b, ref, bound = operands(m, n, k, splits)
    out = np.full((m, n), np.nan, np.float32)
    assert lib.ane_debug_gemm(0, 0, STORE_F, m, n, k, _u16(a.view(np.uint16)), _u16(b.view(np.uint16)), _vp(out),
                              0, 0, 0, 0, splits) == 0, lib.ane_debug_last_error()
    within(out, ref, bound)


@pytest.mark.parametrize("m,n,k", [(64, 64, 64), (256, 768, 192), (576, 512, 320), (1024, 768, 256), (2112, 768, 192)])
def test_epilogues(m, n, k):
    lib = _lib.load()
    r, a, b, acc, bound = operands(m, n, k, 7 * m + k)
    R, X0 = (r.standard_normal((m, n)).astype(np.float32) for _ in range(2))

    def run(epi, out, c2=None, x0=None, res=None, alpha=1.0, beta=0.0, seq=0):
        assert lib.ane_debug_gemm_epi(epi, m, n, k, _u16(a.view(np.uint16)), _u16(b.view(np.uint16)), _vp(out),
                                      _vp(c2), _fp(x0), _fp(res), alpha, beta, seq, 0, 0,
                                      0) == 0, lib.ane_debug_last_error()

    f32 = lambda: np.full((m, n), np.nan, np.float32)
    out, copy = f32(), f32()
    run(RESID, out, c2=copy, x0=X0, res=R, alpha=0.75, beta=-0.5)
    parts = 0.75 * np.abs(R) + np.abs(acc) + 0.5 * np.abs(X0)
    within(out, 0.75 * R.astype(np.float64) + acc - 0.5 * X0, bound + 2.0 ** -21 * parts)
    np.testing.assert_array_equal(copy, out)

    gate, h13 = np.full((m, n // 2), np.nan, np.float16), np.full((m, n), np.nan, np.float16)
    run(SWIGLU, gate, c2=h13)
    within(h13, acc, bound, True)
    blk, bb = acc.reshape(m, n // 64, 2, 32), bound.reshape(m, n // 64, 2, 32)
    h1, h3 = blk[:, :, 0], blk[:, :, 1]
    # |d silu| <= 1.1 |dh1|; the hardware exp and reciprocal: 2^-20 of the factor
    slack = 1.1 * np.abs(h3) * bb[:, :, 0] + np.abs(h1) * bb[:, :, 1] + 2.0 ** -19 * np.abs(h1 * h3)
    within(gate, (h1 / (1 + np.exp(-h1)) * h3).reshape(m, n // 2), slack.reshape(m, n // 2), True)

    rel, pre = (np.full((m, n), np.nan, np.float16) for _ in range(2))
    run(RELU2, rel, c2=pre)
    within(pre, acc, bound, True)
    within(rel, np.maximum(acc, 0) ** 2, 2 * np.abs(acc) * bound + bound ** 2, True)

    seq = 64
    out, act = f32(), f32()
    run(SMEAR, out, c2=act, x0=X0, alpha=0.3, seq=seq)
    g = 1 / (1 + np.exp(-acc))
    prev = np.vstack([np.zeros((1, n), np.float32), X0[:-1]])
    prev[::seq] = 0
    within(act, g, 0.25 * bound + 2.0 ** -20)
    within(out, X0 + 0.3 * g * prev, (0.25 * bound + 2.0 ** -20) * np.abs(prev) + 2.0 ** -21 * np.abs(X0))
