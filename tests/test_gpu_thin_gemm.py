"""GEMMs whose output is too small to fill the chip (gemm_thin_kernel): every
form the shape rule chooses, at the sizes where it can go wrong -- fewer
k-tiles than waves, remainders of the rings, the block counts on either side
of the rule's lines, split K -- and every epilogue, against a float64 product.

Bounds: products of fp16 are exact in fp32; a sum of K of them in fp32, in any
order, is off by at most K 2^-24 sum |a||b|; an fp16 result by 2^-11 of itself
(2^-24 where it is subnormal) more; the epilogues' few fp32 operations by 2^-21 of
their operands."""
import ctypes as C

import numpy as np
import pytest

from ane import _lib

pytestmark = pytest.mark.gpu

STORE_H, STORE_F, RESID, SWIGLU, RELU2, SMEAR, SWIGLU_BWD, RELU2_BWD = 0, 1, 3, 4, 5, 6, 10, 11
RESID_NORM, STORE_H_RR, SWIGLU_RR = 13, 14, 15
# one shape for each form the epilogues below take, and both sides of the lines between them
FORMS = [(64, 64, 64), (256, 768, 192), (576, 512, 320), (1024, 768, 256), (2112, 768, 192)]

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


@pytest.mark.parametrize("m,n,k", FORMS)
def test_accumulating_store_and_scalars_from_memory(m, n, k):
    lib = _lib.load()
    r, a, b, acc, bound = operands(m, n, k, 5 * m + k)
    R, X0 = (r.standard_normal((m, n)).astype(np.float32) for _ in range(2))

    def run(epi, out, x0=None, alpha=1.0, beta=0.0, seq=0):
        assert lib.ane_debug_gemm_epi(epi, m, n, k, _u16(a.view(np.uint16)), _u16(b.view(np.uint16)), _vp(out), None,
                                      _fp(x0), _fp(R), alpha, beta, seq, 0, 0, 0) == 0, lib.ane_debug_last_error()

    out = np.full((m, n), np.nan, np.float32)
    run(STORE_F, out)
    within(out, R + acc, bound + 2.0 ** -21 * (np.abs(R) + np.abs(acc)))
    out[:] = np.nan
    run(RESID, out, x0=X0, alpha=-0.25, beta=1.5, seq=1)  # alpha and beta from device memory
    parts = 0.25 * np.abs(R) + np.abs(acc) + 1.5 * np.abs(X0)
    within(out, -0.25 * R.astype(np.float64) + acc + 1.5 * X0, bound + 2.0 ** -21 * parts)


@pytest.mark.parametrize("m,n,k", FORMS)
def test_backward_epilogues(m, n, k):
    lib = _lib.load()
    r, a, b, dg, bound = operands(m, n, k, 3 * m + k)

    def run(epi, out, saved):
        assert lib.ane_debug_gemm_epi(epi, m, n, k, _u16(a.view(np.uint16)), _u16(b.view(np.uint16)), _vp(out),
                                      _vp(saved), None, None, 1.0, 0.0, 0, 0, 0, 0) == 0, lib.ane_debug_last_error()

    h13 = r.standard_normal((m, 2 * n)).astype(np.float16)
    out = np.full((m, 2 * n), np.nan, np.float16)
    run(SWIGLU_BWD, out, h13.copy())
    h1, h3 = (h13.astype(np.float64).reshape(m, n // 32, 2, 32)[:, :, i].reshape(m, n) for i in range(2))
    sg = 1 / (1 + np.exp(-h1))
    d1, d3 = sg + h1 * sg * (1 - sg), h1 * sg  # d silu and silu
    got = out.reshape(m, n // 32, 2, 32)
    # the hardware exp and reciprocal: 2^-20 of each term
    within(got[:, :, 0].reshape(m, n), dg * h3 * d1, np.abs(h3 * d1) * bound + 2.0 ** -19 * np.abs(dg * h3) * (1 + np.abs(h1)),
           True)
    within(got[:, :, 1].reshape(m, n), dg * d3, np.abs(d3) * bound + 2.0 ** -19 * np.abs(dg * d3), True)

    h = r.standard_normal((m, n)).astype(np.float16)
    out = np.full((m, n), np.nan, np.float16)
    run(RELU2_BWD, out, h.copy())
    relu = np.maximum(h.astype(np.float64), 0)
    within(out, dg * 2 * relu, 2 * relu * bound, True)


@pytest.mark.parametrize("m,n,k", FORMS)
def test_deferred_norm_epilogues(m, n, k):
    lib = _lib.load()
    r, a, b, acc, bound = operands(m, n, k, 11 * m + k)

    def run(epi, out, X=None, gain=None, ssq=None, part=None, dim=0, nw=0):
        assert lib.ane_debug_gemm_norm(epi, m, n, k, _u16(a.view(np.uint16)), _u16(b.view(np.uint16)), _fp(X),
                                       _u16(out.view(np.uint16)), _fp(gain), _fp(ssq), _fp(part),
                                       0 if part is None else len(part), dim, 0, 0, nw) == 0, lib.ane_debug_last_error()

    X0 = r.standard_normal((m, n)).astype(np.float32)
    gain = (1 + 0.3 * r.standard_normal(n)).astype(np.float32)
    for nw in (0, -1):  # aligned; a gain off by 4 bytes: the 64x64 tiles of the other kernel
        X, xg, ssq = X0.copy(), np.full((m, n), np.nan, np.float16), np.full((n // 64, m), np.nan, np.float32)
        run(RESID_NORM, xg, X=X, gain=gain, ssq=ssq, nw=nw)
        within(X, X0 + acc, bound + 2.0 ** -21 * (np.abs(X0) + np.abs(acc)))
        x = X.astype(np.float64)
        within(xg, x * gain, 2.0 ** -23 * np.abs(x * gain), True)
        sums = (x ** 2).reshape(m, n // 64, 64).sum(-1).T
        within(ssq, sums, 64 * 2.0 ** -24 * sums)

    for nparts in (1, 12, 16):
        part = (r.random((nparts, m)) * 40 + 1e-3).astype(np.float32)
        rr = 1 / np.sqrt(part.astype(np.float64).sum(0) / 768 + 1e-5)[:, None]
        out = np.full((m, n), np.nan, np.float16)
        run(STORE_H_RR, out, part=part, dim=768)
        within(out, acc * rr, rr * (bound + 2.0 ** -20 * np.abs(acc)), True)
    gate = np.full((m, n // 2), np.nan, np.float16)
    run(SWIGLU_RR, gate, part=part, dim=768)
    lim = rr * (bound + 2.0 ** -20 * np.abs(acc))
    blk, bb = (acc * rr).reshape(m, n // 64, 2, 32), lim.reshape(m, n // 64, 2, 32)
    h1, h3 = blk[:, :, 0], blk[:, :, 1]
    slack = 1.1 * np.abs(h3) * bb[:, :, 0] + np.abs(h1) * bb[:, :, 1] + bb[:, :, 0] * bb[:, :, 1] + 2.0 ** -19 * np.abs(h1 * h3)
    within(gate, (h1 / (1 + np.exp(-h1)) * h3).reshape(m, n // 2), slack.reshape(m, n // 2), True)
