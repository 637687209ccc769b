"""The softcap of the classifier epilogues over the magnitudes at which its form
changes (cap / 6, 0.6 cap) and beyond, for logits, cross-entropy partials and
the derivative in dlogits, against float64 tanh of the same fp32-exact logits;
and that a value's form is its own.

A is diagonal and B selects one of its rows, so each logit is one exact product."""
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


def test_softcap_is_as_exact_as_tanhf():
    """Every fp16 magnitude from 1/4 to 32 times 64 factors (products of 22
    bits, exact).  cap * tanhf(v / cap) on this GPU is off by 4.6e-8, 4.1e-8
    and 4.7e-8 (rms, relative) in these bands, at most by 2.0e-7."""
    lib = _lib.load()
    mags = np.arange(np.float16(0.25).view(np.uint16), np.float16(32).view(np.uint16), dtype=np.uint16).view(np.float16)
    M, N, K = mags.size, 64, 64
    a = np.zeros((M, K), np.float16)
    a[np.arange(M), np.arange(M) % K] = np.where(np.arange(M) % 2, -mags, mags)
    b = np.repeat((1 + np.arange(N, dtype=np.float16) / 1024).astype(np.float16)[:, None], K, 1)
    x = a.sum(1).astype(np.float64)[:, None] * b[:, 0].astype(np.float64)
    ref = 15.0 * np.tanh(x / 15.0)
    out = np.full((M, N), np.nan, np.float32)
    assert lib.ane_debug_gemm_epi(2, M, N, K, _u16(a), _u16(b), out.ctypes.data_as(C.c_void_p), None, None, None, 1.0,
                                  0.0, -1, 0, 0, 0) == 0, lib.ane_debug_last_error()
    err = np.abs(out - ref) / np.abs(ref)
    assert err.max() <= 1.8e-7, err.max()
    for lo, hi, rms in ((0.25, 6.75, 4.6e-8), (6.75, 9.75, 4.1e-8), (9.75, 15.0, 4.7e-8)):
        band = err[(np.abs(x) >= lo) & (np.abs(x) < hi)]
        assert np.sqrt((band ** 2).mean()) <= rms, (lo, np.sqrt((band ** 2).mean()))


def test_softcap_derivative_does_not_cancel():
    """dlogits of saturated logits: 1 - tanh^2 falls to 2e-6 at 105, where the
    difference of two fp32 numbers keeps two digits.  Bound: dlogits are fp16
    (2^-11), the exponentials' argument is off by 2^-22 at most."""
    lib = _lib.load()
    M = N = K = 256
    r = np.random.default_rng(3)
    v = (r.uniform(7.0, 110.0, M) * r.choice([-1.0, 1.0], M)).astype(np.float16)
    v[0] = 0.0
    a = np.zeros((M, K), np.float16)
    a[np.arange(M), np.arange(M)] = v
    b = np.ones((N, K), np.float16)
    tgt = np.zeros(N, np.uint16)
    lse, scale = np.where(np.arange(N) % 2, -15.0, 15.0).astype(np.float32), np.full(N, 1000.0, np.float32)
    pm, ps, tl = np.zeros((1, N), np.float32), np.zeros((1, N), np.float32), np.zeros(N, np.float32)
    dl = np.zeros((M, N), np.float16)
    assert lib.ane_debug_classifier(M, N, K, _u16(a), _u16(b), tgt.ctypes.data_as(C.POINTER(C.c_uint16)), 1, M, 256, 256,
                                    8, _fp(pm), _fp(ps), _fp(tl), _fp(lse), _fp(scale), _u16(dl),
                                    None) == 0, lib.ane_debug_last_error()
    x = v.astype(np.float64) / 15.0
    ref = np.exp(15.0 * np.tanh(x)[:, None] - lse) * 1000.0 / np.cosh(x)[:, None] ** 2
    normal = (ref > 2.0 ** -14) & (ref < 60000.0)
    normal[0] = False  # the target's row
    assert normal[np.abs(v) > 100].any()
    err = np.abs(dl.astype(np.float64) - ref)[normal] / ref[normal]
    assert err.max() <= 2.0 ** -11 + 4e-6, err.max()


@pytest.mark.parametrize("T", [512, 8192])
def test_a_tokens_loss_does_not_depend_on_its_neighbours(T):
    """The same tokens beside others whose logits are as small or far into the
    cap: bit-identical log-sum-exps (128x128 and 256x256 tiles)."""
    torch = pytest.importorskip("torch")
    lib = _lib.load()
    V, D, seq = 8192, 256, 64
    r = np.random.default_rng(T)
    xn = r.standard_normal((T, D)).astype(np.float16)
    embed = (r.standard_normal((V, D)) * 0.02).astype(np.float16)
    embed[:, :3] *= np.float16(4)  # a few logits past cap / 6 among the rest
    tg = r.integers(0, V, T).astype(np.uint16)
    beside = np.arange(T) % 7 == 3
    dev = lambda a: torch.from_numpy(a.view(np.int16).copy()).cuda()
    ptr = lambda t: C.c_void_p(t.data_ptr())
    lses = []
    for scale in (1.0, 4.0, 20.0):
        x = xn.copy()
        x[beside] *= np.float16(scale)
        x_d, e_d, t_d = dev(x), dev(embed), dev(tg)
        loss, lse = torch.zeros(T // seq, device="cuda"), torch.zeros(T, device="cuda")
        assert lib.ane_head_loss(ptr(x_d), ptr(e_d), ptr(t_d), T, D, V, seq, 1, ptr(loss), ptr(lse),
                                 C.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0, lib.ane_op_last_error()
        lses.append(lse.cpu().numpy())
    assert (lses[0][beside] != lses[2][beside]).all()
    for other in lses[1:]:
        np.testing.assert_array_equal(other[~beside], lses[0][~beside])


def test_softcap_of_infinities_and_nan():
    """+-infinity and the largest fp16 give +-cap exactly, NaN stays, and the
    values beside them (of the same wave) are the softcap of themselves."""
    lib = _lib.load()
    M, N, K = 256, 64, 256
    v = np.linspace(-4, 4, M).astype(np.float16)
    v[[3, 40, 77, 130, 200]] = [np.inf, -np.inf, np.nan, 65504, -65504]
    a = np.zeros((M, K), np.float16)
    a[np.arange(M), np.arange(M)] = v
    out = np.zeros((M, N), np.float32)
    assert lib.ane_debug_gemm_epi(2, M, N, K, _u16(a), _u16(np.ones((N, K), np.float16)),
                                  out.ctypes.data_as(C.c_void_p), None, None, None, 1.0, 0.0, -1, 0, 0,
                                  0) == 0, lib.ane_debug_last_error()
    for row, want in ((3, 15.0), (40, -15.0), (130, 15.0), (200, -15.0)):
        assert (out[row] == want).all(), (row, out[row][:4])
    assert np.isnan(out[77]).all()
    rest = np.delete(np.arange(M), [3, 40, 77, 130, 200])
    ref = 15.0 * np.tanh(v[rest].astype(np.float64) / 15.0)[:, None]
    np.testing.assert_allclose(out[rest], np.broadcast_to(ref, (rest.size, N)), rtol=1.8e-7, atol=1e-30)
