"""Attention of few (sequence, head) pairs (one 32-row block per block, its
other side split over four waves) against the kernels for many: the same
sequence alone and as the first of a batch too large for the few-heads form,
over every form the rule accepts -- fewer blocks than waves, one block per
wave, remainders, the longest sequence, QK-norm, split operands; and the whole
backward through Grads.  The few-heads form is held to float64 and to the
oracle by the small cases of test_gpu_kernels.py and test_gpu_train.py; the
kernels for many are here, past the rules' lines.

Bounds: both round the probabilities and the output to fp16 (2^-11 each), so
their outputs differ by at most 4 2^-11 max|v|; q and k are rounded alike, so
the log-sum-exps differ by fp32 sums only."""
import ctypes as C

import numpy as np
import pytest

import ane
import oracle
from ane import _lib
from test_gpu_kernels import attn_ref
from test_gpu_train import check_grads

pytestmark = pytest.mark.gpu


def attention(qkv, nseq, S, NH, qknorm, scale, hilo):
    lib = _lib.load()
    out = np.full((nseq * S, 64 * NH), np.nan, np.float16)
    lse = np.full((nseq * S, NH), np.nan, np.float32)
    u16 = lambda x: x.view(np.uint16).ctypes.data_as(C.POINTER(C.c_uint16))
    assert lib.ane_debug_attention(nseq, S, NH, qknorm, 1e4, scale, hilo, u16(qkv), u16(out),
                                   lse.ctypes.data_as(C.POINTER(C.c_float))) == 0, lib.ane_debug_last_error()
    return out[:S].astype(np.float64), lse[:S].astype(np.float64)


@pytest.mark.parametrize("S,NH,qknorm,scale,hilo", [
    (64, 1, 0, 0.125, 0), (64, 3, 1, 0.125, 0), (128, 2, 0, 0.125, 0), (192, 5, 1, 1.0, 1), (256, 12, 0, 0.125, 0),
    (256, 12, 1, 1.0, 1), (320, 4, 1, 0.125, 0), (448, 3, 0, 0.125, 0), (512, 12, 0, 0.125, 0)])
def test_forward_matches_the_many_heads_kernels(S, NH, qknorm, scale, hilo):
    many = 512 // (NH * (S // 32)) + 1  # sequences that put the batch past the rule's line
    qkv = np.random.default_rng(S + NH).standard_normal((many * S, 3 * 64 * NH)).astype(np.float16)
    few_o, few_l = attention(qkv[:S].copy(), 1, S, NH, qknorm, scale, hilo)
    ref_o, ref_l = attention(qkv, many, S, NH, qknorm, scale, hilo)
    vmax = float(np.abs(qkv[:S].reshape(S, 3, -1)[:, 2].astype(np.float64)).max())
    assert np.abs(few_o - ref_o).max() <= 4 * 2.0 ** -11 * vmax
    assert np.abs(few_l - ref_l).max() <= 2e-5 * max(1.0, np.abs(ref_l).max())


@pytest.mark.parametrize("arch,mode,seq", [("llama2", "true", 64), ("llama2", "true", 192), ("llama2", "true", 256),
                                           ("nanochat", "compat", 128), ("nanochat", "compat", 256),
                                           ("nanochat", "true", 192)])
def test_backward_matches_the_many_heads_kernels(arch, mode, seq):
    cfg = ane.Config(dim=256, hidden=512, heads=4, layers=2, vocab=512, seq=seq, arch=arch, grad_mode=mode)
    many = 768 // (4 * (seq // 32)) + 1
    tok, tgt = ane.make_tokens(cfg, 1, seed=seq)
    eng = ane.Open(ane.Options(Config=cfg, Params=ane.init_params(cfg, seed=3, std=0.05), MaxBatch=many))
    try:
        loss1, few = eng.Grads(tok, tgt)
        lossn, ref = eng.Grads(np.repeat(tok, many, 0), np.repeat(tgt, many, 0))
    finally:
        eng.Destroy()
    assert abs(loss1 - lossn) <= 1e-4
    for name, off, shape in ane.param_layout(cfg):
        if name.split(".")[-1] in ("resid_lambdas", "x0_lambdas", "smear_lambda", "backout_lambda", "ve_gate"):
            continue  # single sums over the activations
        a, b = (g[off:off + int(np.prod(shape))].astype(np.float64) for g in (few, ref))
        # the contract's bound for a weight gradient
        assert np.linalg.norm(a - b) <= 1e-2 * np.linalg.norm(b), (name, np.linalg.norm(a - b) / np.linalg.norm(b))


# sequences that put each length past the line (S = 64 .. 512); 468 heads: whole-head blocks in one launch
@pytest.mark.parametrize("S,NH,nseq,qknorm", [(64, 12, 11, 1), (128, 12, 6, 0), (192, 12, 4, 1), (256, 12, 3, 0),
                                              (256, 12, 39, 1), (320, 12, 5, 0), (448, 12, 4, 1), (512, 12, 3, 0)])
def test_many_heads_match_f64(S, NH, nseq, qknorm):
    assert nseq * NH * (S // 32) > (512 if S > 256 else 256)
    qkv = np.random.default_rng(S + nseq).standard_normal((nseq * S, 3 * 64 * NH)).astype(np.float16)
    out, lse = np.empty((nseq * S, 64 * NH), np.float16), np.empty((nseq * S, NH), np.float32)
    lib, u16 = _lib.load(), lambda x: x.view(np.uint16).ctypes.data_as(C.POINTER(C.c_uint16))
    assert lib.ane_debug_attention(nseq, S, NH, qknorm, 1e4, 0.125, 0, u16(qkv), u16(out),
                                   lse.ctypes.data_as(C.POINTER(C.c_float))) == 0, lib.ane_debug_last_error()
    ref, ref_l = attn_ref(qkv, nseq, S, NH, qknorm, 1e4)
    tol = 2e-2 if qknorm else 6e-3  # as test_attention_matches_f64's
    np.testing.assert_allclose(out.astype(np.float64), ref, atol=tol)
    np.testing.assert_allclose(lse, ref_l, atol=2 * tol)


def test_many_heads_split_scores_match_f64():
    S, NH, nseq = 256, 12, 3
    qkv = np.random.default_rng(5).standard_normal((nseq * S, 3 * 64 * NH)).astype(np.float16)
    out, lse = attention(qkv, nseq, S, NH, 1, 1.0, 1)
    ref, ref_l = attn_ref(qkv[:S], 1, S, NH, True, 1e4, scale=1.0)
    assert np.abs(lse - ref_l).max() < 1e-3 and np.abs(out - ref).max() < 4e-3  # as the split scores' test


@pytest.mark.parametrize("arch,mode,seq", [("llama2", "true", 64), ("llama2", "true", 128), ("llama2", "true", 192),
                                           ("llama2", "true", 256), ("nanochat", "compat", 128),
                                           ("nanochat", "compat", 192), ("nanochat", "true", 192)])
def test_many_heads_gradients_match_the_oracle(arch, mode, seq):
    """Two windows, repeated past the rule's line: the mean's gradient is theirs."""
    cfg = ane.tiny(arch, grad_mode=mode, seq=seq)
    many = 768 // (2 * (seq // 32)) + 2
    many += many % 2
    p = ane.init_params(cfg, seed=23, std=0.08)
    tok, tgt = ane.make_tokens(cfg, 2, seed=24)
    loss_ref, g_ref = oracle.grads(cfg, p, tok, tgt)
    eng = ane.Open(ane.Options(Config=cfg, Params=p, MaxBatch=many))
    try:
        loss, g = eng.Grads(np.tile(tok, (many // 2, 1)), np.tile(tgt, (many // 2, 1)))
    finally:
        eng.Destroy()
    assert abs(loss - loss_ref) <= 1e-3
    check_grads(cfg, g, g_ref)
