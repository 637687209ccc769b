"""Attention of few (sequence, head) pairs (one 32-row block per block, its
other side split over four waves) against the kernels for many, which the
other tests hold to float64: the same sequence alone and as the first of a
batch too large for the few-heads form, over every form the rule accepts --
fewer blocks than waves, one block per wave, remainders, the longest
sequence, QK-norm, split operands; and the whole backward through Grads.

Bounds: both round the probabilities and the output to fp16 (2^-11 each), so
their outputs differ by at most 4 2^-11 max|v|; q and k are rounded alike, so
the log-sum-exps differ by fp32 sums only."""
import ctypes as C

import numpy as np
import pytest

import ane
from ane import _lib

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
