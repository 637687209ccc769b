"""Copies between the caller's memory and the device through the pool of
pinned slots: bit-exact round trips at sizes around a piece, a slot and the
ring (layer weights set and read back, MoE activations), from several threads
at once, and after every object that shared the pool is closed; what the pool's
threads cost a call that waits for kernels, and that small objects make none."""
import ctypes as C
import os
import threading
import time

import numpy as np
import pytest

import ane
from ane import _lib

pytestmark = pytest.mark.gpu

KB = 1024


def engine(vocab, seed):
    cfg = ane.Config(dim=64, hidden=64, heads=1, layers=1, vocab=vocab, seq=64, arch="llama2")
    p = np.random.default_rng(seed).standard_normal(ane.param_count(cfg)).astype(np.float32)
    return ane.Open(ane.Options(Config=cfg, Params=p)), p


# 64 floats a vocabulary row (and 128 KiB of layer weights): below the least
# size of a copy through the pool, at it and past it, around one slot (4 MiB),
# past the ring of 8 slots, past twice that
@pytest.mark.parametrize("vocab", [256, 512, 1024, 3584, 3648, 15808, 15872, 16384, 131072 + 6400, 65536 * 4 + 64])
def test_params_round_trip(vocab):
    other, _ = engine(40000, 3)  # (so that there is a pool, whatever this one's size)
    eng, p = engine(vocab, vocab)
    try:
        for _ in range(2):
            np.testing.assert_array_equal(eng.Params(), p)
        q = np.ascontiguousarray(p[::-1])
        eng.SetParams(q)
        # an unaligned destination inside a larger buffer; what lies around it stays
        buf = np.full(p.size + 5, np.float32(7))
        rc = _lib.load().ane_get_params(eng._h, buf[3:].ctypes.data_as(C.POINTER(C.c_float)), p.size)
        assert rc == 0
        np.testing.assert_array_equal(buf[3:-2], q)
        assert (buf[:3] == 7).all() and (buf[-2:] == 7).all()
        m, v = (np.random.default_rng(s).random(p.size, dtype=np.float32) for s in (1, 2))
        eng.SetOptState(m, v)
        gm, gv = eng.OptState()
        np.testing.assert_array_equal(gm, m)
        np.testing.assert_array_equal(gv, v)
    finally:
        eng.Destroy()
        other.Destroy()


def test_threads_share_the_pool():
    engs = [engine(40000 + 64 * i, i) for i in range(4)]
    bad = []

    def work(e, p):
        try:
            for _ in range(6):
                if not np.array_equal(e.Params(), p):
                    bad.append("params")
                p = np.ascontiguousarray(np.roll(p, 1))
                e.SetParams(p)
        except Exception as x:  # reported below, in the test's own thread
            bad.append(repr(x))

    ts = [threading.Thread(target=work, args=ep) for ep in engs]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    for e, _ in engs:
        e.Destroy()
    assert not bad
    eng, p = engine(40000, 9)  # the pool again, after the last of them has gone
    np.testing.assert_array_equal(eng.Params(), p)
    eng.Destroy()


def test_threads_sleep_while_a_call_waits_for_kernels():
    """Gradients of 32768 tokens, tens of MB: most of the call is the kernels'
    time, through which the caller alone polls: 3.1 CPU seconds a second.  (With
    six threads that look for work all the while: 6.2.)"""
    cfg = ane.Config(dim=256, hidden=512, heads=4, layers=2, vocab=32000, seq=256, arch="llama2")
    tok, tgt = ane.make_tokens(cfg, 128, seed=5)
    eng = ane.Open(ane.Options(Config=cfg, Params=ane.init_params(cfg, seed=4, std=0.02), MaxBatch=128))
    try:
        eng.Grads(tok, tgt)
        share = []
        for _ in range(3):
            c, w = time.process_time(), time.perf_counter()
            eng.Grads(tok, tgt)
            share.append((time.process_time() - c) / (time.perf_counter() - w))
        print("CPU seconds per second", share)
        assert min(share) < 4.0
    finally:
        eng.Destroy()


def test_small_objects_make_no_pool():
    """A model of 1.5 MB opens and evaluates without the pool's threads (and
    its 32 MB of pinned memory); one of 10 MB has them, and takes them along."""
    threads = lambda: len(os.listdir("/proc/self/task"))
    engine(256, 1)[0].Destroy()  # the runtime's own threads
    before = threads()
    cfg = ane.Config(dim=128, hidden=256, heads=2, layers=2, vocab=512, seq=64, arch="llama2")
    eng = ane.Open(ane.Options(Config=cfg, Params=ane.init_params(cfg, seed=0)))
    tok, _ = ane.make_tokens(cfg, 1, seed=1)
    eng.EvalLogits(tok[0])
    eng.Params()
    assert threads() == before
    big, _ = engine(40000, 2)
    assert threads() > before
    big.Destroy()
    assert threads() == before
    eng.Destroy()
