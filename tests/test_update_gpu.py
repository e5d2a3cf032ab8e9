"""Forwards of more than 128 rows after an optimizer step: every entry point runs the
updated weights, on the same products whichever came first, and a captured
no-alloc forward replays them."""
import contextlib
import ctypes

import numpy as np
import pytest

import cngpt_amd
from test_kat_gpu import LIB
from test_parity_gpu import randomize
from test_zz_no_alloc import DevBuf, hip, reference  # noqa: F401 (hip is the fixture)

pytestmark = pytest.mark.gpu

CFG, T = cngpt_amd.Config(2, 4, 64, 300, 512), 300


def update(m, seed):
    """One AdamW step of random gradients; the weights after it."""
    with cngpt_amd.Trainer(m, 1, 8) as tr:
        g = np.random.default_rng(seed).standard_normal(tr.params.size).astype(np.float32)
        tr.write(cngpt_amd.TRAIN_GRADS, g)
        tr.adamw(1e-2, wd=0.0)
        return tr.params


@pytest.mark.parametrize("mode", [cngpt_amd.LAST, cngpt_amd.ALL])
@pytest.mark.parametrize("first", ["noalloc", "forward", "resident", "few rows"])
def test_every_entry_point_after_an_update(hip, mode, first):  # noqa: F811
    tokens = np.random.default_rng(1).integers(0, CFG.vocab_size, (1, T), dtype=np.int32)
    n = CFG.vocab_size * (1 if mode == cngpt_amd.LAST else T)
    tok, out = DevBuf(hip, tokens.nbytes), DevBuf(hip, 4 * n)
    tok.put(tokens)
    try:
        with cngpt_amd.Model(CFG, randomize(CFG, cngpt_amd.init_weights(CFG, 2), 3)) as m:
            def noalloc():
                m.forward_noalloc(tok.ptr.value, 1, T, mode, out.ptr.value, None)
                m.synchronize()
                return out.get(n, np.float32)

            calls = {"noalloc": noalloc, "forward": lambda: m.forward(tokens, mode).ravel(),
                     "resident": lambda: reference(m, tokens, mode),
                     "few rows": lambda: m.forward(tokens[:, :20], mode)}
            calls["forward"]()  # (a graph of the old weights)
            with cngpt_amd.Model(CFG, update(m, 4)) as fresh:
                want = fresh.forward(tokens, mode).ravel()
                few = fresh.forward(tokens[:, :20], mode)
            for name in [first] + list(calls):
                same = np.array_equal(calls[name](), few if name == "few rows" else want)
                assert same, name
    finally:
        tok.free()
        out.free()


def test_captured_noalloc_forward_reads_the_live_weights(hip, monkeypatch):  # noqa: F811
    """Captured, more than 128 rows read the parameters themselves: replays follow an
    update, and are the fp32 products' bits."""
    kat = ctypes.CDLL(LIB)
    kat.kat_capture_noalloc.argtypes = [ctypes.c_void_p, ctypes.c_void_p] + [ctypes.c_int] * 3 + [ctypes.c_void_p]
    kat.kat_capture_noalloc.restype = ctypes.c_void_p
    kat.kat_replay.argtypes = [ctypes.c_void_p] * 2
    kat.kat_drop.argtypes = [ctypes.c_void_p]
    tokens = np.random.default_rng(5).integers(0, CFG.vocab_size, (1, T), dtype=np.int32)
    n = CFG.vocab_size * T
    tok, out = DevBuf(hip, tokens.nbytes), DevBuf(hip, 4 * n)
    tok.put(tokens)

    def fp32(params):
        monkeypatch.setenv("CNGPT_HIP_SPLIT", "0")
        with cngpt_amd.Model(CFG, params) as m:
            return m.forward(tokens, cngpt_amd.ALL).ravel()

    params = randomize(CFG, cngpt_amd.init_weights(CFG, 6), 7)
    try:
        with cngpt_amd.Model(CFG, params) as m:
            eager = m.forward(tokens, cngpt_amd.ALL)
            ex = kat.kat_capture_noalloc(m._h, tok.ptr.value, 1, T, cngpt_amd.ALL, out.ptr.value)
            assert ex, "capture failed"
            for seed in (None, 8, 9):
                if seed:
                    params = update(m, seed)
                for _ in range(2):
                    assert kat.kat_replay(m._h, ex) == 0
                    assert np.array_equal(out.get(n, np.float32), fp32(params))
                    m.forward(tokens, cngpt_amd.ALL)  # eager work between the replays
            assert not np.array_equal(m.forward(tokens, cngpt_amd.ALL), eager)
            kat.kat_drop(ex)
    finally:
        tok.free()
        out.free()


@contextlib.contextmanager
def capturing(hip, mode):  # noqa: F811
    """The thread captures a stream of its own (mode: 0 global, 1 thread-local, 2
    relaxed)."""
    hip.hipStreamCreate.argtypes = [ctypes.POINTER(ctypes.c_void_p)]
    hip.hipStreamBeginCapture.argtypes = [ctypes.c_void_p, ctypes.c_int]
    hip.hipStreamEndCapture.argtypes = [ctypes.c_void_p, ctypes.POINTER(ctypes.c_void_p)]
    hip.hipStreamDestroy.argtypes = hip.hipGraphDestroy.argtypes = [ctypes.c_void_p]
    s, g = ctypes.c_void_p(), ctypes.c_void_p()
    assert hip.hipStreamCreate(ctypes.byref(s)) == 0
    try:
        assert hip.hipStreamBeginCapture(s, mode) == 0
        try:
            yield
        finally:
            assert hip.hipStreamEndCapture(s, ctypes.byref(g)) == 0
    finally:
        if g:
            hip.hipGraphDestroy(g)
        hip.hipStreamDestroy(s)


@pytest.mark.parametrize("mode", [0, 1, 2])
def test_noalloc_beside_a_capture(hip, mode):  # noqa: F811
    """The first no-alloc forward after an update, called while the thread captures
    another stream."""
    tokens = np.random.default_rng(1).integers(0, CFG.vocab_size, (1, T), dtype=np.int32)
    n = CFG.vocab_size * T
    tok, out = DevBuf(hip, tokens.nbytes), DevBuf(hip, 4 * n)
    tok.put(tokens)
    try:
        with cngpt_amd.Model(CFG, randomize(CFG, cngpt_amd.init_weights(CFG, 2), 3)) as m:
            with cngpt_amd.Model(CFG, update(m, 4)) as fresh:
                want = fresh.forward(tokens, cngpt_amd.ALL).ravel()
            with capturing(hip, mode):
                m.forward_noalloc(tok.ptr.value, 1, T, cngpt_amd.ALL, out.ptr.value, None)
            m.synchronize()
            same = np.array_equal(out.get(n, np.float32), want)
            assert same
    finally:
        tok.free()
        out.free()


@pytest.mark.parametrize("mode", [0, 1, 2])
def test_backward_beside_a_capture(hip, mode):  # noqa: F811
    """A backward whose products take split weights, called likewise."""
    cfg = cngpt_amd.Config(1, 12, 768, 72, 256)
    tok, tgt = (np.random.default_rng(i).integers(0, 72, (3, 256), dtype=np.int32) for i in (1, 2))
    with cngpt_amd.Model(cfg, cngpt_amd.init_weights(cfg, 3)) as m, cngpt_amd.Trainer(m, 3, 256) as tr:
        tr.forward(tok, tgt)
        tr.backward()
        want = tr.grads
        tr.zero_grad()
        tr.forward(tok, tgt)
        with capturing(hip, mode):
            tr.backward()
        assert np.array_equal(tr.grads, want)
