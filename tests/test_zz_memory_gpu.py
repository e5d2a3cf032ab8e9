"""A model and a trainer whose split copies do not fit in the device memory that is
left, where the fp32 products' buffers do: they are made without the copies and run
the fp32 products, bit for bit."""
import contextlib
import ctypes

import numpy as np
import pytest

import cngpt_amd
from test_parity_gpu import say
from test_zz_no_alloc import hip  # noqa: F401 (the fixture)

pytestmark = pytest.mark.gpu

# 1.06 GB of parameters, so that half of a copy is far more than a run needs besides
CFG, B, T = cngpt_amd.Config(6, 25, 1600, 50257, 1024), 2, 256


def free_bytes(hip):  # noqa: F811
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


@contextlib.contextmanager
def only(hip, left):  # noqa: F811
    """All but `left` bytes of the device's free memory taken."""
    held = []
    try:
        while (rest := free_bytes(hip) - left) > 1 << 22:
            p = ctypes.c_void_p()
            if hip.hipMalloc(ctypes.byref(p), min(rest, 32 << 30)) != 0:
                break
            held.append(p)
        say(f"  {free_bytes(hip) / 2**20:.0f} MB left for a want of {left / 2**20:.0f}")
        yield
    finally:
        for p in held:
            hip.hipFree(p)


def test_split_copies_do_not_fit(hip, monkeypatch):  # noqa: F811
    n = cngpt_amd.num_params(CFG)
    block = (0.05 * np.random.default_rng(1).standard_normal(1000003)).astype(np.float32)
    params = np.resize(block, n)
    tok, tgt = (np.random.default_rng(2).integers(0, CFG.vocab_size, (B, T), dtype=np.int32) for _ in range(2))

    def model(split):
        monkeypatch.setenv("CNGPT_HIP_SPLIT", split)
        before = free_bytes(hip)
        m = cngpt_amd.Model(CFG, params)
        return m, before - free_bytes(hip)

    def trainer(m):
        before = free_bytes(hip)
        tr = cngpt_amd.Trainer(m, B, T)
        return tr, before - free_bytes(hip)

    def step(tr):
        loss = tr.forward(tok, tgt)
        tr.backward()
        return loss, tr.grads

    with model("0")[0] as m:  # (what the runtime itself takes)
        m.forward(tok, cngpt_amd.LAST)
    m, small = model("0")
    with m:
        want = m.forward(tok, cngpt_amd.LAST)
        tr, tsmall = trainer(m)
        with tr:
            want_step = step(tr)
    m, large = model("1")
    with m:
        assert not np.array_equal(m.forward(tok, cngpt_amd.LAST), want)
        tr, tlarge = trainer(m)
        tr.close()
        say(f"  model {small / 2**20:.0f} MB, {large / 2**20:.0f} with split copies; "
            f"trainer {tsmall / 2**20:.0f}, {tlarge / 2**20:.0f}")
        with only(hip, (tsmall + tlarge) // 2):
            with trainer(m)[0] as tr:
                got = step(tr)
        assert got[0] == want_step[0] and np.array_equal(got[1], want_step[1])
    with only(hip, (small + large) // 2):
        with model("1")[0] as m:
            got = m.forward(tok, cngpt_amd.LAST)
    assert np.array_equal(got, want)
