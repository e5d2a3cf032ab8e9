"""The training backward's products on the fp16 matrix cores (split_train.hip), which
steps of at least 512 columns and 768 x 768 values take, against the oracle's step at
the edges of their tiles, within test_train_gpu's tolerances; and the verdict
that returns a trainer to the fp32 products."""
import ctypes

import numpy as np
import pytest

import cngpt_amd
import oracle
from test_kat_gpu import LIB, U, fp
from test_parity_gpu import ocfg, randomize, say
from test_train_gpu import batch, compare_grads, tensors

pytestmark = pytest.mark.gpu

# one step, fewer steps than the ring's stages, K split; ragged rows and columns; every
# tile shape (test_products_reach_every_tile)
PRODUCTS = [(65, 16, 32), (130, 72, 64), (768, 768, 4096), (3072, 768, 4096), (2304, 768, 1024),
            (1000, 264, 992), (4096, 3072, 768), (4099, 768, 3072), (6400, 1600, 320), (5121, 2312, 144)]


def test_products_reach_every_tile():
    lib = ctypes.CDLL(LIB)
    assert {lib.kat_split_plan(*s) >> 8 for s in PRODUCTS} == set(range(5))



@pytest.mark.parametrize("M,N,K", PRODUCTS)
@pytest.mark.parametrize("km", [2, 3])
def test_product(M, N, K, km):
    """Within test_split_gpu's bound of a split product, with one scale per tensor."""
    lib = ctypes.CDLL(LIB)
    lib.kat_split_train.argtypes = [ctypes.POINTER(ctypes.c_float)] * 4 + [ctypes.c_int] * 6
    lib.kat_split_train.restype = ctypes.c_long
    rng = np.random.default_rng(M + 7 * N + K)
    ldx, ldw = (M + 7) // 8 * 8 + 8 * (km - 2), N + 8
    X = rng.standard_normal((K, ldx) if km == 3 else (M, K), dtype=np.float32)
    W = rng.standard_normal((K, ldw), dtype=np.float32)
    Y = rng.standard_normal((M, N), dtype=np.float32)
    old, Y32 = Y.copy() * (km == 3), Y.copy()
    top = lib.kat_split_train(fp(X), fp(W), fp(Y), fp(Y32), M, N, K, ldx, ldw, km)
    assert top >= 0, "device call failed"
    x = X[:, :M].T if km == 3 else X
    x, w = x.astype(np.float64), W[:, :N].astype(np.float64)
    ref, mag = old + x @ w, np.abs(old) + np.abs(x) @ np.abs(w)
    bound = (3 * K + 16) * U * mag + 2.0 ** -38 * K * np.abs(X).max() * np.abs(W).max()
    err = np.abs(Y - ref)
    assert (err <= bound).all()
    if km == 2:
        assert top == np.abs(Y).max().view(np.uint32)
    if K % 32 == 0:
        e, e32 = (np.linalg.norm(v - ref) / np.linalg.norm(ref) for v in (Y, Y32))
        say(f"  {M} x {N} x {K} km {km}: error {e:.2e}, fp32 {e32:.2e}")

CASES = {
    # rows padded 1191 -> 1216, odd vocabulary (301 -> 320 columns of dlogits)
    "ragged": (cngpt_amd.Config(2, 8, 512, 301, 400), 3, 397),
    # the fewest rows of the widest head, a vocabulary within one tile
    "fewest": (cngpt_amd.Config(1, 12, 1536, 72, 128), 3, 128),
    # a width of 33 steps (columns past every tile), head size 16
    "c528": (cngpt_amd.Config(1, 33, 528, 97, 256), 5, 241),
    # many rows, so that the larger tiles are taken
    "rows": (cngpt_amd.Config(1, 12, 768, 1000, 512), 5, 509),
    # GPT-2's vocabulary (the lm_head beside the split layers)
    "vocab": (cngpt_amd.Config(1, 12, 768, 50257, 400), 2, 400),
}


@pytest.mark.parametrize("name", list(CASES))
def test_step_vs_oracle(name):
    cfg, B, T = CASES[name]
    params = randomize(cfg, cngpt_amd.init_weights(cfg, 31), 32)
    tok, tgt = batch(cfg, B, T, 33)
    say(f"{name}: B={B} T={T}")
    ref = oracle.Trainer(ocfg(cfg), params, B, T)
    ref.zero_grad()
    ref_loss = ref.forward(tok, tgt)
    ref.backward()
    with cngpt_amd.Model(cfg, params) as m, cngpt_amd.Trainer(m, B, T) as tr:
        loss = tr.forward(tok, tgt)
        tr.backward()
        grads = tr.grads
        tr.zero_grad()
        assert tr.forward(tok, tgt) == loss
        tr.backward()
        assert np.array_equal(tr.grads, grads)  # the same bits again
    assert abs(loss - ref_loss) <= 1e-5 * abs(ref_loss)
    compare_grads(cfg, grads, ref.grads, what=name)
    ref.close()


def test_far_apart_gains_keep_fp32(monkeypatch):
    """Gains 2^-20 of their neighbours, on columns whose weights make up for it: the
    weights' one scale would cost those columns their bits, so the step is the fp32 one,
    to the bit. (Gains alone: test_train_precision_gpu.)"""
    cfg, B, T = CASES["ragged"]
    params = randomize(cfg, cngpt_amd.init_weights(cfg, 41), 42)
    at = {n: (o, k) for n, o, k in tensors(cfg)}
    o, k = at["h1.ln1_w"]
    params[o:o + k:2] *= 2.0 ** -20
    params[at["h1.ln1_b"][0]:][:k:2] *= 2.0 ** -20
    o, k = at["h1.attn_w"]
    w = params[o:o + k].reshape(-1, cfg.n_embd)
    w[:, 0::2] *= 2.0 ** 10
    w[:, 1::2] *= 2.0 ** -10
    tok, tgt = batch(cfg, B, T, 43)
    got = []
    for split in ("1", "0"):
        monkeypatch.setenv("CNGPT_HIP_SPLIT", split)
        with cngpt_amd.Model(cfg, params) as m, cngpt_amd.Trainer(m, B, T) as tr:
            loss = tr.forward(tok, tgt)
            tr.backward()
            got.append((loss, tr.grads))
    assert got[0][0] == got[1][0] and np.array_equal(got[0][1], got[1][1])
