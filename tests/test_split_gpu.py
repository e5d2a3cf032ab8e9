"""The split-operand products (split.hip) against float64, and the rule that
keeps a model on the fp32 kernels.

Bound of a product, u = 2^-24: both operands as hi + lo are within 2u of their
value, the missing lo lo is below 4u of the product, and the sum of 3 K / 16
matrix instructions (16 products each, rounded once per addition at most)
plus the epilogue's roundings is gamma_{3 K + 8} at worst:
|Y - Y64| <= (3 K + 16) u (sum_k |x_k w_k| + |b| + |Y_old|), and the absolute
part of values too small for a full lo, 2^-39 of the largest, per product:
2^-39 K max|x| max|w| each way.
"""
import ctypes
import os

import numpy as np
import pytest

import cngpt_amd
from test_kat_gpu import LIB, U, fp

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def kat():
    lib = ctypes.CDLL(LIB)
    lib.kat_split_gemm.argtypes = ([ctypes.POINTER(ctypes.c_float)] * 4 + [ctypes.c_int] * 8 +
                                   [ctypes.c_float] + [ctypes.POINTER(ctypes.c_float)] * 3)
    lib.kat_attention_split.argtypes = ([ctypes.POINTER(ctypes.c_float)] * 2 + [ctypes.c_int] * 4 +
                                        [ctypes.POINTER(ctypes.c_float)])
    return lib


def run(kat, X, W, b, Y, epi, ldy=None, seg=0, seg_stride=0, ln=None):
    (M, K), N = X.shape, W.shape[0]
    ldy = ldy or N
    lnout = np.zeros((M, N), np.float32) if ln else None
    args = [fp(ln[0]), fp(ln[1]), fp(lnout)] if ln else [None] * 3
    v = kat.kat_split_gemm(fp(X), fp(W), fp(b), fp(Y), M, N, K, ldy, seg, seg_stride, Y.shape[0],
                           epi, float(np.abs(X).max()) * 1.5, *args)
    assert v >= 0, "device call failed"
    return v, lnout


def gelu64(x):
    return 0.5 * x * (1 + np.tanh(np.sqrt(2 / np.pi) * (x + 0.044715 * x ** 3)))


# edges of every tile shape: one k step, fewer than the ring's stages, an odd
# number of steps; ragged rows and columns; K split; the plain stores of an
# odd row length
SHAPES = [(129, 48, 16), (129, 256, 48), (300, 304, 80), (1, 8, 32), (2100, 304, 112), (130, 71, 32),
          (700, 2304, 768), (2047, 776, 3072), (1025, 768, 3072), (4095, 1608, 112),
          (4097, 3064, 176), (4100, 6392, 1600), (513, 4099, 256), (2049, 2312, 768),
          (5121, 2305, 144), (2049, 3073, 512), (5121, 769, 400)]


def test_shapes_reach_every_tile(kat):
    """Both forms of a store (16 bytes a lane; odd row lengths) on every tile shape."""
    for odd in (0, 1):
        assert {kat.kat_split_plan(*s) >> 8 for s in SHAPES if s[1] % 2 == odd} == set(range(5))


@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("epi", [0, 1, 2, 3])
def test_split_product(kat, M, N, K, epi):
    if epi and N % 8:
        pytest.skip("only the lm_head has odd rows")
    rng = np.random.default_rng(M * 7 + N + K)
    X = rng.standard_normal((M, K)).astype(np.float32)
    W = (0.02 * rng.standard_normal((N, K)) * np.exp(rng.standard_normal((N, 1)))).astype(np.float32)
    # small values, and rows that do not fill the fp16 range
    X[:, 0] *= 1e-4
    b = rng.standard_normal(N).astype(np.float32)
    Y = rng.standard_normal((M, N)).astype(np.float32)
    rows = np.unique(np.r_[0, M - 1, rng.integers(0, M, 200)])
    want = X[rows].astype(np.float64) @ W.T.astype(np.float64)
    mag = np.abs(X[rows]).astype(np.float64) @ np.abs(W).T.astype(np.float64)
    old = Y[rows].astype(np.float64)
    verdict, _ = run(kat, X, W, b, Y, epi)
    assert verdict == 0
    tail = 2.0 ** -37 * K * np.abs(X).max() * np.abs(W).max()
    bound = (3 * K + 16) * U * (mag + np.abs(b) + np.abs(old)) + tail
    if epi == 1:
        want = want + b
    elif epi == 2:
        pre = want + b
        want = gelu64(pre)
        # the slope of GELU is below 1.13; its own rounding as in
        # test_kat_gpu; the output is split again, at 1/64 of a unit's step
        bound = 1.13 * bound + (8 + 18 * np.abs(pre)) * U * np.abs(want) + 2.0 ** -31
    elif epi == 3:
        want = old + want + b
    err = np.abs(Y[rows] - want)
    assert (err <= bound).all(), (err / bound).max()
    print(f"{M}x{N}x{K} epi {epi}: rel {np.linalg.norm(Y[rows] - want) / np.linalg.norm(want):.2e} "
          f"worst {(err / bound).max():.3f} of the bound")


@pytest.mark.parametrize("M,N,K", [(300, 256, 64), (2048, 768, 3072), (200, 1600, 6400)])
def test_split_residual_layernorm(kat, M, N, K):
    rng = np.random.default_rng(5)
    X = rng.standard_normal((M, K)).astype(np.float32)
    W = (0.02 * rng.standard_normal((N, K))).astype(np.float32)
    b, g, lb = (rng.standard_normal(N).astype(np.float32) for _ in range(3))
    Y = rng.standard_normal((M, N)).astype(np.float32)
    want = Y + X.astype(np.float64) @ W.T.astype(np.float64) + b
    _, ln = run(kat, X, W, b, Y, 3, ln=(g, lb))
    mean, var = want.mean(1, keepdims=True), want.var(1, keepdims=True)
    wl = (want - mean) / np.sqrt(var + 1e-5) * g + lb
    assert np.linalg.norm(Y - want) <= 1e-6 * np.linalg.norm(want)
    assert np.linalg.norm(ln - wl) <= 2e-6 * np.linalg.norm(wl)


def test_split_rows_into_a_cache(kat):
    """The QKV product of a decode prompt: rows of each sequence seg_stride
    apart, the rows between untouched."""
    rng = np.random.default_rng(6)
    B, T, cap, N, K = 3, 50, 64, 144, 48
    X = rng.standard_normal((B * T, K)).astype(np.float32)
    W = rng.standard_normal((N, K)).astype(np.float32)
    b = rng.standard_normal(N).astype(np.float32)
    Y = np.full((B * cap, N), 7, np.float32)
    run(kat, X, W, b, Y, 1, seg=T, seg_stride=cap)
    want = X.astype(np.float64) @ W.T.astype(np.float64) + b
    Y = Y.reshape(B, cap, N)
    assert np.linalg.norm(Y[:, :T].reshape(-1, N) - want) <= 1e-6 * np.linalg.norm(want)
    assert (Y[:, T:] == 7).all()


@pytest.mark.parametrize("M,N,K", [(150, 144, 48), (129, 2304, 768), (2048, 2304, 768)])
@pytest.mark.parametrize("fp32", [True, False])
def test_split_qkv(kat, M, N, K, fp32):
    """The QKV epilogue: split rows with a scale per third, and the fp32 rows
    (of a cache) beside them."""
    rng = np.random.default_rng(8)
    X = rng.standard_normal((M, K)).astype(np.float32)
    W = (0.05 * rng.standard_normal((N, K))).astype(np.float32)
    b = rng.standard_normal(N).astype(np.float32)
    Y = np.full((M, N), 7, np.float32)
    Ys = np.zeros((M, N), np.float32)
    z = np.zeros(N, np.float32)
    v = kat.kat_split_gemm(fp(X), fp(W), fp(b), fp(Y), M, N, K, N, 0, 0, M, 4,
                           float(np.abs(X).max()), fp(z), fp(z), fp(Ys))
    assert v == 0
    want = X.astype(np.float64) @ W.T.astype(np.float64) + b
    assert np.linalg.norm(Y - want) <= 1e-6 * np.linalg.norm(want)
    # two fp16 halves of a value hold it to one unit of fp32's last place
    assert (np.abs(Ys - Y) <= 2 * U * np.abs(Y) + 2.0 ** -25 / 32).all()


def attention64(qkv, H):
    B, T, C3 = qkv.shape
    q, k, v = (a.reshape(B, T, H, -1).transpose(0, 2, 1, 3) for a in np.split(qkv.astype(np.float64), 3, 2))
    s = q @ k.transpose(0, 1, 3, 2) / np.sqrt(q.shape[-1])
    s[:, :, np.triu(np.ones((T, T), bool), 1)] = -np.inf
    p = np.exp(s - s.max(-1, keepdims=True))
    return (p / p.sum(-1, keepdims=True) @ v).transpose(0, 2, 1, 3).reshape(B, T, C3 // 3)


# head sizes; query and key tiles' edges; scores near zero, ordinary and far
# apart (large ones, where most probabilities vanish, and rows whose maximum
# grows from tile to tile)
@pytest.mark.parametrize("B,T,H,hs", [(1, 1, 2, 64), (2, 31, 3, 32), (1, 64, 2, 64), (3, 65, 1, 128),
                                      (1, 127, 2, 128), (2, 128, 2, 32), (1, 129, 3, 64), (1, 700, 2, 64)])
@pytest.mark.parametrize("size", [1e-3, 1.0, 6.0])
def test_split_attention(kat, B, T, H, hs, size):
    rng = np.random.default_rng(T)
    C = H * hs
    qkv = rng.standard_normal((B, T, 3 * C)).astype(np.float32)
    qkv[..., :C] *= size
    qkv[..., C:2 * C] *= np.linspace(0.1, 2, T, dtype=np.float32)[None, :, None]
    out = np.zeros((B, T, C), np.float32)
    smax = np.array([np.abs(a).max() * 20 for a in np.split(qkv, 3, 2)], np.float32)
    assert kat.kat_attention_split(fp(qkv), fp(out), B, T, C, H, fp(smax)) == 0
    want = attention64(qkv, H)
    # a score s is off by at most (3 hs + 8) u sum|q k| / sqrt(hs), its
    # probability by that times itself; PV adds (3 T + 16) u of sum p |v|
    q, k, v = np.split(np.abs(qkv.astype(np.float64)), 3, 2)
    smag = max(np.einsum("td,sd->ts", q[b][:, h * hs:(h + 1) * hs], k[b][:, h * hs:(h + 1) * hs]).max()
               for b in range(B) for h in range(H)) / np.sqrt(hs)
    bound = ((3 * hs + 8) * smag + 3 * T + 32) * U * 2 * v.max()
    err = np.abs(out - want)
    assert (err <= bound).all(), (err.max(), bound)
    rel = np.linalg.norm(out - want) / np.linalg.norm(want)
    print(f"B{B} T{T} H{H} hs{hs} size {size}: rel {rel:.2e}, worst {err.max() / bound:.3f} of the bound")
    # (a wrong half of any value would show as 2^-11 of it)
    assert rel <= (5e-7 if size <= 1 else 4e-6)
    assert err.max() <= 2.0 ** -16 * v.max()


def test_verdict(kat):
    """Rows of any size are accurate; inputs of a row 2^20 below its bound,
    or weights that are not finite, are not."""
    rng = np.random.default_rng(7)
    X = rng.standard_normal((130, 64)).astype(np.float32)
    W = rng.standard_normal((64, 64)).astype(np.float32)
    b = np.zeros(64, np.float32)

    def verdict(W, scale=1.0):
        Y = np.zeros((130, 64), np.float32)
        return kat.kat_split_gemm(fp(X), fp(W), fp(b), fp(Y), 130, 64, 64, 64, 0, 0, 130, 0,
                                  float(np.abs(X).max() * scale), None, None, None)

    assert verdict(W) == 0
    assert verdict(W * np.exp2(rng.integers(-30, 30, (64, 1))).astype(np.float32)) == 0
    assert verdict(W * 0) == 0
    assert verdict(W, 2.0 ** 20) == 1
    for bad in (np.nan, np.inf, 3e38):
        V = W.copy()
        V[3, 5] = bad
        assert verdict(V) == 1


def test_unsuited_model_keeps_the_fp32_products(monkeypatch):
    """A gain 10^8 times the others leaves the split products less accurate
    than fp32: the logits are those of a handle without them, bit for bit."""
    cfg = cngpt_amd.Config(2, 4, 64, 300, 256)
    p = cngpt_amd.init_weights(cfg, 3)
    tokens = np.random.default_rng(1).integers(0, 300, (2, 200), dtype=np.int32)

    def logits(params):
        with cngpt_amd.Model(cfg, params) as m:
            return m.forward(tokens, cngpt_amd.ALL)

    wild = p.copy()
    wild[300 * 64 + 256 * 64 + 7] = 1e8  # layer 0, ln1_w[7]
    split, got = logits(p), logits(wild)
    monkeypatch.setenv("CNGPT_HIP_SPLIT", "0")
    plain = logits(p)
    assert not np.array_equal(split, plain)
    assert np.abs(split - plain).max() <= 2e-6 * np.abs(plain).max()
    assert np.array_equal(got, logits(wild))


@pytest.mark.parametrize("gain", [1e-9, 1e-16, 1e-25, 300.0, 3e4, 1e6, 1e9, 1e14])
def test_gains_far_from_one(monkeypatch, gain):
    """Small and large gains of a whole LayerNorm: a product of two scales must not
    leave fp32's range (q and k's together, a weight row's and its input's), nor the
    rounding of a large score a probability fp16's; gains too far from 1 for that keep
    the fp32 products, bit for bit."""
    cfg = cngpt_amd.Config(2, 2, 64, 300, 256)
    p = cngpt_amd.init_weights(cfg, 3)
    at = 300 * 64 + 256 * 64
    p[at:at + 64] = gain  # layer 0, ln1_w
    tokens = np.random.default_rng(1).integers(0, 300, (1, 200), dtype=np.int32)

    def logits():
        with cngpt_amd.Model(cfg, p) as m:
            return m.forward(tokens, cngpt_amd.ALL)

    got = logits()
    monkeypatch.setenv("CNGPT_HIP_SPLIT", "0")
    want = logits()
    assert np.isfinite(got).all()
    if gain in (1e-9, 300.0):
        assert not np.array_equal(got, want)
        # scores of up to 13.6 gain^2 (their bound), off by 4 u of themselves on either side
        tol = 2e-6 + 8 * 2.0 ** -24 * 13.6 * gain ** 2
        assert np.abs(got - want).max() <= tol * np.abs(want).max()
    else:
        assert np.array_equal(got, want)
