"""Small rows and columns of the training gradients, each on its own scale: what a
tensor's norm does not show, and AdamW divides by. Steps of the size that takes the
fp16 matrix cores, against float64 autograd and against the fp32 step
(CNGPT_HIP_SPLIT=0) of the same weights."""
import ctypes

import numpy as np
import pytest
import torch

import cngpt_amd
from test_kat_gpu import LIB, U, fp
from test_parity_gpu import randomize, say
from test_train_gpu import tensors

pytestmark = pytest.mark.gpu

# 1191 rows of 512 columns, padded to 1216
CFG, B, T = cngpt_amd.Config(2, 8, 512, 301, 400), 3, 397


def named(cfg, flat):
    """Views of a flat buffer by tensor name, matrices as rows."""
    out = {}
    for n, o, k in tensors(cfg):
        w = flat[o:o + k]
        cols = 4 * cfg.n_embd if n.endswith("mlp_w") else cfg.n_embd
        out[n] = w.reshape(-1, cols) if k > 4 * cfg.n_embd else w
    return out


def grads64(cfg, params, tok, tgt):
    """Gradients of the mean loss by float64 autograd on the CPU, by name."""
    F, C, H = torch.nn.functional, cfg.n_embd, cfg.n_head
    p = {n: torch.tensor(w.astype(np.float64), requires_grad=True) for n, w in named(cfg, params).items()}
    t = torch.from_numpy(tok).long()
    Bt, Tt = t.shape
    x = p["wte"][t] + p["wpe"][:Tt]
    heads = lambda a: a.reshape(Bt, Tt, H, C // H).transpose(1, 2)
    for l in range(cfg.n_layer):
        w = {k[len(f"h{l}."):]: v for k, v in p.items() if k.startswith(f"h{l}.")}
        h = F.layer_norm(x, (C,), w["ln1_w"], w["ln1_b"], 1e-5)
        q, k, v = F.linear(h, w["attn_w"], w["attn_b"]).split(C, -1)
        a = F.scaled_dot_product_attention(heads(q), heads(k), heads(v), is_causal=True)
        x = x + F.linear(a.transpose(1, 2).reshape(Bt, Tt, C), w["proj_w"], w["proj_b"])
        h = F.layer_norm(x, (C,), w["ln2_w"], w["ln2_b"], 1e-5)
        h = F.gelu(F.linear(h, w["fc_w"], w["fc_b"]), approximate="tanh")
        x = x + F.linear(h, w["mlp_w"], w["mlp_b"])
    x = F.layer_norm(x, (C,), p["ln_f_w"], p["ln_f_b"], 1e-5)
    F.cross_entropy(F.linear(x, p["wte"]).view(-1, cfg.vocab_size),
                    torch.from_numpy(tgt).long().view(-1)).backward()
    return {n: v.grad.numpy() for n, v in p.items()}


def step(cfg, params, tok, tgt):
    with cngpt_amd.Model(cfg, params) as m, cngpt_amd.Trainer(m, *tok.shape) as tr:
        loss = tr.forward(tok, tgt)
        tr.backward()
        return loss, tr.grads


# one step, tiles' edges, padding rows, K split, the tile shapes
@pytest.mark.parametrize("M,N,K,pad", [(65, 16, 32, 1), (130, 72, 64, 30), (768, 776, 1216, 25),
                                       (1000, 264, 992, 0), (4096, 3072, 768, 0), (4099, 768, 3072, 3),
                                       (5121, 2312, 144, 5)])
@pytest.mark.parametrize("km", [2, 3])
def test_product_of_far_apart_rows_and_columns(M, N, K, pad, km):
    """Each element within the bound of a product (test_split_gpu) of its own row's and
    column's sizes, 2^60 apart, where values too small for a full lo are off by
    2^-40 of the largest that shares their scale."""
    lib = ctypes.CDLL(LIB)
    lib.kat_split_train_rows.argtypes = [ctypes.POINTER(ctypes.c_float)] * 3 + [ctypes.c_int] * 7
    rng = np.random.default_rng(M + N + K + km)
    ldx, ldw = (M + 7) // 8 * 8, N + 8
    X = rng.standard_normal((K, ldx) if km == 3 else (M, K), dtype=np.float32)
    W = rng.standard_normal((K, ldw), dtype=np.float32)
    if km == 3:
        X *= np.exp2(rng.integers(-30, 30, ldx)).astype(np.float32)
        W *= np.exp2(rng.integers(-30, 30, ldw)).astype(np.float32)
        X[:, 3], W[:, 5] = 0, 0
        X[K - pad:], W[K - pad:] = 0, 0
    else:
        X *= np.exp2(rng.integers(-30, 30, (M, 1))).astype(np.float32)
        X[3] = 0
        X[M - pad:] = 0
    Y = np.zeros((M, N), np.float32)
    assert lib.kat_split_train_rows(fp(X), fp(W), fp(Y), M, N, K, ldx, ldw, km, pad) == 0
    x = (X[:, :M].T if km == 3 else X)[: M - (pad if km == 2 else 0)].astype(np.float64)
    Y = Y[: x.shape[0]]
    w = W[:, :N].astype(np.float64)
    ref, mag = x @ w, np.abs(x) @ np.abs(w)
    wtop = np.abs(w).max(0) if km == 3 else np.abs(w).max()
    bound = (3 * K + 16) * U * mag + 2.0 ** -38 * K * np.abs(x).max(1, keepdims=True) * wtop
    err = np.abs(Y - ref)
    assert (err <= bound).all()
    ok = mag > 0
    say(f"  {M} x {N} x {K} km {km}: at most {(err[ok] / mag[ok]).max():.1e} of the sum of magnitudes")
    assert (err[ok] <= 2.0 ** -20 * mag[ok]).all()  # (a wrong half of a value: 2^-11)


def test_improbable_tokens():
    """Tokens of probability 1e-2 down to 1e-18 in every row that appear nowhere in
    the batch: their embeddings' gradients are (p / N) . x summed over the rows, at
    any p. A logit is off by at most (C + 8) u sum_k |x_k w_k| and p by that
    relative to itself, the sum over N rows by less."""
    params = randomize(CFG, cngpt_amd.init_weights(CFG, 51), 52)
    w = named(CFG, params)
    rng = np.random.default_rng(53)
    away = rng.standard_normal(CFG.n_embd)
    away /= np.linalg.norm(away)
    rare = np.arange(200, 301)
    w["ln_f_b"] += (40 * away).astype(np.float32)
    w["wte"][rare] -= np.outer(np.linspace(0, 1, rare.size), away).astype(np.float32)
    tok, tgt = (rng.integers(0, 200, (B, T), dtype=np.int32) for _ in range(2))
    ref = grads64(CFG, params, tok, tgt)["wte"][rare]
    _, g = step(CFG, params, tok, tgt)
    got = named(CFG, g)["wte"][rare]
    err = np.linalg.norm(got - ref, axis=1) / np.linalg.norm(ref, axis=1)
    say(f"  rows of size {np.linalg.norm(ref, axis=1).min():.1e} .. {np.linalg.norm(ref, axis=1).max():.1e}: "
        f"relative error {err.min():.1e} .. {err.max():.1e}")
    # |x| <= sqrt(C) max|g| + |b|, by Cauchy-Schwarz; the softmax's sum is off likewise
    xn = np.sqrt(CFG.n_embd) * np.abs(w["ln_f_w"]).max() + np.linalg.norm(w["ln_f_b"])
    bound = 2 * (CFG.n_embd + 8) * U * xn * np.linalg.norm(w["wte"], axis=1).max()
    assert (err <= bound).all(), (err.max(), bound)


def test_far_apart_rows_and_columns(monkeypatch):
    """Activations and gradients whose columns and rows are far apart under ordinary
    weights: LayerNorm gains 2^-28 of the others, hidden units that never open, a
    head of small queries and keys, rows whose token is certain. Every row and
    column of every matrix's gradient is that of the fp32 step (whose forward is the
    same to the bit) within what the two sums of up to Np rows may be off,
    (Np + 16) u each, compounded over the layers' own few."""
    params = randomize(CFG, cngpt_amd.init_weights(CFG, 61), 62)
    w = named(CFG, params)
    C = CFG.n_embd
    rng = np.random.default_rng(63)
    for n in ("h0.ln1", "h1.ln2"):
        w[n + "_w"][::2] *= 2.0 ** -28
        w[n + "_b"][::2] *= 2.0 ** -28
    w["h0.fc_b"][:64] = -7
    w["h1.fc_b"][64:128] = -5
    w["h1.mlp_w"][:, 64:128] *= 2.0 ** -11
    for third in (0, C):
        w["h1.attn_w"][third + 192:third + 256] *= 2.0 ** -9
        w["h1.attn_b"][third + 192:third + 256] *= 2.0 ** -9
    tok, tgt = (rng.integers(0, 300, (B, T), dtype=np.int32) for _ in range(2))
    sure = rng.standard_normal(C)
    sure /= np.linalg.norm(sure)
    w["wpe"][T - 1] = 40 * sure
    w["wte"][300] = 0.85 * sure
    tgt[:, -1] = 300
    got = []
    for split in ("1", "0"):
        monkeypatch.setenv("CNGPT_HIP_SPLIT", split)
        got.append(step(CFG, params, tok, tgt))
    assert got[0][0] == got[1][0]
    assert not np.array_equal(got[0][1], got[1][1])  # (the step took the split products)
    tol = 4 * (1216 + 16) * U
    a, b = (named(CFG, g[1]) for g in got)
    worst = {}
    for n in a:
        if a[n].ndim < 2:
            continue
        x, y = a[n].astype(np.float64), b[n].astype(np.float64)
        for axis in (0, 1):
            size = np.linalg.norm(y, axis=axis)
            err = np.linalg.norm(x - y, axis=axis)[size > 0] / size[size > 0]
            worst[n, "columns" if axis == 0 else "rows"] = err.max()
            say(f"  {n} {'columns' if axis == 0 else 'rows'}: of size {size[size > 0].min():.1e} .. {size.max():.1e}, "
                f"off by {np.median(err):.1e}, at most {err.max():.1e}")
    assert max(worst.values()) <= tol, (worst, tol)


def test_weights_with_small_rows_keep_fp32(monkeypatch):
    """Rows of a weight matrix 2^-20 of the others, whose outputs' gradients could be
    that much larger under the same scale: the step is the fp32 one, to the bit."""
    params = randomize(CFG, cngpt_amd.init_weights(CFG, 71), 72)
    named(CFG, params)["h1.fc_w"][100:110] *= 2.0 ** -20
    rng = np.random.default_rng(73)
    tok, tgt = (rng.integers(0, 301, (B, T), dtype=np.int32) for _ in range(2))
    got = []
    for split in ("1", "0"):
        monkeypatch.setenv("CNGPT_HIP_SPLIT", split)
        got.append(step(CFG, params, tok, tgt))
    assert got[0][0] == got[1][0] and np.array_equal(got[0][1], got[1][1])
