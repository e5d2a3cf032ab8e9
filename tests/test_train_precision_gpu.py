"""Small rows and columns of the training gradients, each on its own scale: what a
tensor's norm does not show, and AdamW divides by. Steps of the size that takes the
fp16 matrix cores, against float64 autograd and against the fp32 step
(CNGPT_HIP_SPLIT=0) of the same weights."""
import numpy as np
import pytest
import torch

import cngpt_amd
from test_kat_gpu import U
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
