"""Timed cases over the public entry points: forwards, decode, sampling, training.

The shapes are the package's own configurations (GPT-2 small, medium and XL
widths, the tiny model of the tests) at the batch sizes that the benchmark and
the tests use, with ragged ones between. Deep models that would only repeat
the same layer are cut in depth, so that their weights are made quickly.

Parameters are drawn like GPT-2's initialisation with LayerNorm gains and
biases moved away from 1 and 0, as trained ones are.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import cngpt_amd as cg


def listed() -> list[dict]:
    small = dict(n_layer=12, n_head=12, n_embd=768, vocab=50257)
    medium = dict(n_layer=8, n_head=16, n_embd=1024, vocab=50257)
    xl = dict(n_layer=6, n_head=25, n_embd=1600, vocab=50257)
    return [
        # the smallest call there is: the tests' own tiny model, one window;
        # launches and host work are all of it
        dict(name="tiny_b1_t16_last", kind="forward", api="host", mode="last", B=1, T=16,
             n_layer=3, n_head=4, n_embd=32, vocab=70),
        # next-token logits of one prompt at the shape the CPU code is quoted on
        dict(name="small_b1_t128_last", kind="forward", api="host", mode="last", B=1, T=128, **small),
        # scoring: logits and mean loss of two full windows (one GPU's share of 16)
        dict(name="small_b2_t1024_loss", kind="forward", api="loss", mode="all", B=2, T=1024, **small),
        # the benchmark's workload: every position's logits, left on the device
        dict(name="small_b16_t1024_all", kind="forward", api="resident", mode="all", B=16, T=1024, **small),
        # a ragged batch of prompts, last logits only
        dict(name="medium_b3_t777_last", kind="forward", api="host", mode="last", B=3, T=777, **medium),
        # the widest configuration (25 heads, 1600 columns), every position
        dict(name="xl_b4_t1024_all", kind="forward", api="resident", mode="all", B=4, T=1024, **xl),
        # single-stream completion, greedy
        dict(name="decode_small_b1_greedy", kind="decode", B=1, T=32, n=128, top_k=0, **small),
        # single-stream completion with the sampler's usual options
        dict(name="decode_small_b1_sampled", kind="decode", B=1, T=200, n=64, top_k=40, **small),
        # batched completions after a long prompt
        dict(name="decode_medium_b8", kind="decode", B=8, T=512, n=32, top_k=0, **medium),
        # many short completions of the widest model
        dict(name="decode_xl_b32", kind="decode", B=32, T=32, n=32, top_k=0, **xl),
        # a training step at the training command's default batch
        dict(name="train_small_b4_t1024", kind="train", B=4, T=1024, **small),
        # fine-tuning a small model on short ragged rows
        dict(name="train_ragged_b3_t111", kind="train", B=3, T=111, n_layer=4, n_head=8, n_embd=512,
             vocab=1000),
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng) -> dict:
    n_head, n_embd = rng.choice([(4, 32), (8, 256), (8, 512), (16, 512), (12, 768), (6, 768),
                                 (16, 1024), (25, 1600)])
    case = dict(n_layer=rng.randint(1, 4), n_head=n_head, n_embd=n_embd,
                vocab=rng.choice([70, 1000, 50257]) if n_embd < 768 else 50257)
    kind = rng.choice(["forward", "forward", "forward", "decode", "train"])
    if kind == "decode":
        T = _log_int(rng, 8, 600)
        case.update(kind=kind, B=_log_int(rng, 1, 32), T=T, n=rng.randint(8, 40),
                    top_k=rng.choice([0, 0, 40]))
    elif kind == "train":
        T = _log_int(rng, 16, 1024)
        case.update(kind=kind, T=T, B=_log_int(rng, 1, max(1, min(32, 4096 // T))))
    else:
        T = _log_int(rng, 1, 1024)
        B = _log_int(rng, 1, max(1, min(64, 16384 // T)))
        api = rng.choice(["host", "resident", "loss"])
        # activations in the library's fixed scratch, logits in the caller's tensor
        if B * T <= 600 and rng.random() < 0.5:
            api = "noalloc"
        mode = "all" if api == "loss" else rng.choice(["last", "all"])
        if api == "host" and B * T > 512:
            mode = "last"
        case.update(kind=kind, api=api, mode=mode, B=B, T=T)
    return case


# ------------------------------------------------------------------ inputs

def _config(case) -> cg.Config:
    block = max(16, case["T"] + case.get("n", 0))
    return cg.Config(case["n_layer"], case["n_head"], case["n_embd"], case["vocab"], max(block, 1024)
                     if case["n_embd"] > 32 else block)


def _views(flat, cfg):
    """The named tensors of a flat parameter buffer (the weight file's order)."""
    C, V, at = cfg.n_embd, cfg.vocab_size, 0

    def take(*shape):
        nonlocal at
        n = math.prod(shape)
        at += n
        return flat[at - n:at].view(*shape)

    top = dict(wte=take(V, C), wpe=take(cfg.block_size, C))
    layers = [dict(ln1_w=take(C), ln1_b=take(C), attn_w=take(3 * C, C), attn_b=take(3 * C),
                   proj_w=take(C, C), proj_b=take(C), ln2_w=take(C), ln2_b=take(C),
                   fc_w=take(4 * C, C), fc_b=take(4 * C), mlp_w=take(C, 4 * C), mlp_b=take(C))
              for _ in range(cfg.n_layer)]
    top.update(lnf_w=take(C), lnf_b=take(C))
    assert at == flat.numel()
    return top, layers


def _params(case, seed):
    cfg = _config(case)
    g = torch.Generator(device="cuda").manual_seed(1000003 * seed + 17)
    flat = torch.empty(cg.num_params(cfg), device="cuda").normal_(0.0, 0.02, generator=g)
    top, layers = _views(flat, cfg)
    residual = 1.0 / math.sqrt(2.0 * cfg.n_layer)
    for w in layers:
        w["proj_w"].mul_(residual)
        w["mlp_w"].mul_(residual)
        for k in ("ln1_w", "ln2_w"):
            w[k].mul_(15.0).exp_()  # gains spread over about 0.5 .. 2
    top["lnf_w"].mul_(15.0).exp_()
    return cfg, flat


def _ids(case, seed, count, salt):
    rng = np.random.default_rng((seed, salt))
    return rng.integers(0, case["vocab"], size=count, dtype=np.int32)


class _Held:
    """The logits that a model holds on the device, for torch.as_tensor (no
    copy; the tensor keeps this object, and so the model's memory, alive)."""

    def __init__(self, model, shape):
        self.model = model
        self.__cuda_array_interface__ = dict(
            shape=shape, typestr="<f4", version=2,
            data=(cg.lib().cngpt_hip_logits_device(model._h), False))


class _Pinned:
    """Pinned host memory, for np.asarray (no copy; the array keeps it alive)."""

    def __init__(self, n):
        self.ptr = cg.lib().cngpt_hip_host_alloc(4 * n)
        if not self.ptr:
            raise cg.CngptError("pinned allocation failed")
        self.__array_interface__ = dict(shape=(n,), typestr="<f4", data=(self.ptr, False), version=3)

    def __del__(self):
        if self.ptr:
            cg.lib().cngpt_hip_host_free(self.ptr)


def prepare(case, seed) -> dict:
    cfg, flat = _params(case, seed)
    B, T = case["B"], case["T"]
    s = dict(case=case, cfg=cfg, model=cg.Model(cfg, flat.cpu().numpy()),
             tokens=_ids(case, seed, (B, T), 1))
    if case["kind"] == "forward":
        mode = cg.LAST if case["mode"] == "last" else cg.ALL
        s["mode"] = mode
        rows = (B,) if mode == cg.LAST else (B, T)
        s["shape"] = rows + (cfg.vocab_size,)
        if case["api"] == "loss":
            s["targets"] = _ids(case, seed, (B, T), 2)
        if case["api"] == "noalloc":
            s["tokens_dev"] = torch.from_numpy(s["tokens"]).cuda()
            s["logits_dev"] = torch.empty(s["shape"], device="cuda")
    elif case["kind"] == "decode":
        if case["top_k"]:
            s["draws"] = np.random.default_rng((seed, 3)).random((case["n"], B), dtype=np.float32)
    else:
        s["targets"] = _ids(case, seed, (B, T), 2)
        s["trainer"] = cg.Trainer(s["model"], B, T)
        s["grads"] = np.asarray(_Pinned(flat.numel()))
    return s


# ------------------------------------------------------------------ one pass

def _held(s):
    return torch.as_tensor(_Held(s["model"], s["shape"]), device="cuda")


def run(s):
    case, m = s["case"], s["model"]
    if case["kind"] == "forward":
        if case["api"] == "host":
            return m.forward(s["tokens"], s["mode"])
        if case["api"] == "resident":
            m.forward(s["tokens"], s["mode"], copy=False)
            return _held(s)
        if case["api"] == "loss":
            return dict(loss=m.loss(s["tokens"], s["targets"]), logits=_held(s))
        m.forward_noalloc(s["tokens_dev"].data_ptr(), case["B"], case["T"], s["mode"],
                          s["logits_dev"].data_ptr())
        m.synchronize()  # handles share the scratch: the next one may start only now
        return s["logits_dev"]
    if case["kind"] == "decode":
        first = m.decode_begin(s["tokens"], case["T"] + case["n"])
        if case["top_k"]:
            new = m.generate(case["n"], 0.8, case["top_k"], s["draws"])
        else:
            new = m.generate(case["n"])
        return dict(first=first, tokens=new, last=m.read_logits(0, first.size).reshape(first.shape))
    t = s["trainer"]
    t.zero_grad()
    loss = t.forward(s["tokens"], s["targets"])
    t.backward()
    grads = s["grads"]
    cg._check(cg.lib().cngpt_hip_train_read(t._t, cg.TRAIN_GRADS, cg._fp(grads), grads.size),
              "train_read")
    norm = t.adamw(3e-4)
    return dict(loss=loss, norm=norm, grads=grads)


# ------------------------------------------------------------------ measures

def _forward_flops(c, B, T, last):
    C, L, V = c["n_embd"], c["n_layer"], c["vocab"]
    attn = 2.0 * C * T * (T + 1) * B
    full = B * T * 24.0 * C * C + attn
    if not last:
        return L * full + 2.0 * B * T * V * C
    return (L - 1) * full + B * T * 6.0 * C * C + B * (18.0 * C * C + 4.0 * C * T) + 2.0 * B * V * C


def work(case) -> dict:
    c, B, T = case, case["B"], case["T"]
    C, L, V = c["n_embd"], c["n_layer"], c["vocab"]
    weights = 4.0 * (L * (12.0 * C * C + 13.0 * C) + V * C)
    if c["kind"] == "forward":
        last = c["mode"] == "last"
        return dict(flops=_forward_flops(c, B, T, last),
                    bytes=weights + 4.0 * B * T * 3 + 4.0 * V * (B if last else B * T))
    if c["kind"] == "decode":
        flops, nbytes = _forward_flops(c, B, T, True), weights + 4.0 * B * V
        for i in range(c["n"] - 1):
            keys = T + i + 1.0
            flops += B * (L * (24.0 * C * C + 4.0 * C * keys) + 2.0 * V * C)
            nbytes += weights + 8.0 * B * L * C * keys
        return dict(flops=flops, bytes=nbytes)
    # backward twice the forward; parameters, gradients and both moments are
    # read and written once by the update, and the gradients go to the host
    return dict(flops=3.0 * _forward_flops(c, B, T, False), bytes=9.0 * weights)


def tolerance(case):
    # fp32 sums in another order; what a few layers of them make of the
    # logits, the loss and the gradients
    if case["kind"] == "decode":
        return {"rel": 2e-5, "max": 2e-4, "differ": 0.01}
    if case["kind"] == "train":
        return {"rel": 2e-5, "max": 1e-3}
    return {"rel": 1e-5, "max": 1e-4}


def _attend(q, k, v, H, q0=0):
    """Causal attention of rows q (positions q0 ..) over k, v, one sequence."""
    T, C = q.shape
    hs = C // H
    qh, kh, vh = (x.view(-1, H, hs).transpose(0, 1).contiguous() for x in (q, k, v))
    s = torch.matmul(qh, kh.transpose(1, 2).contiguous()) / math.sqrt(hs)
    hide = torch.arange(k.shape[0], device=q.device)[None, :] > q0 + torch.arange(T, device=q.device)[:, None]
    p = torch.softmax(s.masked_fill(hide, -math.inf), -1)
    return torch.matmul(p, vh).transpose(0, 1).reshape(T, C)


def _forward64(top, layers, cfg, tokens, last=False):
    """Logits [B, T, V] ([B, V] with last) in the parameters' precision."""
    F = torch.nn.functional
    B, T = tokens.shape
    C = cfg.n_embd
    x = top["wte"][tokens] + top["wpe"][:T]
    for w in layers:
        h = F.layer_norm(x, (C,), w["ln1_w"], w["ln1_b"], 1e-5)
        q, k, v = F.linear(h, w["attn_w"], w["attn_b"]).split(C, -1)
        a = torch.stack([_attend(q[b], k[b], v[b], cfg.n_head) for b in range(B)])
        x = x + F.linear(a, w["proj_w"], w["proj_b"])
        h = F.layer_norm(x, (C,), w["ln2_w"], w["ln2_b"], 1e-5)
        h = F.gelu(F.linear(h, w["fc_w"], w["fc_b"]), approximate="tanh")
        x = x + F.linear(h, w["mlp_w"], w["mlp_b"])
    if last:
        x = x[:, -1]
    return F.linear(F.layer_norm(x, (C,), top["lnf_w"], top["lnf_b"], 1e-5), top["wte"])


def exact(case, seed):
    if case["kind"] == "decode" and (case["top_k"] or case["B"] * (case["T"] + case["n"]) * case["n"] > 200000):
        return None  # sampled tokens hang on the draws; long batches take too long
    cfg, flat = _params(case, seed)
    flat = flat.double()
    B, T = case["B"], case["T"]
    tokens = torch.from_numpy(_ids(case, seed, (B, T), 1)).long().cuda()
    if case["kind"] == "train":
        flat.requires_grad_(True)
        top, layers = _views(flat, cfg)
        targets = torch.from_numpy(_ids(case, seed, (B, T), 2)).long().cuda()
        logits = _forward64(top, layers, cfg, tokens)
        loss = torch.nn.functional.cross_entropy(logits.view(-1, cfg.vocab_size), targets.view(-1))
        loss.backward()
        return dict(loss=loss.detach(), norm=flat.grad.norm(), grads=flat.grad)
    with torch.no_grad():
        top, layers = _views(flat, cfg)
        if case["kind"] == "decode":
            first = last = _forward64(top, layers, cfg, tokens, True)
            new = [last.argmax(-1)]
            for _ in range(case["n"] - 1):
                tokens = torch.cat([tokens, new[-1][:, None]], 1)
                last = _forward64(top, layers, cfg, tokens, True)
                new.append(last.argmax(-1))
            return dict(first=first, tokens=torch.stack(new, 1), last=last)
        logits = _forward64(top, layers, cfg, tokens, case["mode"] == "last")
        if case["api"] != "loss":
            return logits
        targets = torch.from_numpy(_ids(case, seed, (B, T), 2)).long().cuda()
        loss = torch.nn.functional.cross_entropy(logits.view(-1, cfg.vocab_size), targets.view(-1))
        return dict(loss=loss, logits=logits)
