"""The work a program built on minitorch_amd has it do, as cases that can be
timed and checked one by one.

A case is a dict of plain sizes; ``prepare`` makes what the program has in hand
before the call (inputs on the GPU, weights, a recorded step), ``run`` is one
pass through the package's public entry points and ``exact`` the same numbers
from plain torch in 64 bits.  Kinds:

  attn    fused causal attention on its own, forward and backward
          (kernels.attn_fwd / attn_bwd), fp32 or bf16
  decode  one query position per sequence against cached keys and values
          (kernels.attn_decode)
  mha     a MultiHeadAttention layer, forward and backward
  block   a TransformerBlock, forward and backward
  head    the vocabulary projection and the cross-entropy loss, forward and
          backward
  train   a GPT training step with Adam, replayed from a recorded HIP graph
  score   a GPT's logits for a batch of contexts, no gradients
  greedy  greedy generation with a KV cache: prompt, then token by token
"""
import math

import numpy as np
import torch

import minitorch_amd as mt
from minitorch_amd import device as dev
from minitorch_amd import kernels as K
from minitorch_amd.device import DeviceArray

# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------


def listed():
    return [
        # one decode step's attention of the 6-head character model, half its
        # batch: a single short launch
        dict(name="decode_step", kind="decode", B=32, H=6, L=200, D=64, dtype="float32"),
        # the attention op alone at the repository's fp32 size
        dict(name="attn_fp32", kind="attn", B=32, H=8, T=256, D=64, dtype="float32"),
        # long-context bf16 attention, the benchmark's size
        dict(name="attn_long", kind="attn", B=8, H=16, T=2048, D=64, dtype="bfloat16"),
        # bf16 attention with wide heads and a length that fills no tile
        dict(name="attn_wide_ragged", kind="attn", B=4, H=12, T=1531, D=128, dtype="bfloat16"),
        # one attention layer of the 384-wide model at its training batch
        dict(name="mha_layer", kind="mha", B=64, T=256, C=384, H=6),
        # a whole block of a wider model on ragged contexts
        dict(name="block_ragged", kind="block", B=8, T=1001, C=512, H=8),
        # the character vocabulary's head and loss over a training batch
        dict(name="head_chars", kind="head", rows=16384, C=384, V=65),
        # the same with a subword vocabulary of odd size
        dict(name="head_words", kind="head", rows=8192, C=384, V=5003),
        # the small character model's training step: bound by its launches
        dict(name="train_small", kind="train", B=16, T=32, C=64, H=4, layers=2, V=65),
        # the 384-wide model's training step (three of its blocks)
        dict(name="train_wide", kind="train", B=64, T=256, C=384, H=6, layers=3, V=65),
        # scoring a few contexts: forward only, few rows
        dict(name="score", kind="score", B=4, T=250, C=384, H=6, layers=6, V=65),
        # generation: a batch of prompts extended token by token
        dict(name="greedy", kind="greedy", B=64, T=32, n=48, C=384, H=6, layers=6, V=65),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["attn", "attn", "decode", "mha", "block", "block", "head", "train", "train", "score", "greedy"])
    if kind == "attn":
        dtype = rng.choice(["bfloat16", "bfloat16", "float32"])
        D = rng.choice([64, 64, 128]) if dtype == "bfloat16" else rng.choice([16, 32, 64, 64])
        T = _log(rng, 48, 4096) if dtype == "bfloat16" else _log(rng, 24, 700)
        H = rng.choice([4, 6, 8, 12, 16])
        top = 8 * 16 * 2048 * 2048 * 64 if dtype == "bfloat16" else 32 * 8 * 512 * 512 * 64
        B = max(1, min(_log(rng, 1, 64), top // (H * T * T * D)))
        return dict(kind=kind, B=B, H=H, T=T, D=D, dtype=dtype)
    if kind == "decode":
        dtype = rng.choice(["float32", "float32", "bfloat16"])
        return dict(kind=kind, B=_log(rng, 1, 96), H=rng.choice([4, 6, 8, 12]), L=_log(rng, 20, 2000),
                    D=rng.choice([64, 64, 128]), dtype=dtype)
    H = rng.choice([2, 4, 6, 6, 8, 12])
    C = 64 * H
    if kind == "head":
        return dict(kind=kind, rows=_log(rng, 300, 16384), C=C, V=rng.choice([65, _log(rng, 90, 6000)]))
    if kind in ("mha", "block"):
        T = _log(rng, 40, 1100)
        B = max(1, min(_log(rng, 2, 64), 64 * 256 * 384 // (T * C)))
        return dict(kind=kind, B=B, T=T, C=C, H=H)
    layers = rng.randint(1, 3)
    if kind == "train":
        T = _log(rng, 24, 400)
        B = max(1, min(_log(rng, 2, 64), 64 * 256 * 384 * 384 // (T * C * C)))
        return dict(kind=kind, B=B, T=T, C=C, H=H, layers=layers, V=rng.choice([65, rng.randint(60, 300)]))
    if kind == "score":
        T = _log(rng, 16, 500)
        return dict(kind=kind, B=max(1, min(_log(rng, 1, 32), 8192 // T)), T=T, C=C, H=H, layers=2 * layers, V=65)
    H = rng.choice([4, 6, 6, 8])
    return dict(kind=kind, B=_log(rng, 1, 64), T=_log(rng, 6, 48), n=_log(rng, 6, 48), C=64 * H, H=H, layers=2 * layers,
                V=65)


# ---------------------------------------------------------------------------
# device arrays and torch
# ---------------------------------------------------------------------------
_TYPESTR = {"float32": "<f4", "bfloat16": "<i2", "int64": "<i8", "int32": "<i4"}


class _Shared:
    """A package buffer under the interface torch reads device memory by."""

    def __init__(self, buf):
        self.buf = buf
        size = buf.element_size()
        self.__cuda_array_interface__ = {
            "shape": tuple(buf.shape), "strides": tuple(s * size for s in buf.stride()),
            "typestr": _TYPESTR[buf.dtype], "data": (buf.data_ptr(), False), "version": 2}


def _torch(a):
    """A torch tensor over the memory of a DeviceArray or DevBuf (no copy)."""
    buf = a.t if isinstance(a, DeviceArray) else a
    t = torch.as_tensor(_Shared(buf), device="cuda")
    return t.view(torch.bfloat16) if buf.dtype == "bfloat16" else t


def _device(x):
    """A package array with a torch tensor's values."""
    out = dev.empty(tuple(x.shape), str(x.dtype).rsplit(".", 1)[-1])
    _torch(out).copy_(x)
    return out


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 7919 + 17)
    return g


def _normal(g, shape, std=1.0, dtype=torch.float32):
    return (torch.randn(tuple(shape), generator=g, device="cuda") * std).to(dtype)


def _ids(g, shape, n):
    return torch.randint(0, n, tuple(shape), generator=g, device="cuda")


# ---------------------------------------------------------------------------
# inputs, from the seed alone (run and exact both start here)
# ---------------------------------------------------------------------------


def _layer_weights(g, C):
    """A block's parameters under their state_dict names, in the package's
    order, at the scale trained models have: weights N(0, 0.02), gains near 1."""
    def norm(at):
        return {f"{at}.gamma": 1.0 + _normal(g, (C,), 0.1), f"{at}.beta": _normal(g, (C,), 0.1)}

    def linear(at, n_in, n_out):
        return {f"{at}.weight": _normal(g, (n_in, n_out), 0.02), f"{at}.bias": _normal(g, (n_out,), 0.02)}

    w = norm("ln1")
    for p in ("q_proj", "k_proj", "v_proj", "out_proj"):
        w.update(linear(f"attn.{p}", C, C))
    w.update(norm("ln2"))
    w.update(linear("mlp.layers.0", C, 4 * C))
    w.update(linear("mlp.layers.2", 4 * C, C))
    return w


def _model_weights(g, case):
    C, V = case["C"], case["V"]
    w = {"tok_emb.weight": _normal(g, (V, C), 0.02), "pos_emb.weight": _normal(g, (_context(case), C), 0.02)}
    for i in range(case["layers"]):
        w.update({f"blocks.{i}.{k}": v for k, v in _layer_weights(g, C).items()})
    w.update({"ln_f.gamma": 1.0 + _normal(g, (C,), 0.1), "ln_f.beta": _normal(g, (C,), 0.1),
              "lm_head.weight": _normal(g, (C, V), 0.02), "lm_head.bias": _normal(g, (V,), 0.02)})
    return w


def _context(case):
    return case["T"] + case.get("n", 0)


def _inputs(case, seed):
    g = _gen(seed)
    kind = case["kind"]
    if kind == "attn":
        dt = getattr(torch, case["dtype"])
        shape = (case["B"], case["H"], case["T"], case["D"])
        q, k, v = (_normal(g, shape, 0.5 if dt == torch.bfloat16 else 1.0, dt) for _ in range(3))
        return dict(q=q, k=k, v=v, do=_normal(g, shape, 1.0, dt))
    if kind == "decode":
        dt = getattr(torch, case["dtype"])
        B, H, L, D = case["B"], case["H"], case["L"], case["D"]
        return dict(q=_normal(g, (B, H, 1, D), 1.0, dt), k=_normal(g, (B, L, H, D), 1.0, dt).transpose(1, 2),
                    v=_normal(g, (B, L, H, D), 1.0, dt).transpose(1, 2),
                    lengths=torch.randint(max(1, case["L"] // 2), case["L"] + 1, (B,), generator=g, device="cuda",
                                          dtype=torch.int32))
    if kind in ("mha", "block"):
        shape = (case["B"], case["T"], case["C"])
        return dict(x=_normal(g, shape), dy=_normal(g, shape), w=_layer_weights(g, case["C"]))
    if kind == "head":
        return dict(x=_normal(g, (case["rows"], case["C"])), w=_normal(g, (case["C"], case["V"]), 0.02),
                    b=_normal(g, (case["V"],), 0.02), labels=_ids(g, (case["rows"],), case["V"]))
    d = dict(w=_model_weights(g, case), idx=_ids(g, (case["B"], case["T"]), case["V"]))
    if kind == "train":
        d["labels"] = _ids(g, (case["B"] * case["T"],), case["V"])
    return d


# ---------------------------------------------------------------------------
# what the program has in hand, and one pass
# ---------------------------------------------------------------------------
_LR, _WARMUP = 3e-4, 2


def _load(module, weights):
    module.load_state_dict({name: _device(w) for name, w in weights.items()})
    return module


def _param_names(case, weights):
    return [n for n in weights if case["kind"] != "mha" or n.startswith("attn.")]


def _model(case, weights):
    return _load(mt.GPT(case["V"], _context(case), n_embd=case["C"], n_head=case["H"], n_layer=case["layers"]), weights)


def _seen(named):
    """Values to return of (state_dict name, value) pairs: all but the key
    bias's gradient.  Softmax does not see a constant added to a row of
    scores, so that gradient is 0 and what comes out is rounding alone."""
    return [v for n, v in named if not n.endswith("k_proj.bias")]


def prepare(case, seed):
    inp = _inputs(case, seed)
    kind = case["kind"]
    st = dict(kind=kind)
    if kind == "attn":
        for k in ("q", "k", "v", "do"):
            st[k] = _device(inp[k]).t
        st["scale"] = 1.0 / math.sqrt(case["D"])
    elif kind == "decode":
        st["q"] = _device(inp["q"]).t
        for k in ("k", "v"):  # (B, L, H, D) caches, read as (B, H, L, D)
            st[k] = _device(inp[k].transpose(1, 2)).t.transpose(1, 2)
        st["lengths"] = _device(inp["lengths"]).t
        st["scale"] = 1.0 / math.sqrt(case["D"])
    elif kind in ("mha", "block"):
        block = _load(mt.TransformerBlock(case["C"], case["H"]), inp["w"])
        st["layer"] = block.attn if kind == "mha" else block
        st["params"] = st["layer"].parameters()
        st["seen"] = _seen((n, p) for n, p in zip(_param_names(case, inp["w"]), st["params"]))
        st["x"] = mt.Tensor(_device(inp["x"]), requires_grad=True)
        st["dy"] = mt.Tensor(_device(inp["dy"]))
    elif kind == "head":
        st["layer"] = _load(mt.Linear(case["C"], case["V"]), dict(weight=inp["w"], bias=inp["b"]))
        st["params"] = st["layer"].parameters()
        st["x"] = mt.Tensor(_device(inp["x"]), requires_grad=True)
        st["labels"] = _device(inp["labels"])
    elif kind == "train":
        model = _model(case, inp["w"])
        opt = mt.Adam(model.parameters(), lr=_LR).capturable()
        idx, labels = _device(inp["idx"]), _device(inp["labels"])

        def step(i, y):
            opt.zero_grad()
            logits = model(i)
            loss = mt.cross_entropy_loss(logits.reshape(-1, case["V"]), y)
            loss.backward()
            opt.step()
            return loss, logits

        rec = mt.CapturedStep(step, optimizer=opt, warmup=_WARMUP)
        for _ in range(_WARMUP + 1):  # the eager steps and the recorded one
            loss, logits = rec(idx, labels)
        # a replay overwrites these buffers
        out = [_torch(loss.data), _torch(logits.data)] + [
            _torch(p.grad) for p in _seen(zip(inp["w"], model.parameters()))]
        st.update(step=rec, idx=idx, labels=labels, out=out, model=model)
    elif kind == "score":
        st.update(model=_model(case, inp["w"]), idx=_device(inp["idx"]))
    else:
        st.update(model=_model(case, inp["w"]), idx=inp["idx"].cpu().numpy(), n=case["n"])
    return st


def run(st):
    kind = st["kind"]
    if kind == "attn":
        o, lse = K.attn_fwd(st["q"], st["k"], st["v"], st["scale"], True)
        grads = K.attn_bwd(st["q"], st["k"], st["v"], o, st["do"], lse, st["scale"], True)
        return [_torch(a) for a in (o, lse, *grads)]
    if kind == "decode":
        o, _ = K.attn_decode(st["q"], st["k"], st["v"], st["scale"], lengths=st["lengths"])
        return [_torch(o)]
    if kind in ("mha", "block"):
        for p in [st["x"], *st["params"]]:
            p.grad = None
        y = st["layer"](st["x"])
        (y * st["dy"]).sum().backward()
        return [_torch(a) for a in (y.data, st["x"].grad, *[p.grad for p in st["seen"]])]
    if kind == "head":
        for p in [st["x"], *st["params"]]:
            p.grad = None
        logits = st["layer"](st["x"])
        loss = mt.cross_entropy_loss(logits, st["labels"])
        loss.backward()
        return [_torch(a) for a in (loss.data, logits.data, st["x"].grad, *[p.grad for p in st["params"]])]
    if kind == "train":
        st["step"](st["idx"], st["labels"])
        return st["out"]
    if kind == "score":
        with mt.no_grad():
            return [_torch(st["model"](st["idx"]).data)]
    ids, margins = st["model"].generate_greedy(st["idx"], st["n"], return_margins=True)
    return [ids, margins]


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------


def _block_flops(rows, T, C, mlp=True):
    """Forward: the four projections, the MLP, causal attention."""
    return 2.0 * rows * C * C * (12 if mlp else 4) + 2.0 * rows * T * C


def _model_flops(case, rows, T):
    return case["layers"] * _block_flops(rows, T, case["C"]) + 2.0 * rows * case["C"] * case["V"]


def _model_params(case):
    C = case["C"]
    return case["layers"] * (12 * C * C + 13 * C) + (2 * case["V"] + _context(case) + 2) * C + case["V"]


def work(case):
    kind = case["kind"]
    if kind == "attn":
        n = case["B"] * case["H"] * case["T"]
        e = 2 if case["dtype"] == "bfloat16" else 4
        # q, k, v, do in, o out, lse, three fp32 gradients
        return dict(bytes=float(n * (case["D"] * (5 * e + 12) + 4)), flops=7.0 * n * case["T"] * case["D"])
    if kind == "decode":
        n = case["B"] * case["H"]
        e = 2 if case["dtype"] == "bfloat16" else 4
        keys = 0.75 * case["L"]  # lengths spread over [L/2, L]
        return dict(bytes=n * case["D"] * e * (2 * keys + 2), flops=4.0 * n * keys * case["D"])
    if kind in ("mha", "block"):
        rows, C = case["B"] * case["T"], case["C"]
        mlp = kind == "block"
        params = (12 if mlp else 4) * C * C
        # x and dy in, y and dx out; weights in, their gradients out
        return dict(bytes=4.0 * (4 * rows * C + 2 * params), flops=3.0 * _block_flops(rows, case["T"], C, mlp)
                    + 1.0 * rows * case["T"] * C)
    if kind == "head":
        rows, C, V = case["rows"], case["C"], case["V"]
        return dict(bytes=4.0 * (2 * rows * C + 2 * C * V + rows * V), flops=6.0 * rows * C * V)
    rows = case["B"] * case["T"]
    params = _model_params(case)
    if kind == "train":
        # weights, both moments in and out, gradients out; logits out
        return dict(bytes=4.0 * (7 * params + rows * case["V"]), flops=3.0 * _model_flops(case, rows, case["T"]))
    if kind == "score":
        return dict(bytes=4.0 * (params + rows * case["V"]), flops=_model_flops(case, rows, case["T"]))
    n, B = case["n"], case["B"]
    # every token step reads the weights and the keys and values so far
    kv = sum(2 * B * case["C"] * case["layers"] * (case["T"] + i) for i in range(1, n))
    return dict(bytes=4.0 * (params * n + kv), flops=_model_flops(case, rows, case["T"])
                + (n - 1) * _model_flops(case, B, 2 * (case["T"] + n / 2)))


def tolerance(case):
    """About four times the distance from ``exact`` that the listed and some
    forty drawn cases showed."""
    kind = case["kind"]
    if case.get("dtype") == "bfloat16":
        return dict(rel=8e-3)  # seen: 2.1e-3, a bf16 result's own rounding
    if kind == "greedy":
        # seen: margins 1.6e-6.  A pick whose two best logits are closer than
        # that may go either way, and the rest of its sequence with it
        return dict(rel=1e-5, differ=0.02)
    return dict(rel={"decode": 2e-6, "attn": 4e-6, "mha": 1e-5, "block": 5e-5, "head": 1e-5, "train": 6e-5,
                     "score": 5e-6}[kind])


# ---------------------------------------------------------------------------
# the same numbers in 64 bits
# ---------------------------------------------------------------------------


def _causal(q, k, v):
    """softmax(q k^T / sqrt(D) + causal mask) v and the log-sum-exp."""
    T = q.shape[-2]
    s = torch.matmul(q, k.transpose(-1, -2).contiguous()) / math.sqrt(q.shape[-1])
    s = s.masked_fill(torch.ones(T, T, dtype=torch.bool, device=s.device).triu(1), float("-inf"))
    return torch.matmul(torch.softmax(s, -1), v), torch.logsumexp(s, -1)


def _ref_mha(x, w, H, at=""):
    B, T, C = x.shape
    heads = lambda t: t.reshape(B, T, H, C // H).transpose(1, 2).contiguous()
    q, k, v = (heads(x @ w[f"{at}attn.{p}.weight"] + w[f"{at}attn.{p}.bias"]) for p in ("q_proj", "k_proj", "v_proj"))
    o = _causal(q, k, v)[0].transpose(1, 2).reshape(B, T, C)
    return o @ w[f"{at}attn.out_proj.weight"] + w[f"{at}attn.out_proj.bias"]


def _ref_ln(x, w, at):
    return torch.nn.functional.layer_norm(x, x.shape[-1:], w[f"{at}.gamma"], w[f"{at}.beta"], 1e-5)


def _ref_block(x, w, H, at=""):
    x = x + _ref_mha(_ref_ln(x, w, f"{at}ln1"), w, H, at)
    h = _ref_ln(x, w, f"{at}ln2") @ w[f"{at}mlp.layers.0.weight"] + w[f"{at}mlp.layers.0.bias"]
    h = torch.nn.functional.gelu(h, approximate="tanh")
    return x + h @ w[f"{at}mlp.layers.2.weight"] + w[f"{at}mlp.layers.2.bias"]


def _ref_model(idx, w, case):
    x = w["tok_emb.weight"][idx] + w["pos_emb.weight"][: idx.shape[1]]
    for i in range(case["layers"]):
        x = _ref_block(x, w, case["H"], f"blocks.{i}.")
    return _ref_ln(x, w, "ln_f") @ w["lm_head.weight"] + w["lm_head.bias"]


def _f64(d, grad=False):
    return {k: v.double().requires_grad_(grad) for k, v in d.items()}


def exact(case, seed):
    inp = _inputs(case, seed)
    kind = case["kind"]
    if kind == "attn":
        outs = [[] for _ in range(5)]
        for b in range(case["B"]):  # one sequence's score matrices at a time
            q, k, v = (inp[n][b].double().requires_grad_() for n in ("q", "k", "v"))
            o, lse = _causal(q, k, v)
            g = torch.autograd.grad(o, (q, k, v), inp["do"][b].double())
            for lst, t in zip(outs, (o.detach(), lse.detach(), *g)):
                lst.append(t)
        return [torch.stack(t) for t in outs]
    if kind == "decode":
        s = (inp["q"].double() * inp["k"].double()).sum(-1) / math.sqrt(case["D"])
        at = torch.arange(case["L"], device="cuda")
        s = s.masked_fill(at >= inp["lengths"][:, None, None], float("-inf"))
        return [(torch.softmax(s, -1)[..., None] * inp["v"].double()).sum(2, keepdim=True)]
    if kind in ("mha", "block"):
        w = _f64(inp["w"], True)
        x = inp["x"].double().requires_grad_()
        y = _ref_mha(x, w, case["H"]) if kind == "mha" else _ref_block(x, w, case["H"])
        params = _seen((n, w[n]) for n in _param_names(case, w))
        return [y.detach(), *torch.autograd.grad(y, [x] + params, inp["dy"].double())]
    if kind == "head":
        x, w, b = (inp[n].double().requires_grad_() for n in ("x", "w", "b"))
        logits = x @ w + b
        loss = torch.nn.functional.cross_entropy(logits, inp["labels"])
        return [loss.detach(), logits.detach(), *torch.autograd.grad(loss, (x, w, b))]
    if kind == "train":
        w = _f64(inp["w"], True)
        m = {k: torch.zeros_like(v) for k, v in w.items()}
        v2 = {k: torch.zeros_like(v) for k, v in w.items()}
        for t in range(1, _WARMUP + 3):  # prepare's steps, then run's
            logits = _ref_model(inp["idx"], w, case)
            loss = torch.nn.functional.cross_entropy(logits.reshape(-1, case["V"]), inp["labels"])
            g = dict(zip(w, torch.autograd.grad(loss, list(w.values()))))
            with torch.no_grad():
                for k in w:
                    m[k] = 0.9 * m[k] + 0.1 * g[k]
                    v2[k] = 0.999 * v2[k] + 0.001 * g[k] ** 2
                    w[k] -= _LR * (m[k] / (1 - 0.9 ** t)) / ((v2[k] / (1 - 0.999 ** t)).sqrt() + 1e-8)
        return [loss.detach(), logits.detach(), *_seen(g.items())]
    w = _f64(inp["w"])
    with torch.no_grad():
        if kind == "score":
            return [_ref_model(inp["idx"], w, case)]
        ids, margins = inp["idx"], []
        for _ in range(case["n"]):
            top = _ref_model(ids, w, case)[:, -1].topk(2, -1)
            ids = torch.cat([ids, top.indices[:, :1]], 1)
            margins.append(top.values[:, 0] - top.values[:, 1])
        return [ids.cpu().numpy(), torch.stack(margins, 1).cpu().numpy()]
