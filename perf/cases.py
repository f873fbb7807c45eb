"""The measured cases of the framework: its FFN layers as a user's program calls them.

Each case is one call (or one training step) of a public layer -- ``MLPBlock`` (SwiGLU and GELU),
``LoopedSwiGLU``, ``TernaryMLPBlock`` -- at sizes taken from the repository's benchmark, tests and
the reference's configurations.  ``listed()`` holds the fixed ones, ``draw(rng)`` gives more of the
same ranges:

  d_model   256 .. 2048 (bf16 tiles of 16, 32, 64), 4096 with tiles of 64; d_ff = 3.5 or 4 d_model
  density   0.1 .. 1.0 of the column blocks of a row
  tokens    1 .. 16384, odd counts included
  kinds     inference, training step (forward + backward), looped inference and training, ternary
"""

from __future__ import annotations

import os
import sys

_PKG = os.path.join(os.getcwd(), "looped-blockell-tpu_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import torch

from looped_blockell.layers import (LoopedSwiGLU, MLPBlock, TernaryBlockELLWeight, TernaryMLPBlock,
                                    create_random_topology)

_DEV = "cuda"
# most work of a drawn case (the largest listed one takes 8.2e11)
_MAX_DRAW_FLOPS = 1.5e11


def _case(name, kind, d_model, d_ff, tile, density, tokens, *, act="swiglu", bias=True, shared=True, dead=0.0, loops=1):
    """kind: infer | train | loop_infer | loop_train | ternary.  shared: gate and up keep the one
    topology they start with; else each has its own, as after regrowth.  dead: share of pruned
    (masked) slots."""
    c = dict(kind=kind, act=act, d_model=d_model, d_ff=d_ff, tile=tile, density=density, tokens=tokens, bias=bias,
             shared=shared, dead=dead, loops=loops)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # generating one token with a small model: launches and host work only
        _case("decode_1_b32", "infer", 1024, 4096, 32, 0.25, 1, shared=False),
        # a batch of 16 sequences generating with a wide model, weights streamed from memory
        _case("decode_16_b64", "infer", 4096, 14336, 64, 0.10, 16, bias=False, shared=False),
        # reading the prompts of that wide model
        _case("prefill_2k_b64", "infer", 4096, 14336, 64, 0.10, 2048, bias=False, shared=False),
        # scoring a large batch with pruned weights (the benchmark's headline layer)
        _case("score_16k_b32", "infer", 1024, 4096, 32, 0.25, 16384, bias=False, shared=False),
        # evaluating the reference's dense-start tile-16 model on a batch of odd size
        _case("eval_4k_b16", "infer", 512, 2048, 16, 1.0, 4099),
        # the default layer of the API: GELU, tile 16
        _case("gelu_8k_b16", "infer", 1024, 4096, 16, 0.25, 8192, act="gelu"),
        # one training step of the headline layer, 32 sequences of 512
        _case("train_16k_b32", "train", 1024, 4096, 32, 0.25, 16384),
        # training the tile-16 model with pruned slots, a micro-batch of ragged length
        _case("train_2k_b16", "train", 512, 2048, 16, 0.5, 2000, shared=False, dead=0.1),
        # training the GELU layer
        _case("train_gelu_4k_b32", "train", 1024, 4096, 32, 0.25, 4096, act="gelu"),
        # the looped model's core at inference: 8 applications, 32 sequences of 512
        _case("loop8_16k_b32", "loop_infer", 1024, 4096, 32, 0.25, 16384, bias=False, shared=False, loops=8),
        # training through 4 applications of the looped tile-16 block, 4 sequences of 512
        _case("loop4_train_2k_b16", "loop_train", 512, 2048, 16, 0.5, 2048, loops=4),
        # the ternary layer on a batch of prompts
        _case("ternary_8k_b64", "ternary", 2048, 8192, 64, 0.125, 8192, bias=False, shared=False),
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    while True:
        kind = rng.choice(["infer", "infer", "infer", "train", "train", "loop_infer", "loop_train", "ternary"])
        act = rng.choice(["swiglu", "swiglu", "gelu"]) if kind in ("infer", "train") else "swiglu"
        if kind == "ternary":
            d_model, tile, density = rng.choice([512, 1024, 2048]), 64, rng.choice([0.125, 0.25])
        elif kind == "infer" and rng.random() < 0.3:
            d_model, tile, density, act = 4096, 64, rng.choice([0.1, 0.25]), "swiglu"
        else:
            d_model = rng.choice([256, 512, 768, 1024, 2048])
            tile = rng.choice([16, 32, 32, 64])
            density = rng.choice([0.1, 0.25, 0.25, 0.5, 1.0])
        d_ff = rng.choice([7 * d_model // 2, 4 * d_model])
        d_ff = d_ff // 128 * 128
        tokens = _log_int(rng, 64 if "train" in kind else 1, 16384)
        loops = rng.randint(2, 8) if kind.startswith("loop") else 1
        c = _case(None, kind, d_model, d_ff, tile, density, tokens, act=act, bias=kind != "ternary" and rng.random() < 0.7,
                  shared=kind != "ternary" and rng.random() < 0.5, dead=0.1 if kind == "train" and rng.random() < 0.3 else 0.0,
                  loops=loops)
        if act == "gelu":
            c["bias"] = True      # the GELU layer's products always carry their biases
        if work(c)["flops"] <= _MAX_DRAW_FLOPS:
            return c


# ------------------------------------------------------------------ geometry
def _weights_geometry(c):
    """(name, block rows, column blocks, slots per row) of the layer's weights."""
    B, d, ff = c["tile"], c["d_model"], c["d_ff"]
    rf, rm = ff // B, d // B
    kf, km = max(1, int(rm * c["density"])), max(1, int(rf * c["density"]))
    if c["act"] == "gelu":
        return [("fc1", rf, rm, kf), ("fc2", rm, rf, km)]
    return [("w_gate", rf, rm, kf), ("w_up", rf, rm, kf), ("w_down", rm, rf, km)]


def work(c):
    B, N, d, ff = c["tile"], c["tokens"], c["d_model"], c["d_ff"]
    geo = _weights_geometry(c)
    tiles = sum(R * K for _, R, _, K in geo)
    index = 4 * tiles
    flops = 2.0 * N * tiles * B * B * c["loops"]
    if c["kind"] == "ternary":
        return {"bytes": 4.0 * N * d + tiles * (B * B / 4.0 + 4) + index, "flops": flops}
    if c["kind"] in ("infer", "loop_infer"):      # x in, result out, bf16 weights once
        return {"bytes": 4.0 * N * d + 2.0 * tiles * B * B + index, "flops": flops}
    # training: x and the result's gradient in, result and the input's gradient out; fp32 weights
    # in and their fp32 gradients out; forward, input-gradient and weight-gradient products
    return {"bytes": 8.0 * N * d + 8.0 * tiles * B * B + index, "flops": 3.0 * flops}


# ------------------------------------------------------------------ inputs
def _gen(seed, device=_DEV):
    return torch.Generator(device=device).manual_seed(int(seed) & 0x7FFFFFFF)


@torch.no_grad()
def _fill_linear(lin, c, g, gc):
    lin.values.normal_(0.0, 0.02, generator=g)
    if lin.bias is not None:
        lin.bias.normal_(0.0, 0.02, generator=g)
    if c["dead"] > 0.0:
        lin.alive_mask.copy_(torch.rand(lin.R, lin.K, generator=gc) >= c["dead"])


@torch.no_grad()
def _mlp(c, mlp, g, gc):
    lins = [getattr(mlp, n) for n, *_ in _weights_geometry(c)]
    for lin in lins:
        if lin.K < lin.C:
            lin.col_indices.copy_(create_random_topology(lin.R, lin.C, lin.K, gc))
        _fill_linear(lin, c, g, gc)
    if c["act"] == "swiglu" and c["shared"]:
        mlp.w_up.col_indices.copy_(mlp.w_gate.col_indices)
        mlp.w_up.alive_mask.copy_(mlp.w_gate.alive_mask)
    return mlp


def prepare(c, seed):
    g, gc = _gen(seed), _gen(seed + 1, "cpu")
    d, ff, B, N = c["d_model"], c["d_ff"], c["tile"], c["tokens"]
    st = {"kind": c["kind"]}
    x = torch.randn(N, d, device=_DEV, generator=g)
    if c["kind"] == "ternary":
        # weights {-1, 0, +1} with equal probability, one scale per tile near the mean |w| of N(0, 0.02)
        parts, tri = [], []
        for _, R, C, K in _weights_geometry(c):
            codes = torch.randint(-1, 2, (R, K, B, B), device=_DEV, dtype=torch.int8, generator=g)
            scales = 0.016 * (0.9 + 0.2 * torch.rand(R, K, device=_DEV, generator=g))
            cols = create_random_topology(R, C, K, gc).to(_DEV)
            parts.append(TernaryBlockELLWeight.from_codes(codes, scales, cols))
            tri.append((codes, scales, cols))
        st["codes"] = tri
        st["model"] = TernaryMLPBlock(*parts)
        st["x"] = x.to(torch.bfloat16)
        return st
    kw = dict(tile_size=B, density=c["density"], device=_DEV, bias=c["bias"])
    if c["kind"].startswith("loop"):
        m = LoopedSwiGLU(d, ff, c["loops"], **kw)
        with torch.no_grad():
            m.norm.scale.uniform_(0.8, 1.2, generator=g)
        _mlp(c, m.mlp, g, gc)
    else:
        m = _mlp(c, MLPBlock(d, ff, use_swiglu=c["act"] == "swiglu", **kw), g, gc)
    st["model"] = m
    st["x"] = x.to(torch.bfloat16)
    if "train" in c["kind"]:
        st["x"].requires_grad_(True)
        st["params"] = [(n, p) for n, p in m.named_parameters()]
        st["dy"] = torch.randn(N, d, device=_DEV, generator=g).to(torch.bfloat16)
    return st


def run(st):
    m, x = st["model"], st["x"]
    if "train" not in st["kind"]:
        with torch.inference_mode():
            return {"out": m(x)}
    out = m(x)
    grads = torch.autograd.grad(out, [x] + [p for _, p in st["params"]], st["dy"])
    res = {"out": out.detach(), "dx": grads[0]}
    for (n, _), gr in zip(st["params"], grads[1:]):
        res["d_" + n] = gr
    return res


# ------------------------------------------------------------------ precision
def tolerance(c):
    # About four times the error against 64 bits that the layers show.  Two correct bf16
    # implementations differ by the rounding of the hidden state and of the result (2.2e-3 of the
    # whole output); gradients also carry the rounded dg and du (2.9e-3); a looped block's state
    # stays in fp32 (1.7e-3).  The ternary layer re-quantises its hidden state to int8, where a
    # rounding that goes the other way moves a value by one step (9.6e-3).
    if c["kind"] == "ternary":
        return {"rel": 3e-2}
    if c["kind"] in ("infer", "loop_infer"):
        return {"rel": 8e-3}
    return {"rel": 1.2e-2}


def _dense(values, cols, alive, C):
    """[R, K, B_in, B_out] tiles -> dense [R * B, C * B] (differentiable)."""
    R, K, B, _ = values.shape
    v = values.transpose(-1, -2)
    if alive is not None:
        v = v * alive[:, :, None, None].to(v.dtype)
    rows = torch.arange(R, device=cols.device)[:, None].expand(R, K)
    w = torch.zeros(R, C, B, B, dtype=v.dtype, device=v.device).index_put((rows, cols.long()), v, accumulate=True)
    return w.permute(0, 2, 1, 3).reshape(R * B, C * B)


def _quant(x):
    m = x.abs().amax(-1, keepdim=True).clamp_min(1e-8)
    return (x * (128.0 / m)).round().clamp(-128, 127), m / 128.0


def exact(c, seed):
    st = prepare(c, seed)
    x = st["x"].detach().double()
    if c["kind"] == "ternary":
        wg, wu, wd = [_dense(t.double() * s.double()[:, :, None, None], cols, None, C)
                      for (t, s, cols), (_, _, C, _) in zip(st["codes"], _weights_geometry(c))]
        q, sx = _quant(x)
        h = torch.nn.functional.silu(q @ wg.T * sx) * (q @ wu.T * sx)
        qh, sh = _quant(h)
        return {"out": qh @ wd.T * sh}
    m = st["model"]
    train = "train" in c["kind"]
    loop = c["kind"].startswith("loop")
    mlp = m.mlp if loop else m
    leaves, dense = {}, {}
    for n, _, C, _ in _weights_geometry(c):
        lin = getattr(mlp, n)
        # the layer computes with its weights in bf16
        v = lin.values.detach().to(torch.bfloat16).double().requires_grad_(train)
        b = None if lin.bias is None else lin.bias.detach().double().requires_grad_(train)
        pre = ("mlp." if loop else "") + n
        leaves[pre + ".values"], leaves[pre + ".bias"] = v, b
        dense[n] = (_dense(v, lin.col_indices, lin.alive_mask, C), b)
    x.requires_grad_(train)

    def ffn(z):
        def lin(n, t):
            return torch.nn.functional.linear(t, *dense[n])
        if c["act"] == "gelu":
            return lin("fc2", torch.nn.functional.gelu(lin("fc1", z), approximate="tanh"))
        return lin("w_down", torch.nn.functional.silu(lin("w_gate", z)) * lin("w_up", z))

    with torch.set_grad_enabled(train):
        if loop:
            sc = m.norm.scale.detach().double().requires_grad_(train)
            leaves["norm.scale"] = sc
            out = x
            for _ in range(c["loops"]):
                out = out + ffn(out / torch.sqrt(out.pow(2).mean(-1, keepdim=True) + m.norm.eps) * sc)
        else:
            out = ffn(x)
    res = {"out": out.detach()}
    if train:
        names = [n for n, _ in st["params"]]
        grads = torch.autograd.grad(out, [x] + [leaves[n] for n in names], st["dy"].double())
        res["dx"] = grads[0]
        for n, gr in zip(names, grads[1:]):
            res["d_" + n] = gr
    return res
