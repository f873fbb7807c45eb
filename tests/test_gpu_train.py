"""The training operators on fp32 master tiles against the bf16 operators they fuse the casts of."""

import numpy as np
import pytest
import torch

import lbk_testlib as T

pytestmark = pytest.mark.gpu


def _weights(rng, d, ff, B, dens, dead):
    ws = []
    for w in T.ffn_weights(rng, d, ff, B, dens, sentinel_frac=dead):
        v, c = T.gpu_weight(w)
        ws += [v.float() + 1e-5 * torch.randn(v.shape, device="cuda"), c]     # not bf16 numbers
    return ws


# packed geometries (B = 16, 32), unpacked ones (B = 64, more than 2048 wide), one and several token chunks
@pytest.mark.parametrize("case", [(256, 512, 16, 0.5, 1, 0.1), (256, 1024, 32, 0.25, 70, 0.2), (512, 1024, 64, 0.25, 100, 0.1),
                                  (256, 512, 32, 0.5, 2100, 0.0), (128, 256, 64, 1.0, 2049, 0.3), (2080, 64, 32, 0.1, 5, 0.0),
                                  (128, 256, 16, 1.0, 0, 0.0)])
@pytest.mark.parametrize("bias", [False, True])
def test_train_operators_equal_cast_and_bf16_operators(gpu, case, bias):
    from looped_blockell import kernels
    d, ff, B, dens, N, dead = case
    rng = np.random.default_rng(N + d + B)
    vg, cg, vu, cu, vd, cd = _weights(rng, d, ff, B, dens, dead)
    bs = [T.to_gpu((0.1 * rng.standard_normal(n)).astype(np.float32)) if bias else None for n in (ff, ff, d)]
    x, dy = T.to_gpu_bf16(T.act(rng, N, d)), T.to_gpu_bf16(T.act(rng, N, d))
    out, h, gp, uo, wg, wu, wd = kernels.ops().block_ell_swiglu_fwd_train(x, vg, cg, bs[0], vu, cu, bs[1], vd, cd, bs[2],
                                                                          False)
    for w, v in ((wg, vg), (wu, vu), (wd, vd)):
        assert torch.equal(w, v.to(torch.bfloat16))
    ref = kernels.ops().block_ell_swiglu_fwd_bias(x, wg, cg, bs[0], wu, cu, bs[1], wd, cd, bs[2], False, True)
    assert all(torch.equal(a, b) for a, b in zip((out, h, gp, uo), ref))
    got = kernels.ops().block_ell_swiglu_bwd_train(dy, x, gp, uo, h, wg, cg, wu, cu, wd, cd, False, bias)
    want = kernels.ops().block_ell_swiglu_bwd_bias(dy, x, gp, uo, h, wg, cg, wu, cu, wd, cd, False)
    assert torch.equal(got[0], want[0])
    for a, b in zip(got[1:4], want[1:4]):
        assert a.dtype == torch.float32 and torch.equal(a.to(torch.bfloat16), b)
    if bias:
        assert all(torch.equal(a, b) for a, b in zip(got[4:], want[4:]))


def test_train_values_off_alignment(gpu):
    """fp32 tiles 4 bytes off a 16-byte boundary (views of one flat buffer) give the same step."""
    from looped_blockell import kernels
    rng = np.random.default_rng(2)
    vg, cg, vu, cu, vd, cd = _weights(rng, 128, 256, 32, 0.5, 0.1)
    flat = torch.empty(vg.numel() + 1, device="cuda")
    off = flat[1:].view(vg.shape)
    off.copy_(vg)
    x = T.to_gpu_bf16(T.act(rng, 40, 128))
    a = kernels.ops().block_ell_swiglu_fwd_train(x, vg, cg, None, vu, cu, None, vd, cd, None, True)
    b = kernels.ops().block_ell_swiglu_fwd_train(x, off, cg, None, vu, cu, None, vd, cd, None, True)
    assert all(torch.equal(p, q) for p, q in zip(a, b))


def test_layer_step_with_bf16_parameters(gpu):
    """Parameters that are bf16 themselves keep the operators on bf16 tiles and get bf16 gradients."""
    from looped_blockell.layers import MLPBlock
    torch.manual_seed(0)
    m = MLPBlock(128, 256, use_swiglu=True, tile_size=32, density=0.5, device="cuda")
    ref = MLPBlock(128, 256, use_swiglu=True, tile_size=32, density=0.5, device="cuda")
    m.load_state_dict(ref.state_dict())
    for n in ("w_gate", "w_up", "w_down"):
        getattr(m, n).values.data = getattr(ref, n).values.data.to(torch.bfloat16)
    x = torch.randn(50, 128, device="cuda").to(torch.bfloat16)
    y, yr = m(x), ref(x)
    assert torch.equal(y, yr)
    y.float().square().sum().backward()
    yr.float().square().sum().backward()
    for n in ("w_gate", "w_up", "w_down"):
        a, b = getattr(m, n).values.grad, getattr(ref, n).values.grad
        assert a.dtype == torch.bfloat16 and b.dtype == torch.float32 and torch.equal(a, b.to(torch.bfloat16))


def test_train_node_hooks_double_backward_and_transforms(gpu):
    """The native node keeps what a Python autograd function did: saved-tensor hooks see its saved
    tensors, a second derivative and functorch transforms are refused, frozen tiles get no gradient."""
    from looped_blockell.layers import MLPBlock
    torch.manual_seed(1)
    m = MLPBlock(64, 128, use_swiglu=True, tile_size=32, density=0.5, device="cuda")
    x = torch.randn(3, 5, 64, device="cuda").to(torch.bfloat16).requires_grad_(True)
    seen = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: (seen.append(t.shape), t)[1], lambda t: t):
        y = m(x)
    assert y.shape == x.shape and torch.Size([15, 128]) in seen and m.w_gate.values.shape in seen
    y.float().sum().backward()
    gx = x.grad.clone()
    x.grad = None
    m.w_up.values.requires_grad_(False)
    m.w_up.values.grad = None
    m(x).float().sum().backward()
    assert torch.equal(x.grad, gx) and m.w_up.values.grad is None and m.w_gate.values.grad is not None
    g, = torch.autograd.grad(m(x).float().sum(), x, create_graph=True)
    with pytest.raises(RuntimeError):
        torch.autograd.grad(g.float().sum(), m.w_down.values)
    with pytest.raises(RuntimeError):
        torch.func.grad(lambda t: m(t).float().sum())(x.detach())
    with torch.autograd.forward_ad.dual_level():
        with pytest.raises((RuntimeError, NotImplementedError)):
            m(torch.autograd.forward_ad.make_dual(x.detach(), torch.ones_like(x)))


def test_frozen_weights_follow_replacement(gpu):
    """Gradient-free forwards notice in-place writes, replaced parameters and replaced topologies."""
    from looped_blockell.layers import MLPBlock
    torch.manual_seed(2)
    m = MLPBlock(64, 128, use_swiglu=True, tile_size=32, density=0.5, device="cuda")
    x = torch.randn(70, 64, device="cuda").to(torch.bfloat16)

    def fresh():
        n = MLPBlock(64, 128, use_swiglu=True, tile_size=32, density=0.5, device="cuda")
        n.load_state_dict(m.state_dict())
        with torch.no_grad():
            return n(x)

    with torch.no_grad():
        first = m(x)
        m.w_gate.values.mul_(2)
        assert torch.equal(m(x), fresh()) and not torch.equal(m(x), first)
        m.w_down.values = torch.nn.Parameter(torch.randn_like(m.w_down.values) * 0.02)
        assert torch.equal(m(x), fresh())
        m.w_up.alive_mask[0, 0] = False
        assert torch.equal(m(x), fresh())
        m.w_up.col_indices = m.w_up.col_indices.flip(0).contiguous()
        assert torch.equal(m(x), fresh())
    with pytest.raises(RuntimeError):
        m(torch.zeros(4, 128, device="cuda", dtype=torch.bfloat16))


def _dense(v, c, C):
    R, K, B, _ = v.shape
    w = torch.zeros(R, C, B, B, dtype=torch.float64, device=v.device)
    for k in range(K):
        col = c[:, k].long()
        ok = (col >= 0) & (col < C)
        w[torch.arange(R, device=v.device)[ok], col[ok]] += v[ok, k].double().transpose(-1, -2)
    return w.permute(0, 2, 1, 3).reshape(R * B, C * B)


def _gelu_grad(z):
    z = z.detach().requires_grad_(True)
    y = torch.nn.functional.gelu(z, approximate="tanh")
    return torch.autograd.grad(y.sum(), z)[0]


# epilogues of the panel product (B = 16, 32, up to 2048 wide) and of the B = 64 product, and the pass
# over the product's result (wider inputs, more than 128 slots a row); the backward's panel kernel and
# the general one (d_model above 2048); one and several token chunks
@pytest.mark.parametrize("case", [(256, 512, 16, 0.5, 70), (256, 1024, 32, 0.25, 2100), (2048, 256, 32, 0.1, 33),
                                  (2176, 256, 32, 0.1, 65), (128, 2304, 16, 1.0, 20), (512, 1024, 64, 0.25, 130),
                                  (256, 512, 64, 0.5, 2), (128, 256, 32, 1.0, 0)])
def test_gelu_operators(gpu, case):
    from looped_blockell import kernels
    d, ff, B, dens, N = case
    rng = np.random.default_rng(N + d + ff)
    v1, c1, _, _, v2, c2 = _weights(rng, d, ff, B, dens, 0.1)
    v1 *= 20.0                                   # pre-activations of order 1
    b1, b2 = (T.to_gpu((0.3 * rng.standard_normal(n)).astype(np.float32)) for n in (ff, d))
    x, dy = T.to_gpu_bf16(T.act(rng, N, d)), T.to_gpu_bf16(T.act(rng, N, d))
    ops = kernels.ops()
    out, h, pre, r1, r2 = ops.block_ell_gelu_fwd_train(x, v1, c1, b1, v2, c2, b2)
    assert torch.equal(r1, v1.to(torch.bfloat16)) and torch.equal(r2, v2.to(torch.bfloat16))
    assert torch.equal(pre, ops.block_ell_matmul(x, r1, c1, b1))
    assert torch.equal(out, ops.block_ell_matmul(h, r2, c2, b2))
    # the epilogue applies GELU to the fp32 sum: the exported pre-activation differs by its bf16
    # rounding (2^-9 of it, slope at most 1.13), h by its own
    hr = torch.nn.functional.gelu(pre.double(), approximate="tanh")
    assert ((h.double() - hr).abs() <= 2.0 ** -8 * (hr.abs() + pre.double().abs()) + 1e-6).all()
    p1, p2 = ops.block_ell_matmul_prepack(r1, c1, d), ops.block_ell_matmul_prepack(r2, c2, ff)
    assert torch.equal(out, kernels.gelu_fwd_prepacked(x, p1, r1, c1, p2, r2, c2, b1, b2))
    dx, d1, d2, db1, db2 = ops.block_ell_gelu_bwd_train(dy, x, pre, h, r1, c1, r2, c2, True)
    w1, w2 = _dense(r1, c1, d // B), _dense(r2, c2, ff // B)
    da = (dy.double() @ w2) * _gelu_grad(pre.double())
    D1, D2 = da.T @ x.double(), dy.double().T @ h.double()
    # bf16 da and dx: 2^-9 each of values that add up over a row; sums in fp32
    rel = 6e-3
    for got, want in ((dx, da @ w1), (db1, da.sum(0)), (db2, dy.double().sum(0))):
        assert (got.double() - want).norm() <= rel * want.norm() + 1e-12
    for got, c, D, C in ((d1, c1, D1, d // B), (d2, c2, D2, ff // B)):
        R, K = c.shape
        tiles = D.reshape(R, B, C, B)[torch.arange(R, device=c.device)[:, None], :, c.clamp(min=0).long()]
        tiles = tiles.transpose(-1, -2) * (c >= 0)[:, :, None, None]
        assert got.dtype == torch.float32 and (got[c < 0] == 0).all()
        assert (got.double() - tiles).norm() <= rel * tiles.norm() + 1e-12
    none = ops.block_ell_gelu_bwd_train(dy, x, pre, h, r1, c1, r2, c2, False)
    assert torch.equal(none[0], dx) and none[3].numel() == 0


def test_gelu_layer_hooks_and_extremes(gpu):
    """A hook on fc1 or fc2 still sees its call; the fused forward agrees with the two layers, also at
    pre-activations where the exponential overflows."""
    from looped_blockell.layers import MLPBlock
    torch.manual_seed(4)
    m = MLPBlock(128, 256, tile_size=32, density=0.5, device="cuda")
    x = torch.randn(2, 70, 128, device="cuda").to(torch.bfloat16)
    with torch.no_grad():
        m.fc1.bias[:4] = torch.tensor([-1e15, 1e15, -60.0, 60.0])
        fused = m(x)
        seen = []
        hook = m.fc1.register_forward_hook(lambda mod, args, y: seen.append(y.shape))
        split = m(x)
        hook.remove()
    assert seen == [torch.Size([2, 70, 256])] and fused.shape == x.shape and torch.isfinite(fused).all()
    assert (fused.double() - split.double()).norm() <= 8e-3 * split.double().norm()
    m(x).float().sum().backward()
    assert all(torch.isfinite(p.grad).all() for p in m.parameters())


def _loop_pair(d, ff, B, dens, L, shared, bias):
    """A looped block, and the same one whose modules' calls are made one by one (a hook asks for it)."""
    from looped_blockell.layers import LoopedSwiGLU
    ms = []
    for _ in range(2):
        torch.manual_seed(11)
        m = LoopedSwiGLU(d, ff, L, tile_size=B, density=dens, device="cuda", bias=bias)
        with torch.no_grad():
            m.norm.scale.uniform_(0.8, 1.2)
            for lin in (m.mlp.w_gate, m.mlp.w_up, m.mlp.w_down):
                lin.values.normal_(0, 0.05)
                lin.alive_mask.copy_(torch.rand(lin.R, lin.K) >= 0.1)
                if lin.bias is not None:
                    lin.bias.normal_(0, 0.1)
            if not shared:
                m.mlp.w_up.alive_mask.copy_(torch.rand(m.mlp.w_up.R, m.mlp.w_up.K) >= 0.1)
        ms.append(m)
    ms[1].mlp.register_forward_hook(lambda *a: None)
    return ms


# state kept by the down kernel (B = 16, 32) and by a pass of its own (B = 64, wide rows); odd widths of
# the norm's kernels; one row
@pytest.mark.parametrize("case", [(256, 512, 16, 0.5, 70, 3), (256, 1024, 32, 0.25, 700, 4), (128, 256, 64, 0.5, 200, 2),
                                  (2112, 128, 64, 0.2, 20, 2), (128, 256, 32, 1.0, 1, 5), (256, 512, 32, 0.5, 33, 1)])
@pytest.mark.parametrize("bias", [False, True])
def test_looped_training_matches_the_modules(gpu, case, bias):
    d, ff, B, dens, N, L = case
    one, many = _loop_pair(d, ff, B, dens, L, shared=bias, bias=bias)
    x = torch.randn(N, d, device="cuda").to(torch.bfloat16)
    dy = torch.randn(N, d, device="cuda").to(torch.bfloat16)
    got, want = [], []
    for m, res in ((one, got), (many, want)):
        xi = x.clone().requires_grad_(True)
        y = m(xi)
        res += [y.detach(), *torch.autograd.grad(y, [xi] + list(m.parameters()), dy)]
    # the module path rounds y and the norm's gradient to bf16 at every application (2^-9 each)
    for a, b in zip(got, want):
        assert a.dtype == b.dtype and a.shape == b.shape
        assert (a.double() - b.double()).norm() <= 4e-3 * (1 + L) * b.double().norm() + 1e-12
    again = one(x.clone().requires_grad_(True))
    assert torch.equal(again, got[0])


def test_looped_training_groups_of_applications(gpu):
    """The backward's weight-gradient passes over several groups of applications (the last one shorter)
    add up: the operator on 5 applications of a size where a group holds two."""
    from looped_blockell import kernels
    rng = np.random.default_rng(6)
    d, ff, B, N, L = 64, 8192, 32, 32768, 5          # 2 GiB of dg and du: two applications
    ws = _weights(rng, d, ff, B, 0.5, 0.0)
    x = T.to_gpu_bf16(T.act(rng, N, d))
    dy = T.to_gpu_bf16(T.act(rng, N, d))
    sc = torch.ones(d, device="cuda")
    ops = kernels.ops()
    out, st, xn, h, gp, uo, wg, wu, wd = ops.looped_swiglu_fwd_train(x, sc, ws[0], ws[1], None, ws[2], ws[3], None, ws[4],
                                                                     ws[5], None, L, 1e-5)
    got = ops.looped_swiglu_bwd_train(dy, st, xn, h, gp, uo, sc, wg, ws[1], wu, ws[3], wd, ws[5], 1e-5, True)
    # the same applications one at a time, the state gradient carried in fp32
    g, tot = dy.float(), None
    for t in range(L - 1, -1, -1):
        r = ops.block_ell_swiglu_bwd_train(g.to(torch.bfloat16), xn[t], gp[t], uo[t], h[t], wg, ws[1], wu, ws[3], wd,
                                           ws[5], False, True)
        dx, ds = ops.rmsnorm_bwd(r[0], st[t], sc, 1e-5)
        g = g + dx.float()
        parts = [ds, *r[1:]]
        tot = parts if tot is None else [a + b for a, b in zip(tot, parts)]
    for a, b in zip(got, [g.to(torch.bfloat16), *tot]):
        assert (a.double() - b.double()).norm() <= 4e-3 * b.double().norm()


@pytest.mark.parametrize("kind", ["tile64", "gelu16", "gelu64", "loop16", "down16"])
def test_gradient_free_forwards_replay_from_a_graph(gpu, kind):
    """The forwards captured once replay on new inputs, with eager work between the replays."""
    from looped_blockell.layers import LoopedSwiGLU, MLPBlock
    torch.manual_seed(8)
    kw = dict(device="cuda")
    m = {"tile64": lambda: MLPBlock(256, 512, use_swiglu=True, tile_size=64, density=0.5, **kw),
         "gelu16": lambda: MLPBlock(256, 512, tile_size=16, density=0.5, **kw),
         "gelu64": lambda: MLPBlock(256, 512, tile_size=64, density=0.5, **kw),
         "loop16": lambda: LoopedSwiGLU(256, 512, 3, tile_size=16, density=0.5, **kw),
         "down16": lambda: MLPBlock(256, 2048, use_swiglu=True, tile_size=16, density=1.0, **kw)}[kind]()
    x = torch.randn(130, 256, device="cuda").to(torch.bfloat16)
    with torch.no_grad():
        m(x)
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            y = m(x)
        for k in range(3):
            x.copy_(torch.randn(130, 256, device="cuda"))
            g.replay()
            torch.cuda.synchronize()
            got = y.clone()
            assert torch.equal(got, m(x)), k
