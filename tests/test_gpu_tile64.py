"""The B = 64 product kernels (more tokens than the decode kernels take) against float64 dense
products: token blocks of 64, 128 and 256 with remainders, block rows that are and are not a
multiple of 8, slot lists past one 64-entry window, dead slots, rows without a live slot."""

import numpy as np
import pytest
import torch

import lbk_testlib as T

pytestmark = pytest.mark.gpu
# bf16 results of fp32 sums: half an ulp (2^-9 of the value) and the sums' own rounding, with room
# for the bf16 hidden state's rounding carried through the down product (2^-9 of a norm)
REL = 6e-3


def _dense(v, c, C):
    """[R, K, B_in, B_out] tiles -> float64 dense [out, in]."""
    R, K, B, _ = v.shape
    w = torch.zeros(R, C, B, B, dtype=torch.float64, device=v.device)
    for k in range(K):
        col = c[:, k].long()
        ok = (col >= 0) & (col < C)
        w[torch.arange(R, device=v.device)[ok], col[ok]] += v[ok, k].double().transpose(-1, -2)
    return w.permute(0, 2, 1, 3).reshape(R * B, C * B)


def _weight(rng, R, C, K, dead=0.0, dead_row=None):
    vals, col = T.bell_weight(rng, R, C, K, 64)
    if dead:
        col[rng.random(col.shape) < dead] = -1
    if dead_row is not None:
        col[dead_row] = -1
    return T.gpu_weight((vals, col))


def _close(got, want):
    return (got.double() - want).norm() <= REL * want.norm() + 1e-12


# (N, block rows, input blocks, slots): grids that take token blocks of 64, 128 and 256
@pytest.mark.parametrize("N,R,C,K", [(1, 3, 2, 1), (64, 8, 4, 2), (65, 5, 6, 6), (127, 8, 3, 3), (700, 16, 80, 80),
                                     (16385, 3, 4, 2), (8191, 8, 5, 3), (32770, 4, 2, 2)])
@pytest.mark.parametrize("bias", [False, True])
def test_product(gpu, N, R, C, K, bias):
    from looped_blockell import kernels
    rng = np.random.default_rng(N + K)
    v, c = _weight(rng, R, C, K, dead=0.2, dead_row=R - 1)
    x = T.to_gpu_bf16(T.act(rng, N, C * 64))
    b = T.to_gpu(rng.standard_normal(R * 64).astype(np.float32)) if bias else None
    y = kernels.block_ell_matmul(x, v, c, b)
    ref = x.double() @ _dense(v, c, C).T + (b.double() if bias else 0.0)
    assert _close(y, ref)
    rows = (y.double() - ref).abs().amax(0)            # a wrong column cannot hide in the norm
    assert (rows <= 2.0 ** -7 * ref.abs().amax(0) + 1e-5).all()


@pytest.mark.parametrize("N", [65, 130, 512, 4099])
@pytest.mark.parametrize("geo", [(256, 896, 4, 7), (512, 2048, 3, 9), (576, 1024, 9, 16)])
@pytest.mark.parametrize("shared", [False, True])
def test_swiglu_and_intermediates(gpu, N, geo, shared):
    from looped_blockell import kernels
    d, ff, K, Kd = geo
    rng = np.random.default_rng(N + d)
    g = _weight(rng, ff // 64, d // 64, K, dead=0.1, dead_row=1)
    u = (g[0].flip(0).contiguous(), g[1]) if shared else _weight(rng, ff // 64, d // 64, K, dead=0.1, dead_row=2)
    dn = _weight(rng, d // 64, ff // 64, Kd, dead=0.1)
    bs = [T.to_gpu((0.1 * rng.standard_normal(n)).astype(np.float32)) for n in (ff, ff, d)]
    x = T.to_gpu_bf16(T.act(rng, N, d))
    wg, wu, wd = (_dense(*w, C) for w, C in ((g, d // 64), (u, d // 64), (dn, ff // 64)))
    G, U = x.double() @ wg.T + bs[0].double(), x.double() @ wu.T + bs[1].double()
    H = torch.nn.functional.silu(G) * U
    out, h, gp, uo = kernels.ops().block_ell_swiglu_fwd_bias(x, *g, bs[0], *u, bs[1], *dn, bs[2], True, True)
    for got, want in ((gp, G), (uo, U), (h, H), (out, H @ wd.T + bs[2].double() + x.double())):
        assert _close(got, want)
    plain = kernels.ops().block_ell_swiglu_fwd_bias(x, *g, bs[0], *u, bs[1], *dn, bs[2], True, False)[0]
    assert torch.equal(plain, out)


def test_unaligned_tiles_take_the_rowblock_kernel(gpu):
    """Tiles 8 bytes off a 16-byte boundary: the same product from the general kernel."""
    from looped_blockell import kernels
    rng = np.random.default_rng(9)
    v, c = _weight(rng, 4, 6, 3)
    buf = torch.empty(v.numel() + 8, dtype=torch.bfloat16, device="cuda")
    off = buf[4:4 + v.numel()].view(v.shape)
    off.copy_(v)
    x = T.to_gpu_bf16(T.act(rng, 200, 6 * 64))
    assert _close(kernels.block_ell_matmul(x, off, c), x.double() @ _dense(v, c, 6).T)


# the transposed product of the backward: token blocks of 64, 128 and 256, one and two sources, lists past
# one 64-entry window, an input block that no slot reads, output blocks that are no multiple of 8
@pytest.mark.parametrize("case", [(1, 3, 2, 1), (65, 8, 5, 3), (700, 80, 16, 16), (3000, 40, 17, 9), (8200, 20, 12, 5),
                                  (127, 130, 3, 3)])
def test_product_backward(gpu, case):
    from looped_blockell import kernels
    N, R, C, K = case
    rng = np.random.default_rng(N)
    vals, col = T.bell_weight(rng, R, C, K, 64)
    col[rng.random(col.shape) < 0.15] = -1
    if C > 2 * K:
        col[col == 1] = -1
    v, c = T.gpu_weight((vals, col))
    x, dy = T.to_gpu_bf16(T.act(rng, N, C * 64)), T.to_gpu_bf16(T.act(rng, N, R * 64))
    dx, _ = kernels.ops().block_ell_matmul_bwd(dy, x, v, c)
    ref = dy.double() @ _dense(v, c, C)
    assert ((dx.double() - ref).abs() <= 2.0 ** -8 * ref.abs() + 1e-4 * ref.abs().amax()).all()


@pytest.mark.parametrize("N", [130, 2100])
def test_swiglu_backward_two_sources(gpu, N):
    from looped_blockell import kernels
    d, ff = 512, 1024
    rng = np.random.default_rng(N)
    g, u, dn = (_weight(rng, *s, dead=0.1) for s in ((ff // 64, d // 64, 5), (ff // 64, d // 64, 5), (d // 64, ff // 64, 7)))
    x, dy = T.to_gpu_bf16(T.act(rng, N, d)), T.to_gpu_bf16(T.act(rng, N, d))
    ops = kernels.ops()
    _, h, gp, uo = ops.block_ell_swiglu_fwd_with_intermediate(x, *g, *u, *dn, True)
    wg, wu, wd = (_dense(*w, C) for w, C in ((g, d // 64), (u, d // 64), (dn, ff // 64)))
    G, U, dh = gp.double(), uo.double(), dy.double() @ wd
    s = torch.sigmoid(G)
    ref = (dh * U * (s + G * s * (1 - s))) @ wg + (dh * G * s) @ wu
    for res in (False, True):
        dx = ops.block_ell_swiglu_bwd_ex(dy, x, gp, uo, h, *g, *u, *dn, res)[0]
        assert _close(dx, ref + (dy.double() if res else 0))


# slot lists past one 64-entry window: gate ending within the first window with up running on into the
# second (40 a side), gate itself crossing it (70 a side); rows without a live gate or up slot
@pytest.mark.parametrize("K", [40, 70])
@pytest.mark.parametrize("N", [70, 520])
def test_gate_up_over_windows(gpu, K, N):
    from looped_blockell import kernels
    d, ff = 72 * 64, 5 * 64
    rng = np.random.default_rng(N + K)
    g = _weight(rng, 5, 72, K, dead=0.1, dead_row=1)
    u = _weight(rng, 5, 72, K, dead=0.1, dead_row=2)
    dn = _weight(rng, 72, 5, 3, dead=0.1)
    x = T.to_gpu_bf16(T.act(rng, N, d))
    wg, wu, wd = (_dense(*w, C) for w, C in ((g, 72), (u, 72), (dn, 5)))
    G, U = x.double() @ wg.T, x.double() @ wu.T
    out, h, gp, uo = kernels.ops().block_ell_swiglu_fwd_with_intermediate(x, *g, *u, *dn, False)
    H = torch.nn.functional.silu(G) * U
    for got, want in ((gp, G), (uo, U), (h, H), (out, H @ wd.T)):
        assert _close(got, want)
    for got, want in ((gp, G), (uo, U)):               # per block row
        e = (got.double() - want).reshape(N, 5, 64).norm(dim=(0, 2))
        assert (e <= REL * want.reshape(N, 5, 64).norm(dim=(0, 2)) + 1e-9).all()


@pytest.mark.parametrize("N", [70, 520])
def test_two_source_lists_over_windows(gpu, N):
    """dx lists of about 45 gate and 45 up entries: the boundary of the two sources lies within the first
    64-entry window and up crosses into the second; one input block that no gate slot reads."""
    from looped_blockell import kernels
    d, ff = 3 * 64, 135 * 64
    rng = np.random.default_rng(N)
    vg, cg = T.bell_weight(rng, 135, 3, 1, 64)
    cg[cg == 1] = -1
    g, u, dn = T.gpu_weight((vg, cg)), _weight(rng, 135, 3, 1, dead=0.05), _weight(rng, 3, 135, 30, dead=0.1)
    x, dy = T.to_gpu_bf16(T.act(rng, N, d)), T.to_gpu_bf16(T.act(rng, N, d))
    ops = kernels.ops()
    _, h, gp, uo = ops.block_ell_swiglu_fwd_with_intermediate(x, *g, *u, *dn, True)
    wg, wu, wd = (_dense(*w, C) for w, C in ((g, 3), (u, 3), (dn, 135)))
    G, U, dh = gp.double(), uo.double(), dy.double() @ wd
    s = torch.sigmoid(G)
    ref = (dh * U * (s + G * s * (1 - s))) @ wg + (dh * G * s) @ wu
    dx = ops.block_ell_swiglu_bwd_ex(dy, x, gp, uo, h, *g, *u, *dn, False)[0]
    for c in range(3):
        assert _close(dx[:, 64 * c:64 * c + 64], ref[:, 64 * c:64 * c + 64]), c


@pytest.mark.parametrize("case", [(1, 3, 2), (300, 14, 4), (3000, 14, 4), (10, 40, 32)])
def test_one_slot_products(gpu, case):
    """Products of one slot a row take the row-block kernel, with and without a live slot."""
    from looped_blockell import kernels
    N, R, C = case
    rng = np.random.default_rng(N)
    v, c = _weight(rng, R, C, 1, dead=0.1, dead_row=R - 1)
    x, b = T.to_gpu_bf16(T.act(rng, N, C * 64)), T.to_gpu(rng.standard_normal(R * 64).astype(np.float32))
    ref = x.double() @ _dense(v, c, C).T + b.double()
    y = kernels.block_ell_matmul(x, v, c, b)
    assert _close(y, ref) and torch.equal(y[:, -64:], b[-64:].to(torch.bfloat16).expand(N, 64))
