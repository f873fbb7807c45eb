"""Backward kernels at B = 16 at the edges of their dispatch: token blocks of 32 and 64 and their
remainders, stages of 512, 1024 and 2048 columns with a short last one, output blocks that are no
multiple of a workgroup's waves, odd runs, lists past 64 entries, empty columns; and the tile
gradients' three kernels at their token chunks."""

import numpy as np
import pytest
import torch

import lbk_testlib as T

pytestmark = pytest.mark.gpu
REL = 6e-3        # bf16 dg, du and results, 2^-9 each, added over a row


def _dense(v, c, C):
    R, K, B, _ = v.shape
    w = torch.zeros(R, C, B, B, dtype=torch.float64, device=v.device)
    for k in range(K):
        col = c[:, k].long()
        ok = (col >= 0) & (col < C)
        w[torch.arange(R, device=v.device)[ok], col[ok]] += v[ok, k].double().transpose(-1, -2)
    return w.permute(0, 2, 1, 3).reshape(R * B, C * B)


def _tiles(D, c, B):
    """Dense gradient [R B, C B] -> the gradient of every live slot's tile, zeros for dead ones."""
    R, C = c.shape[0], D.shape[1] // B
    t = D.reshape(R, B, C, B)[torch.arange(R, device=c.device)[:, None], :, c.clamp(min=0).long()]
    return t.transpose(-1, -2) * (c >= 0)[:, :, None, None]


def _close(a, b):
    return (a.double() - b).norm() <= REL * b.norm() + 1e-12


# (N, block rows R, input blocks C, slots K): dx takes 32-token blocks (few workgroups) or 64-token
# blocks with 1, 2 or 4 output blocks a wave
@pytest.mark.parametrize("case", [(1, 8, 3, 2), (31, 130, 9, 3), (33, 128, 32, 16), (65, 200, 33, 33), (64, 64, 64, 64),
                                  (700, 150, 16, 16), (8200, 16, 32, 5), (16400, 20, 9, 4), (16400, 66, 24, 7),
                                  (16400, 16, 64, 64), (3000, 129, 70, 3)])
def test_product_backward(gpu, case):
    from looped_blockell import kernels
    N, R, C, K = case
    B = 16
    rng = np.random.default_rng(N + R)
    vals, col = T.bell_weight(rng, R, C, K, B)
    col[rng.random(col.shape) < 0.15] = -1
    if C > 2 * K:
        col[col == 1] = -1                                  # an input block that no slot reads
    v, c = T.gpu_weight((vals, col))
    x, dy = T.to_gpu_bf16(T.act(rng, N, C * B)), T.to_gpu_bf16(T.act(rng, N, R * B))
    dx, dv, db = kernels.ops().block_ell_matmul_bwd_bias(dy, x, v, c)
    w = _dense(v, c, C)
    ref = dy.double() @ w
    assert _close(dx, ref)
    worst = (dx.double() - ref).reshape(N, C, B).norm(dim=(0, 2))       # per output block
    assert (worst <= 2 * REL * ref.reshape(N, C, B).norm(dim=(0, 2)) + 1e-9).all()
    assert _close(dv, _tiles(dy.double().T @ x.double(), c, B)) and (dv[c < 0] == 0).all()


# gate/up weights that take the row kernel and down weights that take the transposed-list kernel, at
# chunks of 256 to 2048 tokens and their remainders, and shapes that take neither
@pytest.mark.parametrize("case", [(256, 2048, 0.5, 2000), (512, 2048, 0.5, 2000), (512, 2048, 0.25, 8200), (1024, 2048, 0.25, 1500),
                                  (256, 896, 1.0, 700), (512, 2048, 1.0, 513), (256, 1024, 0.25, 255)])
def test_swiglu_backward(gpu, case):
    from looped_blockell import kernels
    d, ff, dens, N = case
    B = 16
    rng = np.random.default_rng(N + d)
    g, u, dn = T.ffn_weights(rng, d, ff, B, dens, sentinel_frac=0.1)
    (vg, cg), (vu, cu), (vd, cd) = (T.gpu_weight(w) for w in (g, u, dn))
    x, dy = T.to_gpu_bf16(T.act(rng, N, d)), T.to_gpu_bf16(T.act(rng, N, d))
    ops = kernels.ops()
    _, h, gp, uo = ops.block_ell_swiglu_fwd_bias(x, vg, cg, None, vu, cu, None, vd, cd, None, False, True)
    dx, dvg, dvu, dvd, dbg, dbu, dbd = ops.block_ell_swiglu_bwd_train(dy, x, gp, uo, h, vg, cg, vu, cu, vd, cd, False, True)
    Wg, Wu, Wd = _dense(vg, cg, d // B), _dense(vu, cu, d // B), _dense(vd, cd, ff // B)
    G, U, dh = gp.double(), uo.double(), dy.double() @ Wd
    s = torch.sigmoid(G)
    dG, dU = dh * U * (s + G * s * (1 - s)), dh * G * s
    assert _close(dx, dG @ Wg + dU @ Wu)
    assert _close(dvg, _tiles(dG.T @ x.double(), cg, B)) and _close(dvu, _tiles(dU.T @ x.double(), cu, B))
    assert _close(dvd, _tiles(dy.double().T @ h.double(), cd, B))
    assert _close(dbg, dG.sum(0)) and _close(dbu, dU.sum(0)) and _close(dbd, dy.double().sum(0))
    again = ops.block_ell_swiglu_bwd_train(dy, x, gp, uo, h, vg, cg, vu, cu, vd, cd, False, True)
    assert all(torch.equal(a, b) for a, b in zip(again, (dx, dvg, dvu, dvd, dbg, dbu, dbd)))


# 32-token blocks, and 64-token blocks with 1, 2 and 4 output blocks a wave
@pytest.mark.parametrize("case", [(70, 40, 9, 3), (16400, 20, 9, 4), (16400, 66, 24, 7), (16400, 16, 64, 33)])
def test_infinite_gradients_stay_infinite(gpu, case):
    """An infinite gradient reaches the inputs of its block row's live tiles as an infinity of the
    weight's sign, in runs of odd and even length, and no other value."""
    from looped_blockell import kernels
    N, R, C, K = case
    B = 16
    rng = np.random.default_rng(R)
    vals, col = T.bell_weight(rng, R, C, K, B)
    col[rng.random(col.shape) < 0.15] = -1
    v, c = T.gpu_weight((vals, col))
    x, dy = T.to_gpu_bf16(T.act(rng, N, C * B)), T.to_gpu_bf16(T.act(rng, N, R * B))
    w = _dense(v, c, C)
    ref = dy.double() @ w
    for r in range(R):                                      # token r: infinite in block row r
        f = r * B + (r * 5) % B
        ref[r] = torch.where(w[f] != 0, torch.sign(w[f]) * float("inf"), ref[r] - dy[r, f].double() * w[f])
        dy[r, f] = float("inf")
    dx = kernels.ops().block_ell_matmul_bwd(dy, x, v, c)[0].double()
    assert torch.equal(torch.isinf(dx), torch.isinf(ref)) and torch.equal(dx[torch.isinf(ref)], ref[torch.isinf(ref)])
    ok = torch.isfinite(ref)
    assert not torch.isnan(dx).any() and _close(dx[ok], ref[ok])
