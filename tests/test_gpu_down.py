"""The down / wide-input product at every workgroup shape its dispatch picks (64, 32 and 16 tokens, one
and two slot chunks a row), with ragged tokens, rows and last stages, against float64 dense products;
and the looped block, whose fp32 state the same kernels update."""

import numpy as np
import pytest
import torch

import lbk_testlib as T
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _dense(v, c, C):
    R, K, B, _ = v.shape
    w = torch.zeros(R, C, B, B, dtype=torch.float64, device=v.device)
    for k in range(K):
        col = c[:, k].long()
        ok = (col >= 0) & (col < C)
        w[torch.arange(R, device=v.device)[ok], col[ok]] += v[ok, k].double().transpose(-1, -2)
    return w.permute(0, 2, 1, 3).reshape(R * B, C * B)


# inputs that are no multiple of 128 or wider than 2048 take the down kernels
@pytest.mark.parametrize("case", [
    # (B, N, block rows, input blocks, slots)
    (16, 4099, 31, 132, 128), (16, 4099, 31, 132, 9), (16, 8200, 5, 132, 64), (16, 8200, 9, 139, 100),
    (16, 2000, 17, 131, 65), (16, 17, 7, 129, 1), (16, 1, 3, 300, 128), (16, 16500, 16, 257, 2), (16, 16500, 17, 132, 40),
    (32, 3001, 30, 65, 33), (32, 700, 31, 129, 70), (32, 9000, 5, 67, 64), (32, 2338, 9, 66, 5), (32, 5, 2, 65, 1),
    (32, 5000, 8, 131, 128), (32, 16390, 17, 66, 20)])
def test_wide_product(gpu, case):
    from looped_blockell import kernels
    B, N, R, C, K = case
    rng = np.random.default_rng(N + R)
    vals, col = T.bell_weight(rng, R, C, K, B)
    col[rng.random(col.shape) < 0.1] = -1
    col[R - 1] = -1
    v, c = T.gpu_weight((vals, col))
    x = T.to_gpu_bf16(T.act(rng, N, C * B))
    b = T.to_gpu(rng.standard_normal(R * B).astype(np.float32))
    w = _dense(v, c, C)
    for bias in (None, b):
        y = kernels.block_ell_matmul(x, v, c, bias)
        ref = x.double() @ w.T + (0 if bias is None else bias.double())
        # bf16 results of fp32 sums: 2^-9 of the value, and the sum's own rounding
        assert ((y.double() - ref).abs() <= 2.0 ** -8 * ref.abs() + 1e-4 * ref.abs().amax()).all()
        assert torch.equal(y, kernels.block_ell_matmul(x, v, c, bias))


@pytest.mark.parametrize("case", [(16, 512, 2048, 0.25, 65), (16, 512, 1024, 1.0, 1100), (16, 256, 896, 0.5, 2100),
                                  (32, 256, 1024, 0.5, 300), (32, 1024, 1024, 0.25, 1300), (32, 512, 1024, 1.0, 2050)])
def test_looped_state(gpu, case):
    from looped_blockell import kernels
    B, d, ff, dens, N = case
    rng = np.random.default_rng(N)
    g, u, dn = T.ffn_weights(rng, d, ff, B, dens)
    bs = [(0.05 * rng.standard_normal(n)).astype(np.float32) for n in (ff, ff, d)]
    h = T.act(rng, N, d)
    sc = (1 + 0.1 * rng.standard_normal(d)).astype(np.float32)
    ws = [t for w in (g, u, dn) for t in T.gpu_weight(w)]
    bt = [T.to_gpu(b) for b in bs]
    out = kernels.looped_swiglu_bias(T.to_gpu_bf16(h), T.to_gpu(sc), ws[0], ws[1], bt[0], ws[2], ws[3], bt[1], ws[4], ws[5],
                                     bt[2], L=2)
    x = torch.from_numpy(h).double().cuda()
    wg, wu, wd = (_dense(ws[2 * t], ws[2 * t + 1], C) for t, C in enumerate((d // B, d // B, ff // B)))
    for _ in range(2):
        xn = x / torch.sqrt(x.pow(2).mean(-1, keepdim=True) + 1e-5) * T.to_gpu(sc).double()
        x = x + (torch.nn.functional.silu(xn @ wg.T + bt[0].double()) * (xn @ wu.T + bt[1].double())) @ wd.T + bt[2].double()
    assert (out.double() - x).norm() <= 6e-3 * x.norm()


# the ring kernel's forms at B = 16 (64 x 16, 32 x 8 with 1024 and 2048 columns, 16 x 4) and at B = 32
@pytest.mark.parametrize("case", [(16, 4099, 31, 132, 127), (16, 3001, 30, 131, 9), (16, 1500, 30, 131, 65),
                                  (16, 150, 7, 129, 33), (32, 3001, 30, 65, 33), (32, 150, 9, 66, 5)])
def test_infinite_inputs_stay_infinite(gpu, case):
    """An infinite input reaches the rows whose live tiles read its block as an infinity of the weight's
    sign, in runs of odd and even length, and no other value."""
    from looped_blockell import kernels
    B, N, R, C, K = case
    rng = np.random.default_rng(N)
    vals, col = T.bell_weight(rng, R, C, K, B)
    col[rng.random(col.shape) < 0.1] = -1
    v, c = T.gpu_weight((vals, col))
    x = T.to_gpu_bf16(T.act(rng, N, C * B))
    w = _dense(v, c, C)
    ref = x.double() @ w.T
    for t in range(min(N, C)):                              # token t: infinite in input block t
        f = t * B + (t * 5) % B
        ref[t] = torch.where(w[:, f] != 0, torch.sign(w[:, f]) * float("inf"), ref[t] - x[t, f].double() * w[:, f])
        x[t, f] = float("inf")
    y = kernels.block_ell_matmul(x, v, c, None).double()
    assert not torch.isnan(y).any()
    assert torch.equal(torch.isinf(y), torch.isinf(ref)) and torch.equal(y[torch.isinf(ref)], ref[torch.isinf(ref)])
    ok = torch.isfinite(ref)
    assert (y[ok] - ref[ok]).norm() <= 6e-3 * ref[ok].norm()
