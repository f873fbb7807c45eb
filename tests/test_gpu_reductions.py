"""Column-sum reductions (bias and norm-scale gradients) against float64 sums at the edges of their
row chunks, column groups and tails."""

import numpy as np
import pytest
import torch

import lbk_testlib as T
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _sum_tol(n):
    """fp32 sums of n bf16 values in strands of at most n / 8 terms: (n / 8 + 12) ulp of the sum of
    magnitudes bounds the error of any column."""
    return (n / 8 + 12) * 2.0 ** -24


# row chunks of 64 (to 8192 rows) and 256, column groups of 256, a last group of 16 and 8-wide lanes
@pytest.mark.parametrize("N", [0, 1, 7, 25, 63, 64, 65, 2000, 8192, 8193, 9000])
@pytest.mark.parametrize("out_f", [16, 256, 272, 528])
def test_matmul_bias_gradient(gpu, N, out_f):
    from looped_blockell import kernels
    rng = np.random.default_rng(N * 7 + out_f)
    B, in_f = 16, 32
    vals, col = T.bell_weight(rng, out_f // B, in_f // B, 1, B)
    v, c = T.gpu_weight((vals, col))
    x = T.to_gpu_bf16(T.act(rng, N, in_f))
    dy = T.to_gpu_bf16(T.act(rng, N, out_f))
    dx, dv, db = kernels.ops().block_ell_matmul_bwd_bias(dy, x, v, c)
    ref = dy.double().sum(0)
    bound = _sum_tol(N) * dy.double().abs().sum(0) + 1e-30
    assert db.shape == (out_f,) and db.dtype == torch.float32
    assert ((db.double() - ref).abs() <= bound).all()
    dx0, dv0 = kernels.ops().block_ell_matmul_bwd(dy, x, v, c)
    assert torch.equal(dx, dx0) and torch.equal(dv, dv0)
    assert torch.equal(db, kernels.ops().block_ell_matmul_bwd_bias(dy, x, v, c)[2])


def test_matmul_bias_gradient_keeps_nonfinite_columns(gpu):
    """An infinity or NaN in grad_out reaches its own column's sum and no other."""
    from looped_blockell import kernels
    rng = np.random.default_rng(5)
    v, c = T.gpu_weight(T.bell_weight(rng, 17, 2, 1, 16))
    x = T.to_gpu_bf16(T.act(rng, 130, 32))
    dy = T.to_gpu_bf16(T.act(rng, 130, 272))
    dy[3, 5], dy[129, 271] = float("inf"), float("nan")
    db = kernels.ops().block_ell_matmul_bwd_bias(dy, x, v, c)[2]
    assert torch.isinf(db[5]) and torch.isnan(db[271])
    rest = torch.ones(272, dtype=torch.bool, device=db.device)
    rest[[5, 271]] = False
    assert torch.isfinite(db[rest]).all()


@pytest.mark.parametrize("case", [(64, 160, 32, 8193), (80, 272, 16, 65), (192, 320, 64, 2000)])
def test_swiglu_bias_gradients_three_sums(gpu, case):
    """The three bias gradients of one backward: widths that are no multiple of a column group."""
    from looped_blockell import kernels
    d_model, d_ff, B, N = case
    rng = np.random.default_rng(N)
    g, u, d = T.ffn_weights(rng, d_model, d_ff, B, 0.5)
    ws = [t for w in (g, u, d) for t in T.gpu_weight(w)]
    x, dy = T.act(rng, N, d_model), T.act(rng, N, d_model)
    _, h, gp, uo = kernels.ops().block_ell_swiglu_fwd_bias(T.to_gpu_bf16(x), ws[0], ws[1], None, ws[2], ws[3], None,
                                                           ws[4], ws[5], None, False, True)
    db = kernels.ops().block_ell_swiglu_bwd_bias(T.to_gpu_bf16(dy), T.to_gpu_bf16(x), gp, uo, h, *ws, False)[4:]
    ref = O.swiglu_bias_grads(dy, T.to_np(gp).astype(np.float64), T.to_np(uo).astype(np.float64),
                              (d[0].astype(np.float64), d[1]))
    for got, want, tol in zip(db, ref, (1e-2, 1e-2, 1e-5)):   # dg, du are summed from bf16; dy is exact
        assert T.rel_err(T.to_np(got), want)[0] <= tol


# row widths of the register form (one lane group, two, four; a part of the last) and of the general
# form (no multiple of 8, wider than 2048, rows off 16-byte alignment)
@pytest.mark.parametrize("d", [8, 96, 512, 520, 1024, 2040, 2048, 2056, 513])
@pytest.mark.parametrize("N", [1, 5, 8, 9, 2049, 16385])
def test_rmsnorm_forward_backward_widths(gpu, N, d):
    from looped_blockell import kernels
    if N * d > 2 ** 23:
        N = 4100
    rng = np.random.default_rng(N + d)
    x, dy = T.to_gpu_bf16(T.act(rng, N, d)), T.to_gpu_bf16(T.act(rng, N, d))
    s = T.to_gpu((1 + 0.2 * rng.standard_normal(d)).astype(np.float32))
    xd, gd, sd = x.double(), dy.double(), s.double()
    rs = 1 / torch.sqrt(xd.pow(2).mean(-1, keepdim=True) + 1e-5)
    # bf16 results: half an ulp, 2^-9 of the value, plus the fp32 arithmetic before the rounding
    y = kernels.rmsnorm(x, s)
    ref = xd * rs * sd
    assert ((y.double() - ref).abs() <= 2.0 ** -8 * ref.abs() + 1e-5).all()
    dx, ds = kernels.rmsnorm_bwd(dy, x, s, 1e-5)
    t1, t2 = rs * sd * gd, xd * rs.pow(3) * (sd * gd * xd).mean(-1, keepdim=True)
    assert ((dx.double() - (t1 - t2)).abs() <= 2.0 ** -8 * (t1 - t2).abs() + 1e-5 * (1 + t1.abs() + t2.abs())).all()
    terms = gd * xd * rs
    # each term carries about 8 roundings of its own beside those of the sum
    assert ((ds.double() - terms.sum(0)).abs() <= (_sum_tol(N) + (d / 64 + 16) * 2.0 ** -24) * terms.abs().sum(0) + 1e-30).all()


def test_rmsnorm_backward_unaligned_rows(gpu):
    """Rows that start off 16-byte alignment take the general form and give the same result."""
    from looped_blockell import abi as A
    rng = np.random.default_rng(3)
    N, d = 70, 256
    s = T.to_gpu((1 + 0.2 * rng.standard_normal(d)).astype(np.float32))
    x, dy = T.to_gpu_bf16(T.act(rng, N, d)), T.to_gpu_bf16(T.act(rng, N, d))
    lib = A.load()
    wsb = lib.lbk_rmsnorm_bwd_workspace_bytes(N, d)
    outs = []
    for off in (0, 1):
        bufs = []
        for t in (x, dy, None):
            b = torch.zeros(N * d + 8, dtype=torch.bfloat16, device="cuda")
            v = b[off:off + N * d]
            if t is not None:
                v.copy_(t.reshape(-1))
            bufs.append(v)
        ds = torch.empty(d, dtype=torch.float32, device="cuda")
        ws = torch.empty(wsb, dtype=torch.uint8, device="cuda")
        A.check(lib.lbk_rmsnorm_bwd_bf16(T.ptr(bufs[0]), T.ptr(bufs[1]), N, d, T.ptr(s), 1e-5, T.ptr(bufs[2]),
                                         T.ptr(ds), T.ptr(ws), wsb, T.stream()), "rmsnorm_bwd")
        outs.append((bufs[2].clone(), ds))
    assert T.rel_err(T.to_np(outs[1][0]), T.to_np(outs[0][0]))[0] <= 2.0 ** -8
    assert T.rel_err(T.to_np(outs[1][1]), T.to_np(outs[0][1]))[0] <= 1e-5
