"""Row slices of the gate/up kernels: from one row a workgroup (few tokens) to slices of uneven length, a
last round that is short, and one slice, at every form of the kernel."""

import numpy as np
import pytest
import torch

import lbk_testlib as T

pytestmark = pytest.mark.gpu


def _dense(v, c, C):
    R, K, B, _ = v.shape
    w = torch.zeros(R, C, B, B, dtype=torch.float64, device=v.device)
    for k in range(K):
        col = c[:, k].long()
        ok = (col >= 0) & (col < C)
        w[torch.arange(R, device=v.device)[ok], col[ok]] += v[ok, k].double().transpose(-1, -2)
    return w.permute(0, 2, 1, 3).reshape(R * B, C * B)


def _close(a, b):
    # a bf16 result of fp32 sums (2^-9), or the rounded gate and up products of a hidden value
    return (a.double() - b).norm() <= 6e-3 * b.norm() + 1e-9


# (B, d_model, d_ff, tokens): block rows 3 to 256, token blocks 1 to 281
@pytest.mark.parametrize("case", [(16, 128, 128, 1), (16, 256, 1024, 300), (16, 512, 4096, 70), (16, 256, 176, 4200),
                                  (32, 128, 96, 33), (32, 512, 2048, 700), (32, 256, 1056, 9000), (32, 256, 544, 17950),
                                  (32, 2048, 2080, 65), (16, 2048, 1040, 33)])
@pytest.mark.parametrize("shared", [False, True])
def test_gate_up(gpu, case, shared):
    from looped_blockell import kernels
    B, d, ff, N = case
    rng = np.random.default_rng(N)
    g, u, dn = T.ffn_weights(rng, d, ff, B, 0.4, sentinel_frac=0.1)
    if shared:
        u = (u[0], g[1])
    ws = [t for w in (g, u, dn) for t in T.gpu_weight(w)]
    if shared:
        ws[3] = ws[1]
    bs = [T.to_gpu((0.05 * rng.standard_normal(n)).astype(np.float32)) for n in (ff, ff, d)]
    x = T.to_gpu_bf16(T.act(rng, N, d))
    wg, wu, wd = (_dense(ws[2 * t], ws[2 * t + 1], C) for t, C in enumerate((d // B, d // B, ff // B)))
    for b in (None, bs):
        bg, bu, bd = b or (None, None, None)
        add = [0.0 if t is None else t.double() for t in (bg, bu, bd)]
        zg, zu = x.double() @ wg.T + add[0], x.double() @ wu.T + add[1]
        h = torch.nn.functional.silu(zg) * zu
        out, hh, gp, uo = kernels.ops().block_ell_swiglu_fwd_bias(x, ws[0], ws[1], bg, ws[2], ws[3], bu, ws[4], ws[5], bd,
                                                                  False, True)
        plain = kernels.ops().block_ell_swiglu_fwd_bias(x, ws[0], ws[1], bg, ws[2], ws[3], bu, ws[4], ws[5], bd, False,
                                                        False)[0]
        assert _close(gp, zg) and _close(uo, zu) and _close(hh, h)
        assert _close(out, h @ wd.T + add[2]) and _close(plain, h @ wd.T + add[2])
        lin = kernels.block_ell_matmul(x, ws[0], ws[1], bg)
        assert _close(lin, zg)
