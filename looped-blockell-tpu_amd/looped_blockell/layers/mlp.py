"""Block-ELL MLP layers (PyTorch), mirroring the reference's Flax module.

Reference: ``looped_blockell/layers/mlp.py``.

Weight layout per projection:
  values:      [R, K, B, B] parameter (tiles [B_in, B_out]), init N(0, 0.02)
  col_indices: [R, K] int32 buffer (topology, updated externally by pruning)
  alive_mask:  [R, K] bool buffer; dead tiles contribute nothing
  bias:        [out_features] parameter, zeros (BlockELLLinear only)

``MLPBlock(use_swiglu=True)`` runs the whole SwiGLU FFN as one fused HIP
operator (``titan::block_ell_swiglu_fwd_bias``, differentiable through
``titan::block_ell_swiglu_bwd_bias``); each projection carries a zero-initialised
trainable bias, as every ``BlockELLLinear`` of the reference's Flax module does
(``mlp.py:56-60``, ``:82``), added in fp32 in the kernels' epilogues.  ``bias=False``
gives the bias-free form of the reference's PyTorch mirror (``interop/pt_model.py:865-867``)
and CUDA operator (``csrc/block_ell/swiglu_fwd.cuh:75-84``).  The GELU form uses the tanh
approximation, ``jax.nn.gelu``'s default (``mlp.py:156``).

Forwards that need no gradient (``torch.no_grad()`` / ``torch.inference_mode()``) run from
weights prepared once per weight version: the bf16 tiles and their fragment-major packed copy
(``titan::block_ell_swiglu_prepack``, ``titan::block_ell_matmul_prepack`` for ``BlockELLLinear``)
are cached on the module and rebuilt when a value tensor,
a column-index buffer or an alive mask changes (tensor version counters), so such a forward is
the gate/up and down launches only.  Writes through ``.data`` bypass the version counter: call
``release_inference_cache()`` after them.  The cache holds about two bytes per weight element
twice (bf16 tiles, packed tiles); ``release_inference_cache()`` drops it.

The GELU form is one operator too (``titan::block_ell_gelu_fwd_prepacked``, ``..._gelu_train``)
unless a hook, a subclass or a replaced method of ``fc1`` / ``fc2`` has to see the two calls.
"""

from __future__ import annotations

import torch
import torch.nn.functional as F
from torch import nn

from .. import kernels
from .block_ell import BlockELLConfig, BlockELLTensor, create_random_topology


def _tensors(lin):
    """(values, col_indices, alive_mask) of a projection, without ``nn.Module``'s attribute lookup
    (about 0.4 us a name, and a small forward reads nine)."""
    try:
        b = lin._buffers
        return lin._parameters["values"], b["col_indices"], b["alive_mask"]
    except KeyError:                                     # replaced by plain attributes (weight norm)
        return lin.values, lin.col_indices, lin.alive_mask


def _versions(lins):
    """Pointer and version of every value tensor, column-index buffer and alive mask of ``lins``."""
    key = []
    for lin in lins:
        v, c, a = _tensors(lin)
        key += (v.data_ptr(), v._version, c.data_ptr(), c._version, a.data_ptr(), a._version)
    return key


_HOOKS = ("_forward_hooks", "_forward_pre_hooks", "_backward_hooks", "_backward_pre_hooks")


def _plain(mod, cls):
    """Whether calling ``mod`` does no more than ``cls.forward``: no subclass, no replaced method, no
    hooks on it or on every module."""
    d = mod.__dict__
    g = nn.modules.module
    return (type(mod) is cls and "forward" not in d and "kernel_values" not in d
            and not any(d[h] for h in _HOOKS) and not any(getattr(g, "_global" + h) for h in _HOOKS))


class BlockELLLinear(nn.Module):
    """Single Block-ELL linear layer (reference ``mlp.py:28-95``).

    ``K = max(1, int(C * density))``; at density 1.0 the topology is sequential,
    otherwise random and seeded from ``hash((out_features, in_features))`` so
    that layers of equal shape start with the same topology, as in the
    reference (``mlp.py:84-95``).
    """

    def __init__(self, out_features: int, in_features: int, tile_size: int = 16, density: float = 1.0,
                 dtype: torch.dtype = torch.bfloat16, bias: bool = True, device=None):
        super().__init__()
        B = tile_size
        if out_features % B or in_features % B:
            raise ValueError("features must be multiples of tile_size")
        self.out_features, self.in_features, self.tile_size = out_features, in_features, B
        self.density, self.dtype = density, dtype
        self.R, self.C = out_features // B, in_features // B
        self.K = max(1, int(self.C * density))
        self.values = nn.Parameter(torch.randn(self.R, self.K, B, B, device=device) * 0.02)
        self.bias = nn.Parameter(torch.zeros(out_features, device=device)) if bias else None
        self.register_buffer("col_indices", self._init_topology().to(device))
        self.register_buffer("alive_mask", torch.ones(self.R, self.K, dtype=torch.bool, device=device))
        self._eff_cache = None
        self._frozen = None

    def _init_topology(self) -> torch.Tensor:
        if self.density >= 1.0:
            return torch.arange(self.C, dtype=torch.int32).repeat(self.R, 1)[:, :self.K].contiguous()
        seed = hash((self.out_features, self.in_features)) % 2 ** 31
        return create_random_topology(self.R, self.C, self.K, seed)

    @property
    def config(self) -> BlockELLConfig:
        return BlockELLConfig(R=self.R, C=self.C, K=self.K, B=self.tile_size)

    def effective_col_indices(self) -> torch.Tensor:
        """col_indices with dead tiles (alive_mask False) set to the -1 sentinel (cached per version)."""
        _, cols, alive = _tensors(self)
        key = (cols.data_ptr(), cols._version, alive.data_ptr(), alive._version)
        if self._eff_cache is None or self._eff_cache[0] != key:
            # an ordinary tensor even when built under inference mode: a later forward with
            # gradients saves it for the backward
            with torch.inference_mode(False):
                eff = torch.where(alive, cols, torch.full_like(cols, -1))
                self._eff_cache = (key, eff.to(torch.int32).contiguous())
        return self._eff_cache[1]

    def kernel_values(self) -> torch.Tensor:
        return self.values.to(torch.bfloat16)

    def as_block_ell(self) -> BlockELLTensor:
        return BlockELLTensor(self.kernel_values(), self.effective_col_indices(), self.config)

    def _frozen_weight(self):
        """(bf16 tiles, effective columns, packed copy), rebuilt when the values or the topology change."""
        key = _versions((self,))
        if self._frozen is None or self._frozen[0] != key:
            cols = self.effective_col_indices()
            with torch.inference_mode(False):
                v = self.kernel_values()
                self._frozen = (key, v, cols, kernels.block_ell_matmul_prepack(v, cols, self.in_features))
        return self._frozen[1:]

    def release_inference_cache(self) -> None:
        """Drop the cached bf16 and packed tiles of gradient-free forwards."""
        self._frozen = None

    def forward(self, x: torch.Tensor) -> torch.Tensor:
        grad = torch.is_grad_enabled() and (x.requires_grad or any(p.requires_grad for p in self.parameters()))
        if grad:
            return kernels.block_ell_matmul(x, self.kernel_values(), self.effective_col_indices(), self.bias)
        # weights fixed across gradient-free forwards: bf16 tiles and their packed copy cached
        v, cols, packed = self._frozen_weight()
        lead = x.shape[:-1]
        x2 = x.reshape(-1, x.shape[-1]).to(torch.bfloat16).contiguous()
        y = kernels.block_ell_matmul_prepacked(x2, packed, v, cols, self.bias)
        return y.reshape(*lead, y.shape[-1])


class MLPBlock(nn.Module):
    """Block-ELL MLP (reference ``mlp.py:98-168``).

    SwiGLU: ``out = w_down(silu(w_gate(x)) * w_up(x))`` as one fused operator.
    GELU:   ``out = fc2(gelu(fc1(x)))`` with two Block-ELL products.
    """

    def __init__(self, d_model: int, d_ff: int, use_swiglu: bool = False, dropout: float = 0.0,
                 tile_size: int = 16, density: float = 1.0, dtype: torch.dtype = torch.bfloat16, device=None,
                 bias: bool = True):
        super().__init__()
        self.d_model, self.d_ff, self.use_swiglu, self.dropout = d_model, d_ff, use_swiglu, dropout
        kw = dict(tile_size=tile_size, density=density, dtype=dtype, device=device)
        if use_swiglu:
            self.w_gate = BlockELLLinear(d_ff, d_model, bias=bias, **kw)
            self.w_up = BlockELLLinear(d_ff, d_model, bias=bias, **kw)
            self.w_down = BlockELLLinear(d_model, d_ff, bias=bias, **kw)
        else:
            self.fc1 = BlockELLLinear(d_ff, d_model, **kw)
            self.fc2 = BlockELLLinear(d_model, d_ff, **kw)
        self._frozen = None

    def swiglu_columns(self):
        """(ci_gate, ci_up, ci_down) in kernel form.

        When gate and up have the same topology (as initialised: both are seeded from the
        same hash, reference ``mlp.py:94``) the same index tensor is passed for both, which
        lets the kernel read each activation tile once for the two products.  The comparison
        runs once per topology version."""
        cg, cu = self.w_gate.effective_col_indices(), self.w_up.effective_col_indices()
        key = (self.w_gate._eff_cache[0], self.w_up._eff_cache[0])   # (pointer, version) of both
        if getattr(self, "_shared_key", None) != key:
            self._shared_key, self._shared = key, bool(torch.equal(cg, cu))
        return cg, (cg if self._shared else cu), self.w_down.effective_col_indices()

    def swiglu_weights(self):
        """(v_gate, ci_gate, v_up, ci_up, v_down, ci_down) in kernel form."""
        cg, cu, cd = self.swiglu_columns()
        return (self.w_gate.kernel_values(), cg, self.w_up.kernel_values(), cu, self.w_down.kernel_values(), cd)

    def _fp32_values(self):
        """Whether the projections' values are fp32 and rounded to bf16 without more ado: no replaced
        ``swiglu_weights`` or ``kernel_values`` to ask for them."""
        return (type(self).swiglu_weights is MLPBlock.swiglu_weights and "swiglu_weights" not in self.__dict__
                and all(lin.values.dtype == torch.float32 and type(lin).kernel_values is BlockELLLinear.kernel_values
                        and "kernel_values" not in lin.__dict__ for lin in (self.w_gate, self.w_up, self.w_down)))

    def _swiglu_grad(self, x2, bg, bu, bd):
        """The differentiable forward: fp32 values go to the kernels as they are, rounded there."""
        if self._fp32_values():
            cg, cu, cd = self.swiglu_columns()
            return kernels.swiglu_train(x2, self.w_gate.values, cg, self.w_up.values, cu, self.w_down.values, cd,
                                        add_residual=False, b_gate=bg, b_up=bu, b_down=bd)
        return kernels.swiglu(x2, *self.swiglu_weights(), add_residual=False, b_gate=bg, b_up=bu, b_down=bd)

    def _frozen_swiglu(self):
        """(kernel-form weights, packed copy), rebuilt when any weight's version changes."""
        key = _versions((self.w_gate, self.w_up, self.w_down))
        if self._frozen is None or self._frozen[0] != key:
            w = self.swiglu_weights()
            self._frozen = (key, w, kernels.swiglu_prepack(*w))
        return self._frozen[1], self._frozen[2]

    def release_inference_cache(self) -> None:
        """Drop the cached bf16 and packed weights of gradient-free forwards."""
        self._frozen = None

    def swiglu_biases(self):
        """(b_gate, b_up, b_down): the projections' biases (None where a projection has none)."""
        return self.w_gate.bias, self.w_up.bias, self.w_down.bias

    def _gelu(self, x):
        """The GELU form as one operator, the activation in the first product's epilogue."""
        fc1, fc2 = self.fc1, self.fc2
        x2 = x.reshape(-1, x.shape[-1]).to(torch.bfloat16).contiguous()
        if torch.is_grad_enabled() and (x.requires_grad or any(p.requires_grad for p in self.parameters())):
            if fc1.values.dtype != torch.float32 or fc2.values.dtype != torch.float32:
                return fc2(F.gelu(fc1(x).float(), approximate="tanh").to(torch.bfloat16))
            out = kernels.gelu_train(x2, fc1.values, fc1.effective_col_indices(), fc2.values,
                                     fc2.effective_col_indices(), fc1.bias, fc2.bias)
        else:
            (v1, c1, p1), (v2, c2, p2) = fc1._frozen_weight(), fc2._frozen_weight()
            out = kernels.gelu_fwd_prepacked(x2, p1, v1, c1, p2, v2, c2, fc1.bias, fc2.bias)
        return out if x.dim() == 2 else out.reshape(*x.shape[:-1], out.shape[-1])

    def forward(self, x: torch.Tensor, deterministic: bool = True) -> torch.Tensor:
        if self.use_swiglu:
            x2 = x.reshape(-1, self.d_model).to(torch.bfloat16).contiguous()
            bg, bu, bd = self.swiglu_biases()
            grad = torch.is_grad_enabled() and (x2.requires_grad or any(p.requires_grad for p in self.parameters()))
            if grad:
                out = self._swiglu_grad(x2, bg, bu, bd)
            else:
                w, packed = self._frozen_swiglu()
                out = kernels.swiglu_fwd_prepacked(x2, packed, *w, add_residual=False, b_gate=bg, b_up=bu, b_down=bd)
            if x.dim() != 2 or x.shape[1] != self.d_model:
                out = out.reshape(*x.shape[:-1], self.d_model)
        elif x.shape[-1] == self.d_model and _plain(self.fc1, BlockELLLinear) and _plain(self.fc2, BlockELLLinear):
            out = self._gelu(x)
        else:                       # the two layers one by one: their hooks and overrides see each
            out = self.fc2(F.gelu(self.fc1(x).float(), approximate="tanh").to(torch.bfloat16))
        if self.dropout > 0.0 and not deterministic:
            out = F.dropout(out, p=self.dropout, training=True)
        return out
