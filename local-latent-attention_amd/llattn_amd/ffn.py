"""The LM's FeedForward ``w2(gelu(w1 x))`` (reference models.py:50-58) on the gfx950 MFMA GEMM under bf16
autocast, with the GELU in the GEMM epilogues:

* forward: one GEMM forms ``h = x W1^T + b1`` and writes ``gelu(h)`` (the input of ``w2``) and ``gelu'(h)``
  (what the backward multiplies by; the epilogue has both from one evaluation of Phi and phi), a second one
  ``y = gelu(h) W2^T + b2``;
* backward: the input gradient of ``w2`` leaves its GEMM already multiplied by ``gelu'(h)``, so no separate
  elementwise pass reads or writes the ``[tokens, d_ff]`` gradients; weight gradients in fp32 with the bias
  gradients from the same passes (or the column-sum kernel where the width does not allow it).

Numerics are those of the reference under bf16 autocast: bf16 operands, fp32 accumulation, ``h`` rounded to
bf16 before the exact (erf) GELU, ``gelu(h)`` rounded to bf16, the GELU backward on the bf16 upstream
gradient, except that ``gelu'(h)`` is kept in bf16 (one rounding more than autocast's backward makes) and
weight gradients are accumulated in fp32 instead of being rounded to bf16.
"""
from __future__ import annotations

import torch

from . import _lib as L
from . import gemm, ops
from .linear import pack_params, weight_grad
from .steps import Ffn, plain_as

BF16 = torch.bfloat16


def _bias(b: torch.Tensor | None) -> torch.Tensor | None:
    if b is None:
        return None
    b = b.detach().float().contiguous()
    return b if b.data_ptr() % 16 == 0 else b.clone()


class _FeedForward(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, w1, b1, w2, b2):
        lead, D = tuple(x.shape[:-1]), x.shape[-1]
        with torch.autocast(device_type="cuda", enabled=False):
            x2 = x.reshape(-1, D).to(BF16)
            if not x2.is_contiguous():
                x2 = x2.contiguous()
            # the autocast casts, one launch; both also transposed for the input gradients, w2 where its input
            # gradient runs on the persistent kernel (below that the copy would cost more than it saves)
            (w1b, w1t), w2p = pack_params([([w1], BF16, True),
                                           ([w2], BF16, gemm.input_grad_persistent(x2.shape[0], *w2.shape))])
            w2b, w2t = w2p if isinstance(w2p, tuple) else (w2p, None)
            g, gp = gemm.linear_gelu(x2, w1b, _bias(b1))
            y = gemm.linear(g, w2b, _bias(b2))
        ctx.save_for_backward(x2, gp, g, w1b, w1t, w2b, w2t)
        ctx.meta = (lead, x.dtype, w1.dtype, w2.dtype, None if b1 is None else b1.dtype,
                    None if b2 is None else b2.dtype)
        return y.view(*lead, w2.shape[0])

    @staticmethod
    def backward(ctx, dy):
        x2, gp, g, w1b, w1t, w2b, w2t = ctx.saved_tensors
        lead, xdt, w1dt, w2dt, b1dt, b2dt = ctx.meta
        has_b1, has_b2 = b1dt is not None, b2dt is not None
        with torch.autocast(device_type="cuda", enabled=False):
            dy2 = dy.reshape(-1, dy.shape[-1]).to(BF16)
            if not dy2.is_contiguous():
                dy2 = dy2.contiguous()
            dh = gemm.matmul_nn_scaled(dy2, w2b, gp, w2t)    # (dy W2) * gelu'(h), bf16
            dw2, db2 = weight_grad(dy2, g, has_b2)           # fp32
            dx = gemm.input_grad(dh, w1b, w_t=w1t) if ctx.needs_input_grad[0] else None
            dw1, db1 = weight_grad(dh, x2, has_b1)
        return (None if dx is None else dx.view(*lead, x2.shape[1]).to(xdt), dw1.to(w1dt),
                None if db1 is None else db1.to(b1dt), dw2.to(w2dt), None if db2 is None else db2.to(b2dt))


def _param(m, name: str):
    """``getattr(m, name)``, without nn.Module's search where the parameter is registered as itself."""
    held = getattr(m, "_parameters", ())
    return held[name] if name in held else getattr(m, name)


def _step_cfg(x: torch.Tensor, ps) -> L.LlattnFfnCfg | None:
    """The native step's configuration for ``x`` and ``(w1, b1, w2, b2)``, or None where it does not take them: it
    sees pointers alone, so every shape is compared here."""
    d = x.shape[-1]
    rows = x.numel() // max(1, d)
    d_ff, d_out = ps[0].shape[0], ps[2].shape[0]
    if not 0 < rows < 1 << 31 or d % 8 or d_ff % 8 or d_out % 8 or x.dtype is not BF16 or not x.is_contiguous() \
            or x.data_ptr() & 15:
        return None
    if not plain_as(ps, ((d_ff, d), (d_ff,), (d_out, d_ff), (d_out,)), x.device):
        return None
    saved = torch.is_grad_enabled() and (x.requires_grad or any(p is not None and p.requires_grad for p in ps))
    return L.LlattnFfnCfg(rows, d, d_ff, d_out, int(saved))


def feed_forward(x: torch.Tensor, w1: torch.nn.Linear, w2: torch.nn.Linear) -> torch.Tensor:
    """bf16 ``w2(gelu(w1(x)))`` on the GEMM kernels (GPU only; widths multiples of 8)."""
    ps = (_param(w1, "weight"), _param(w1, "bias"), _param(w2, "weight"), _param(w2, "bias"))
    cfg = _step_cfg(x, ps) if x.is_cuda and not ops.observed() else None
    return _FeedForward.apply(x, *ps) if cfg is None else Ffn.apply(x, cfg, *ps)
