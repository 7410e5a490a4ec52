"""The block, its core and the feed-forward as one native call per direction (``include/llattn_steps.h``).

Each autograd function here is the whole of a step that :mod:`llattn_amd.module`, :mod:`llattn_amd.ops` and
:mod:`llattn_amd.ffn` otherwise issue product by product from Python: the same products with what the backward
reads in one buffer (two independent ones may share a launch).  The calls that take this path have parameters of the
layout's shapes in fp32, whole, 16-byte aligned and on the activations' device, activations in the compute dtype,
and nobody looking at the single calls (:func:`llattn_amd.ops.observed`).  The others, and profiling, stay on the
Python path.  Forward-only calls are applied as functions too: a tangent, a batched tensor or a tracer is then met as by any other autograd function.
"""
from __future__ import annotations

import ctypes

import torch

from . import _lib as L

_ref = ctypes.byref
_F32, _BF16 = torch.float32, torch.bfloat16


def plain(t: torch.Tensor, device, dtype=_F32) -> bool:
    """A dense tensor of ``dtype`` on ``device`` whose data a kernel can read in 16-byte pieces."""
    return t.dtype is dtype and t.device == device and t.is_contiguous() and not t.data_ptr() & 15


def plain_as(params, shapes, device) -> bool:
    """Whether every parameter that is there is :func:`plain` fp32 of its shape (a native step sees its pointer alone)."""
    index = device.index if device.type == "cuda" else -1
    for p, s in zip(params, shapes):
        if p is not None and (p.dtype is not _F32 or p.shape != s or p.get_device() != index or not p.is_contiguous()
                              or p.data_ptr() & 15):
            return False
    return True


def _bytes(n: int, device):
    return torch.empty((n,), dtype=torch.uint8, device=device) if n else None


def _ptr(t):
    return None if t is None else t.data_ptr()


def _call(name, *args):
    L.check(getattr(L.load(), name)(*args), name)


def _size(name, cfg, which: int) -> int:
    return getattr(L.load(), name)(_ref(cfg), which)


def _forward_sizes(name, ref):
    """Bytes that a forward keeps and its scratch."""
    fn = getattr(L.load(), name)
    kept = fn(ref, 0)
    if kept == 0:
        L.check(L.ERR_SHAPE, name)
    return kept, fn(ref, 1)


def _dense(t: torch.Tensor, dtype) -> torch.Tensor:
    t = t.to(dtype).contiguous()
    return t.clone() if t.data_ptr() & 15 else t


# ---------------------------------------------------------------------------
# block
# ---------------------------------------------------------------------------

def block_forward(x, cfg, params):
    """``(out, kept)`` of the block on ``x [B, T, D]``; ``params``: the twelve parameters of ``L.BLOCK_PARAMS``
    (biases None without)."""
    dev, ref = x.device, _ref(cfg)
    k, n = _forward_sizes("llattn_block_bytes", ref)
    if cfg.saved:
        kept, ws = _bytes(k, dev), _bytes(n, dev)
        at = _ptr(ws)
    else:  # nothing outlives the call: one buffer
        k = (k + 255) & ~255
        kept = _bytes(k + n, dev)
        at = kept.data_ptr() + k if n else None
    out = torch.empty_like(x)
    ptrs = L.LlattnBlockParams(*[None if p is None else p.data_ptr() for p in params])
    _call("llattn_block_fwd", ref, _ref(ptrs), x.data_ptr(), kept.data_ptr(), at, n, out.data_ptr(), L.stream_ptr(dev))
    return out, kept


# what the backward reads of the parameters themselves: the gates; in fp32 also the weights that are not copied
_BWD_BF16 = (10, 11)
_BWD_F32 = (4, 6, 8, 10, 11)
_BWD_F32_MACRO = (0, 2, 4, 6, 8, 10, 11)


class Block(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, cfg, *params):
        if not cfg.saved:
            return block_forward(x, cfg, params)[0]
        params = [None if p is None else p.detach() for p in params]
        out, kept = block_forward(x.detach(), cfg, params)
        which = _BWD_BF16 if cfg.shape.dtype == L.BF16 else _BWD_F32_MACRO if cfg.macro else _BWD_F32
        ctx.save_for_backward(x, kept, *[params[i] for i in which])
        ctx.which, ctx.cfg = which, cfg
        ctx.shapes = [None if p is None else tuple(p.shape) for p in params]
        return out

    @staticmethod
    def backward(ctx, dy):
        x, kept, *held = ctx.saved_tensors
        cfg, dev = ctx.cfg, x.device
        dy = _dense(dy, x.dtype)
        p = L.LlattnBlockParams()
        for i, t in zip(ctx.which, held):
            setattr(p, L.BLOCK_PARAMS[i], t.data_ptr())
        new = lambda shape: torch.empty(shape, dtype=_F32, device=dev)  # noqa: E731
        dx = torch.empty_like(x) if ctx.needs_input_grad[0] else None
        shapes = ctx.shapes
        if cfg.macro:
            grads = [None if s is None else new(s) for s in shapes]
            ptrs = [_ptr(g) for g in grads]
        else:  # q|k|v and the token-wise latent queries: one weight gradient, one bias gradient
            n, m = shapes[0][0], shapes[2][0]
            w = new((n + m, shapes[0][1]))
            b = None if shapes[1] is None else new((n + m,))
            grads = [w[:n], None if b is None else b[:n], w[n:], None if b is None else b[n:]]
            grads += [None if s is None else new(s) for s in shapes[4:]]
            ptrs = [w.data_ptr(), _ptr(b), None, None] + [_ptr(g) for g in grads[4:]]
        n = _size("llattn_block_bytes", cfg, 3 if dx is None else 2)
        ws = _bytes(n, dev)
        _call("llattn_block_bwd", _ref(cfg), _ref(p), x.data_ptr(), kept.data_ptr(), dy.data_ptr(), _ptr(dx),
              _ref(L.LlattnBlockParams(*ptrs)), _ptr(ws), n, L.stream_ptr(dev))
        return (dx, None, *grads)


# ---------------------------------------------------------------------------
# core on head tensors
# ---------------------------------------------------------------------------

def core_forward(cfg, views, gl, gr, r_w, r_b, y_view, device):
    """Runs the core into ``y_view``; returns what its backward reads."""
    ref = _ref(cfg)
    k, n = _forward_sizes("llattn_core_bytes", ref)
    kept, ws = _bytes(k, device), _bytes(n, device)
    _call("llattn_core_fwd", ref, _ref(views), gl.data_ptr(), gr.data_ptr(), r_w.data_ptr(), _ptr(r_b),
          kept.data_ptr(), _ptr(ws), n, _ref(y_view), L.stream_ptr(device))
    return kept


def core_backward(cfg, views, gl, gr, r_w, has_rb, kept, dy_view, grad_views, device):
    """Writes the gradients of the head tensors; returns (dgate_l, dgate_r, dr_w, dr_b), gates per head or shared."""
    H, Dh = cfg.shape.H, cfg.shape.Dh
    gshape = (H, Dh) if cfg.shape.gate_per_head else (Dh,)
    dgl, dgr = (torch.empty(gshape, dtype=_F32, device=device) for _ in range(2))
    dr_w = torch.empty(tuple(r_w.shape), dtype=_F32, device=device)
    dr_b = torch.empty((H * Dh,), dtype=_F32, device=device) if has_rb else None
    n = _size("llattn_core_bytes", cfg, 2)
    ws = _bytes(n, device)
    _call("llattn_core_bwd", _ref(cfg), _ref(views), gl.data_ptr(), gr.data_ptr(), r_w.data_ptr(), kept.data_ptr(),
          _ref(dy_view), _ref(grad_views), dgl.data_ptr(), dgr.data_ptr(), dr_w.data_ptr(), _ptr(dr_b), _ptr(ws), n,
          L.stream_ptr(device))
    return dgl, dgr, dr_w, dr_b


# ---------------------------------------------------------------------------
# feed-forward
# ---------------------------------------------------------------------------

def ffn_forward(x, cfg, w1, b1, w2, b2):
    dev, ref = x.device, _ref(cfg)
    k, n = _forward_sizes("llattn_ffn_bytes", ref)
    kept, ws = _bytes(k, dev), _bytes(n, dev)
    y = torch.empty((*x.shape[:-1], cfg.d_out), dtype=_BF16, device=dev)
    _call("llattn_ffn_fwd", ref, x.data_ptr(), w1.data_ptr(), _ptr(b1), w2.data_ptr(), _ptr(b2), kept.data_ptr(),
          _ptr(ws), n, y.data_ptr(), L.stream_ptr(dev))
    return y, kept


class Ffn(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, cfg, w1, b1, w2, b2):
        if not cfg.saved:
            return ffn_forward(x, cfg, w1, b1, w2, b2)[0]
        y, kept = ffn_forward(x.detach(), cfg, w1, b1, w2, b2)
        ctx.save_for_backward(x, kept)
        ctx.cfg, ctx.bias = cfg, (b1 is not None, b2 is not None)
        return y

    @staticmethod
    def backward(ctx, dy):
        x, kept = ctx.saved_tensors
        cfg, dev = ctx.cfg, x.device
        dy = _dense(dy, _BF16)
        new = lambda *shape: torch.empty(shape, dtype=_F32, device=dev)  # noqa: E731
        dx = torch.empty_like(x) if ctx.needs_input_grad[0] else None
        dw1, dw2 = new(cfg.d_ff, cfg.d), new(cfg.d_out, cfg.d_ff)
        db1, db2 = (new(n) if has else None for has, n in zip(ctx.bias, (cfg.d_ff, cfg.d_out)))
        n = _size("llattn_ffn_bytes", cfg, 3 if dx is None else 2)
        ws = _bytes(n, dev)
        _call("llattn_ffn_bwd", _ref(cfg), x.data_ptr(), kept.data_ptr(), dy.data_ptr(), _ptr(dx), dw1.data_ptr(),
              _ptr(db1), dw2.data_ptr(), _ptr(db2), _ptr(ws), n, L.stream_ptr(dev))
        return dx, None, dw1, db1, dw2, db2
