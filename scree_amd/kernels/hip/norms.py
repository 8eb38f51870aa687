"""Varlen RMSNorm / LayerNorm on the HIP kernels: tensor-level launchers.

* :func:`varlen_rmsnorm_hip` <- ``varlen_rmsnorm_triton``
  (``src/scree/kernels/triton/varlen_rmsnorm.py:49-99``)
* :func:`varlen_layernorm_hip` <- ``varlen_layernorm_triton``
  (``src/scree/kernels/triton/varlen_layernorm.py:52-109``)
* :func:`varlen_add_rmsnorm_hip` -- fused residual add + RMSNorm (no
  counterpart in the reference; its block adds then normalises,
  ``examples/03_train_step.py:46-48``)

As in the reference, ``x`` of any rank is normalised over its last axis,
``weight`` / ``bias`` are rounded to ``x``'s dtype before the multiply
(``varlen_rmsnorm.py:79``, ``varlen_layernorm.py:84,89``) and the statistics
are computed in fp32.  Unlike the reference, these launchers are
autograd-aware: when ``x``, ``weight`` or ``bias`` requires grad the call
records a ``torch.autograd.Function`` whose backward runs the HIP backward
kernels (the reference has no norm backward).  The explicit backward
launchers are :func:`varlen_rmsnorm_hip_backward` and
:func:`varlen_layernorm_hip_backward`.
"""

from __future__ import annotations

import functools

import torch

from . import _ffi

_CODE_DTYPES = {code: dtype for dtype, code in _ffi._DTYPE_CODES.items()}


def _flat(x):
    assert x.is_cuda, "varlen norms on HIP require ROCm device tensors"
    d = x.shape[-1]
    if x.dim() == 2 and x.is_contiguous():
        return x, d
    return x.reshape(-1, d).contiguous(), d


def _like(y2, shape):
    return y2 if y2.shape == shape else y2.reshape(shape)


def _param(p, d, device, dtype, name):
    if p is None:
        return None
    assert p.shape == (d,), f"{name} must have shape ({d},)"
    assert p.device == device, f"{name} must be on {device}"
    return p.to(dtype).contiguous()


def _dparam_code(p):
    return _ffi._DTYPE_CODES.get(p.dtype, _ffi.DTYPE_F32)


def rmsnorm_fwd(x2, w, eps, want_stats):
    rows, d = x2.shape
    y = torch.empty_like(x2)
    rstd = torch.empty(rows, dtype=torch.float32, device=x2.device) if want_stats else None
    _ffi.launch(_ffi.lib().scree_rmsnorm_fwd, x2, x2.data_ptr(), _ffi.ptr(w), y.data_ptr(),
                _ffi.ptr(rstd), rows, d, float(eps), _ffi.dtype_code(x2.dtype))
    return y, rstd


def layernorm_fwd(x2, w, b, eps, want_stats):
    rows, d = x2.shape
    y = torch.empty_like(x2)
    mean = rstd = None
    if want_stats:
        mean = torch.empty(rows, dtype=torch.float32, device=x2.device)
        rstd = torch.empty_like(mean)
    _ffi.launch(_ffi.lib().scree_layernorm_fwd, x2, x2.data_ptr(), _ffi.ptr(w), _ffi.ptr(b),
                y.data_ptr(), _ffi.ptr(mean), _ffi.ptr(rstd), rows, d, float(eps),
                _ffi.dtype_code(x2.dtype))
    return y, mean, rstd


@functools.lru_cache(maxsize=256)
def _workspace_bytes(rows, d):
    return max(int(_ffi.lib().scree_norm_bwd_workspace_bytes(rows, d)), 16)


def _workspace(rows, d, device):
    """Room for the partial parameter gradients (only a call that wants them needs it)."""
    return torch.empty(_workspace_bytes(rows, d), dtype=torch.uint8, device=device)


def rmsnorm_bwd(dy2, x2, w, rstd, want_dw, dw_like=None):
    rows, d = x2.shape
    dx = torch.empty_like(x2)
    dw, code, ws, nws = None, _ffi.DTYPE_F32, None, 0
    if want_dw:
        code = _dparam_code(dw_like) if dw_like is not None else _ffi.DTYPE_F32
        dw = torch.empty(d, dtype=_CODE_DTYPES[code], device=x2.device)
        ws = _workspace(rows, d, x2.device)
        nws = ws.numel()
    _ffi.launch(_ffi.lib().scree_rmsnorm_bwd, x2, dy2.data_ptr(), x2.data_ptr(), _ffi.ptr(w),
                rstd.data_ptr(), dx.data_ptr(), _ffi.ptr(dw), code, rows, d,
                _ffi.dtype_code(x2.dtype), _ffi.ptr(ws), nws)
    return dx, dw


def layernorm_bwd(dy2, x2, w, mean, rstd, want_dw, want_db, p_like=None):
    rows, d = x2.shape
    dx = torch.empty_like(x2)
    code = _dparam_code(p_like) if p_like is not None else _ffi.DTYPE_F32
    dw = db = ws = None
    nws = 0
    if want_dw:
        dw = torch.empty(d, dtype=_CODE_DTYPES[code], device=x2.device)
    if want_db:
        db = torch.empty(d, dtype=_CODE_DTYPES[code], device=x2.device)
    if want_dw or want_db:
        ws = _workspace(rows, d, x2.device)
        nws = ws.numel()
    _ffi.launch(_ffi.lib().scree_layernorm_bwd, x2, dy2.data_ptr(), x2.data_ptr(), _ffi.ptr(w),
                mean.data_ptr(), rstd.data_ptr(), dx.data_ptr(), _ffi.ptr(dw), _ffi.ptr(db), code,
                rows, d, _ffi.dtype_code(x2.dtype), _ffi.ptr(ws), nws)
    return dx, dw, db


def add_rmsnorm_fwd(x2, r2, w, eps, want_stats):
    rows, d = x2.shape
    h = torch.empty_like(x2)
    y = torch.empty_like(x2)
    rstd = torch.empty(rows, dtype=torch.float32, device=x2.device) if want_stats else None
    _ffi.launch(_ffi.lib().scree_add_rmsnorm_fwd, x2, x2.data_ptr(), r2.data_ptr(), _ffi.ptr(w),
                h.data_ptr(), y.data_ptr(), _ffi.ptr(rstd), rows, d, float(eps),
                _ffi.dtype_code(x2.dtype))
    return h, y, rstd


def add_rmsnorm_bwd(dy2, dh2, h2, w, rstd, want_dw, dw_like=None):
    rows, d = h2.shape
    dx = torch.empty_like(h2)
    dw, code, ws, nws = None, _ffi.DTYPE_F32, None, 0
    if want_dw:
        code = _dparam_code(dw_like) if dw_like is not None else _ffi.DTYPE_F32
        dw = torch.empty(d, dtype=_CODE_DTYPES[code], device=h2.device)
        ws = _workspace(rows, d, h2.device)
        nws = ws.numel()
    _ffi.launch(_ffi.lib().scree_add_rmsnorm_bwd, h2, dy2.data_ptr(), _ffi.ptr(dh2), h2.data_ptr(),
                _ffi.ptr(w), rstd.data_ptr(), dx.data_ptr(), _ffi.ptr(dw), code, rows, d,
                _ffi.dtype_code(h2.dtype), _ffi.ptr(ws), nws)
    return dx, dw


class _RMSNormFn(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, weight, eps):
        x2, d = _flat(x)
        w = _param(weight, d, x.device, x.dtype, "weight")
        y, rstd = rmsnorm_fwd(x2, w, eps, want_stats=True)
        ctx.save_for_backward(x2, w, rstd, weight)
        ctx.shape = x.shape
        return _like(y, x.shape)

    @staticmethod
    def backward(ctx, dy):
        x2, w, rstd, weight = ctx.saved_tensors
        dy2 = _like(dy, x2.shape).contiguous()
        want_dw = weight is not None and ctx.needs_input_grad[1]
        dx, dw = rmsnorm_bwd(dy2, x2, w, rstd, want_dw, dw_like=weight)
        if dw is not None and dw.dtype != weight.dtype:
            dw = dw.to(weight.dtype)
        return _like(dx, ctx.shape), dw, None


class _LayerNormFn(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, weight, bias, eps):
        x2, d = _flat(x)
        w = _param(weight, d, x.device, x.dtype, "weight")
        b = _param(bias, d, x.device, x.dtype, "bias")
        y, mean, rstd = layernorm_fwd(x2, w, b, eps, want_stats=True)
        ctx.save_for_backward(x2, w, mean, rstd, weight, bias)
        ctx.shape = x.shape
        return _like(y, x.shape)

    @staticmethod
    def backward(ctx, dy):
        x2, w, mean, rstd, weight, bias = ctx.saved_tensors
        dy2 = _like(dy, x2.shape).contiguous()
        want_dw = weight is not None and ctx.needs_input_grad[1]
        want_db = bias is not None and ctx.needs_input_grad[2]
        like = weight if weight is not None else bias
        dx, dw, db = layernorm_bwd(dy2, x2, w, mean, rstd, want_dw, want_db, p_like=like)
        if dw is not None and dw.dtype != weight.dtype:
            dw = dw.to(weight.dtype)
        if db is not None and db.dtype != bias.dtype:
            db = db.to(bias.dtype)
        return _like(dx, ctx.shape), dw, db, None


class _AddRMSNormFn(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, residual, weight, eps):
        x2, d = _flat(x)
        r2, _ = _flat(residual)
        w = _param(weight, d, x.device, x.dtype, "weight")
        h, y, rstd = add_rmsnorm_fwd(x2, r2, w, eps, want_stats=True)
        ctx.save_for_backward(h, w, rstd, weight)
        ctx.shape = x.shape
        return _like(h, x.shape), _like(y, x.shape)

    @staticmethod
    def backward(ctx, dh, dy):
        h2, w, rstd, weight = ctx.saved_tensors
        want_dw = weight is not None and ctx.needs_input_grad[2]
        dy2 = (torch.zeros_like(h2) if dy is None else _like(dy, h2.shape).contiguous())
        dh2 = None if dh is None else _like(dh, h2.shape).contiguous()
        dx, dw = add_rmsnorm_bwd(dy2, dh2, h2, w, rstd, want_dw, dw_like=weight)
        if dw is not None and dw.dtype != weight.dtype:
            dw = dw.to(weight.dtype)
        dx = _like(dx, ctx.shape)
        # x and residual receive the same gradient (as torch's own add backward does)
        return dx, dx, dw, None


def _needs_grad(*ts):
    return torch.is_grad_enabled() and any(t is not None and t.requires_grad for t in ts)


def varlen_rmsnorm_hip(x, weight=None, eps: float = 1e-6):
    """RMSNorm over the last axis; same shape and dtype as ``x``."""
    if _needs_grad(x, weight):
        return _RMSNormFn.apply(x, weight, eps)
    x2, d = _flat(x)
    w = _param(weight, d, x.device, x.dtype, "weight")
    y, _ = rmsnorm_fwd(x2, w, eps, want_stats=False)
    return _like(y, x.shape)


def varlen_layernorm_hip(x, weight=None, bias=None, eps: float = 1e-5):
    """LayerNorm (population variance) over the last axis; same shape and dtype as ``x``."""
    if _needs_grad(x, weight, bias):
        return _LayerNormFn.apply(x, weight, bias, eps)
    x2, d = _flat(x)
    w = _param(weight, d, x.device, x.dtype, "weight")
    b = _param(bias, d, x.device, x.dtype, "bias")
    y, _, _ = layernorm_fwd(x2, w, b, eps, want_stats=False)
    return _like(y, x.shape)


def varlen_add_rmsnorm_hip(x, residual, weight=None, eps: float = 1e-6):
    """Fused residual add + RMSNorm: returns ``(h, y)`` with ``h = x + residual``
    (rounded to ``x``'s dtype exactly as ``x + residual`` is) and
    ``y = varlen_rmsnorm_hip(h, weight, eps)``, in one pass over HBM.

    The pre-norm transformer step of the reference's block
    (``examples/03_train_step.py:46-48``); autograd-aware like the other
    launchers (``x`` and ``residual`` receive the same gradient).
    """
    assert residual.shape == x.shape, "residual must have x's shape"
    assert residual.dtype == x.dtype and residual.device == x.device, (
        "residual must share x's dtype and device")
    if _needs_grad(x, residual, weight):
        return _AddRMSNormFn.apply(x, residual, weight, eps)
    x2, d = _flat(x)
    r2, _ = _flat(residual)
    w = _param(weight, d, x.device, x.dtype, "weight")
    h, y, _ = add_rmsnorm_fwd(x2, r2, w, eps, want_stats=False)
    return _like(h, x.shape), _like(y, x.shape)


def varlen_add_rmsnorm_hip_backward(dy, dh, h, weight=None, eps: float = 1e-6, rstd=None):
    """``(dx, dweight)`` of the fused add + RMSNorm: ``dx = dh + dRMSNorm(h)``
    (``dh`` may be None); ``rstd`` from the forward is recomputed when absent."""
    h2, d = _flat(h)
    w = _param(weight, d, h.device, h.dtype, "weight")
    if rstd is None:
        _, rstd = rmsnorm_fwd(h2, w, eps, want_stats=True)
    dh2 = None if dh is None else _like(dh, h2.shape).contiguous()
    dx, dw = add_rmsnorm_bwd(_like(dy, h2.shape).contiguous(), dh2, h2, w,
                             rstd.reshape(-1).contiguous(), weight is not None, dw_like=weight)
    return _like(dx, h.shape), dw


def varlen_rmsnorm_hip_autograd(x, weight=None, eps: float = 1e-6):
    """Always records the autograd node (for callers that set requires_grad later)."""
    return _RMSNormFn.apply(x, weight, eps)


def varlen_layernorm_hip_autograd(x, weight=None, bias=None, eps: float = 1e-5):
    return _LayerNormFn.apply(x, weight, bias, eps)


def varlen_rmsnorm_hip_backward(dy, x, weight=None, eps: float = 1e-6, rstd=None):
    """``(dx, dweight)`` of RMSNorm; ``rstd`` from the forward is recomputed when absent."""
    x2, d = _flat(x)
    w = _param(weight, d, x.device, x.dtype, "weight")
    if rstd is None:
        _, rstd = rmsnorm_fwd(x2, w, eps, want_stats=True)
    dx, dw = rmsnorm_bwd(_like(dy, x2.shape).contiguous(), x2, w, rstd.reshape(-1).contiguous(),
                         weight is not None, dw_like=weight)
    return _like(dx, x.shape), dw


def varlen_layernorm_hip_backward(dy, x, weight=None, bias=None, eps: float = 1e-5, mean=None,
                                  rstd=None):
    """``(dx, dweight, dbias)`` of LayerNorm; statistics recomputed when absent."""
    x2, d = _flat(x)
    w = _param(weight, d, x.device, x.dtype, "weight")
    if mean is None or rstd is None:
        _, mean, rstd = layernorm_fwd(x2, w, None, eps, want_stats=True)
    like = weight if weight is not None else bias
    dx, dw, db = layernorm_bwd(_like(dy, x2.shape).contiguous(), x2, w,
                               mean.reshape(-1).contiguous(), rstd.reshape(-1).contiguous(),
                               weight is not None, bias is not None, p_like=like)
    return _like(dx, x.shape), dw, db
