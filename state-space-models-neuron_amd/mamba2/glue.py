"""Elementwise glue of the mixer core: softplus(dt + dt_bias) and the gated, grouped RMSNorm, forward and
backward (``mamba2/fused_kernel.py:33-73,76-175``; torch twins ``mamba2/mamba2_mixer.py:36-38,88-105``).

The ``*_hip`` functions call the HIP kernels (one pass over each tensor, strided rows taken in place) and are what the
fused mixer core uses.  ``rmsnorm_gated_fn`` is the differentiable form, for the norm
modules (``MambaRMSNormGated``, the blocks' ``Mamba2RMSNorm``) and the one-token decode step.  There is no other path:
shapes the kernels do not take (a group wider than 8192 channels, or not a multiple of the 16-byte vector) raise.
"""
import torch

from . import _lib


# --------------------------------------------------------------------------------------------- HIP kernels
def _rows2d(t, name):
    """(rows, channels, row stride) of a (..., channels) tensor whose leading dimensions collapse to one stride."""
    if t.stride(-1) != 1 and t.shape[-1] > 1:
        raise ValueError(f"{name}: innermost dimension must be contiguous")
    ch = t.shape[-1]
    rows = t.numel() // ch if ch else 0
    if t.dim() == 1:
        return 1, ch, ch
    sr = t.stride(-2)
    # the leading dimensions must be walkable with the one row stride (true for contiguous tensors and column slices of them)
    exp = sr
    for k in range(t.dim() - 2, -1, -1):
        if t.shape[k] != 1 and t.stride(k) != exp:
            raise ValueError(f"{name}: rows are not evenly strided (shape {tuple(t.shape)}, strides {t.stride()})")
        exp *= t.shape[k]
    return rows, ch, sr


def softplus_bias_hip(dt, dt_bias):
    """softplus(dt + dt_bias), threshold form; dt (..., h) may be a column slice; result contiguous, dtype of dt."""
    _lib.require_gpu(dt, dt_bias)
    lib = _lib.load()
    rows, h, sr = _rows2d(dt, "dt")
    out = torch.empty(dt.shape, dtype=dt.dtype, device=dt.device)
    bias = dt_bias.detach().float().contiguous()
    rc = lib.m2_softplus_bias_fwd(_lib.ptr(dt), sr, _lib.ptr(bias), _lib.ptr(out), h, rows, h, _lib.dtype_code(dt.dtype),
                                  _lib.stream_ptr(dt.device))
    _lib.check(rc, "m2_softplus_bias_fwd")
    return out


def softplus_bias_bwd_hip(dt, dt_bias, d_out, out_d_in=None):
    """Returns (d_in, d_bias fp32 (h)); d_in is written into ``out_d_in`` (a view with the dtype of dt) when given."""
    _lib.require_gpu(dt, dt_bias, d_out)
    lib = _lib.load()
    rows, h, sr = _rows2d(dt, "dt")
    if d_out.dtype != dt.dtype or d_out.stride(-1) != 1:
        d_out = d_out.to(dt.dtype).contiguous()
    _, _, dosr = _rows2d(d_out, "d_out")
    d_in = out_d_in if out_d_in is not None else torch.empty(dt.shape, dtype=dt.dtype, device=dt.device)
    if d_in.dtype != dt.dtype or d_in.shape != dt.shape:
        raise ValueError("softplus_bias_bwd: out_d_in must have the shape and dtype of dt")
    _, _, disr = _rows2d(d_in, "out_d_in")
    bias = dt_bias.detach().float().contiguous()
    d_bias = torch.empty(h, dtype=torch.float32, device=dt.device)
    nbytes = lib.m2_softplus_bias_bwd_workspace_bytes(rows, h)
    ws = _lib.Workspace.get(nbytes, dt.device)
    rc = lib.m2_softplus_bias_bwd(_lib.ptr(dt), sr, _lib.ptr(bias), _lib.ptr(d_out), dosr, _lib.ptr(d_in), disr, _lib.ptr(d_bias),
                                  _lib.ptr(ws), ws.numel(), rows, h, _lib.dtype_code(dt.dtype), _lib.stream_ptr(dt.device))
    _lib.check(rc, "m2_softplus_bias_bwd")
    return d_in, d_bias


def _weight(w):
    """The norm weight for the native calls: fp32 values kept across calls while autograd is off."""
    return w if w.dtype == torch.float32 or torch.is_grad_enabled() else _lib.f32_param(w)


def rmsnorm_gated_hip(x, z, weight, n_groups, eps, out_dtype=None):
    """out = weight * h * rsqrt(mean_group(h^2) + eps), h = x * silu(z); out in ``out_dtype`` (fp32 or the dtype of x)."""
    return _lib.native().rmsnorm_forward(x, z, _weight(weight), n_groups, eps, torch.float32 if out_dtype is None else out_dtype)


def rmsnorm_gated_bwd_hip(x, z, weight, d_out, n_groups, eps, out_dz=None):
    """Returns (dx, dw fp32, dz); dz is written into ``out_dz`` (a view with the dtype of x) or a fresh tensor."""
    return _lib.native().rmsnorm_backward(x, z, weight, d_out, n_groups, eps, out_dz)


def add_rmsnorm_ok(channels, out_dtype):
    """True if ``add_rmsnorm_`` takes rows of this width: a multiple of 4, at most 8192 channels, fp32 or bf16 output."""
    return channels % 4 == 0 and 0 < channels <= 8192 and out_dtype in (torch.float32, torch.bfloat16)


def add_rmsnorm_(residual, delta, weight, eps, out_dtype):
    """``residual += delta`` in place (fp32), then RMSNorm of the sum, in one kernel (inference; the block boundary of the
    token-by-token loop, ``modeling_mamba2.py:133-140`` + ``:94-103``).  ``delta`` (dtype ``out_dtype``) may be None.
    Returns weight * residual * rsqrt(mean(residual^2) + eps) in ``out_dtype``."""
    return _lib.native().add_rmsnorm(residual, delta, _lib.f32_param(weight), eps, out_dtype)


# --------------------------------------------------------------------------------------------- autograd form
def norm_kernel_ok(x, n_groups):
    """True if the HIP norm kernels take this shape: group width a multiple of the vector width and within a row's registers."""
    if x.dtype not in (torch.float32, torch.bfloat16) or n_groups < 1 or x.shape[-1] % n_groups:
        return False
    gw = x.shape[-1] // n_groups
    vec = 8 if x.dtype == torch.bfloat16 else 4
    return gw % vec == 0 and 0 < gw <= 8192


def rmsnorm_gated_fn(x, z, weight, n_groups, eps, out_dtype=None):
    """Differentiable gated grouped RMSNorm; output fp32 unless ``out_dtype`` says the dtype of x.
    Raises ValueError for shapes outside the kernels' limits."""
    _lib.require_gpu(x, z, weight)
    if not norm_kernel_ok(x, n_groups):
        raise ValueError(f"rmsnorm_gated: {x.shape[-1]} channels in {n_groups} groups, dtype {x.dtype}: a group must be a "
                         "multiple of 16 bytes and at most 8192 channels wide, in float32 or bfloat16")
    if z is not None and z.dtype != x.dtype:
        raise ValueError("rmsnorm_gated: z must have the dtype of x")
    return _lib.native().rmsnorm(x, z, _weight(weight), n_groups, eps, torch.float32 if out_dtype is None else out_dtype)
