"""SSD chunked scan: ``Mamba2Kernel`` / ``mamba2_kernel`` with the reference's call signature
(``mamba2/mamba2_kernel.py:488-519``), computed by the gfx950 HIP kernels.

    mamba2_kernel(dt[b,l,h], A[h], X[b,l,h,p], B[b,l,g,n], C[b,l,g,n], D[h]) -> Y[b,l,h,p]

Extensions (keyword-only, default off): ``initial_state`` (b,h,p,n) fp32 and
``return_final_state`` -> (Y, S[b,h,p,n] fp32).  X, B, C may be strided views into a packed
[x | B | C] buffer as long as their innermost dimension is contiguous.
"""
import os

import torch

from . import _lib
from ._lib import SsdParams, ptr


def _strides3(t):
    return t.stride(0), t.stride(1), t.stride(2)


def _fill_common(p, dt, A, X, B, C, D, dt_bias=None):
    b, l, h, hd = X.shape
    p.dt_bias = ptr(dt_bias)
    g, n = B.shape[2], B.shape[3]
    p.x, p.dt, p.A, p.B, p.C, p.D = ptr(X), ptr(dt), ptr(A), ptr(B), ptr(C), ptr(D)
    p.batch, p.seqlen, p.nheads, p.headdim, p.dstate, p.ngroups = b, l, h, hd, n, g
    p.x_stride_b, p.x_stride_l, p.x_stride_h = _strides3(X)
    p.dt_stride_b, p.dt_stride_l = dt.stride(0), dt.stride(1)
    p.B_stride_b, p.B_stride_l, p.B_stride_g = _strides3(B)
    p.C_stride_b, p.C_stride_l, p.C_stride_g = _strides3(C)
    p.dtype = _lib.dtype_code(X.dtype)
    p.dt_dtype = _lib.dtype_code(dt.dtype)


def alloc_chunk_states(dt, A, X, B, C):
    """Carry-over buffer from ``ssd_forward(..., chunk_states=buf)`` to ``ssd_backward(..., chunk_states=buf)``
    (opaque bytes): the SSM state entering each 128-token chunk -- the first b*ceil(l/128)*h*p*n elements, in
    X's dtype -- followed by the decay tables and the per-chunk operand tiles."""
    return _lib.native().alloc_chunk_states(dt, A, X, B, C)


def ssd_forward(dt, A, X, B, C, D=None, initial_state=None, want_final_state=False, chunk_states=None, dt_bias=None):
    """Raw forward through the C ABI.  Returns (Y, final_state or None).
    With ``dt_bias`` (h), ``dt`` is the raw projection output and the step size is softplus(dt + dt_bias), applied inside."""
    return _lib.native().ssd_forward(dt, A, X, B, C, D, initial_state, want_final_state, chunk_states, dt_bias)


def ssd_backward(dt, A, X, B, C, D, dY, initial_state=None, d_final_state=None, want_dinitial=False,
                 out_dX=None, out_dB=None, out_dC=None, chunk_states=None, dt_bias=None, out_ddt=None):
    """Raw backward through the C ABI.
    Returns (ddt, dA fp32 (h), dX, dB, dC, dD fp32 (h) or None, d_initial_state or None), and as an eighth element
    d_dt_bias fp32 (h) when ``dt_bias`` is given (``dt`` is then the raw projection output and ddt its gradient).
    ``out_dX/out_dB/out_dC/out_ddt`` let the caller provide (strided) destinations, e.g. views of a packed
    [dx | dB | dC] buffer.  ``chunk_states``: what the forward wrote for the same inputs (skips the recompute)."""
    return _lib.native().ssd_backward(dt, A, X, B, C, D, dY, initial_state, d_final_state, want_dinitial, out_dX, out_dB, out_dC,
                                      chunk_states, dt_bias, out_ddt)


# The reference saves only the inputs and recomputes the chunk states in the backward
# (``mamba2/mamba2_kernel.py:492,363-367``) because its device memory is scarce.  With 288 GB of HBM the
# states entering each chunk (as many bytes as X) are kept instead, which removes two kernels and
# ~0.5 GB of traffic from the backward at the 2.7B shape.  M2_SSD_SAVE_STATES=0 restores recompute.
SAVE_CHUNK_STATES = os.environ.get("M2_SSD_SAVE_STATES", "1") != "0"


class Mamba2Kernel(torch.autograd.Function):
    """apply(dt, A, X, B, C, D) -> Y; backward -> (ddt, dA, dX, dB, dC, dD)
    (``mamba2/mamba2_kernel.py:490,498,515``).  Two optional trailing arguments carry the
    extensions: ``initial_state`` and ``return_final_state``.  The node itself is C++ (csrc/binding.cpp)."""

    @staticmethod
    def apply(dt, A, X, B, C, D, initial_state=None, return_final_state=False):
        return _lib.native().mamba2_kernel(dt, A, X, B, C, D, initial_state, return_final_state, SAVE_CHUNK_STATES)


def mamba2_kernel(dt, A, X, B, C, D, *, initial_state=None, return_final_state=False):
    return _lib.native().mamba2_kernel(dt, A, X, B, C, D, initial_state, return_final_state, SAVE_CHUNK_STATES)
