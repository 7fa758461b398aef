"""Single-token decode step with the reference's signature
(``mamba2/mamba2_kernel_inference.py:107-122``), computed by the gfx950 HIP kernels.

    mamba2_kernel_inference(xBC[b,1,Cx], conv_state[b,Cx,W], conv_weight[Cx,k], conv_bias[Cx],
                            S[b,h,p,n], dt[b,1,h], logA[h], D[h]=None, n_groups=1)
        -> (Y[b,1,h*p], conv_state, S)

Unlike the reference, which writes fresh output tensors, ``conv_state`` and ``S`` are updated IN
PLACE and the same tensors are returned, which is compatible with the caller's re-binding of the
cache entries (``mamba2/mamba2_mixer.py:275-276``).  W may be k-1 or k columns.  The SSM state must
be float32.  ``xBC`` and ``dt`` may be column slices of the packed projection output.  With the keyword
``dt_bias`` (h), ``dt`` is the raw projection output and the kernel applies softplus(dt + dt_bias) itself
(the caller's ``softplus`` pass of ``mamba2_mixer.py:268`` is then not needed).  ``out`` takes a preallocated Y;
``static_scratch=True`` runs the step through ``m2_decode_step_static``, whose scratch lives inside the library (nothing
is allocated for it; batch x channels is limited, and calls that overlap on one GPU must not use it at the same time).
"""
from . import _lib


def mamba2_kernel_inference(xBC_tensor, conv_state_tensor, conv_weight_tensor, conv_bias_tensor, S_tensor, dt_tensor,
                            logA_tensor, D_tensor=None, n_groups=1, activation="silu", dt_bias=None, out=None, static_scratch=False):
    batch_size, n_heads, d_head, d_state = S_tensor.shape
    seq_len = xBC_tensor.shape[1]
    assert seq_len == 1
    d_inner = n_heads * d_head
    d_xBC = xBC_tensor.shape[-1]
    assert d_xBC == d_inner + 2 * n_groups * d_state, f"Expected d_xBC {d_inner + 2 * n_groups * d_state}, got {d_xBC}"
    assert n_heads % n_groups == 0, "Number of heads must be divisible by number of groups"
    assert dt_tensor.shape == (batch_size, 1, n_heads)
    return _lib.native().decode_step(xBC_tensor, conv_state_tensor, conv_weight_tensor, conv_bias_tensor, S_tensor, dt_tensor, logA_tensor,
                                     D_tensor, n_groups, _lib.ACT[activation], dt_bias, out, static_scratch)
