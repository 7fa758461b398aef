"""Mixer core ``zxBCdt -> norm_out`` with the reference's signatures (``mamba2/fused_kernel.py:423-487``):

    mamba2_fused_kernel(zxBCdt, logA, D, conv1d_weight, conv1d_bias, dt_bias, norm_weight,
                        n_groups, ssm_state_size, intermediate_size, head_dim) -> norm_out[b,l,d_inner]

Pipeline (``fused_kernel.py:252-282``): split [z | xBC | dt] -> depthwise conv + SiLU ->
softplus(dt + dt_bias) -> SSD scan -> gated RMSNorm per group (eps 1e-5).  Here that is three kernel
stages: conv, scan (softplus applied where the scan builds its decay tables, its gradient and d_dt_bias
formed where the scan writes ddt), norm.

Every stage is a HIP kernel.  The split is never materialised: the kernels take strided views of ``zxBCdt`` (the conv reads
the xBC columns in place; the scan reads x, B, C as views of the conv output), and in the backward
the scan writes dx, dB, dC straight into one packed buffer and the conv writes its dx straight into
the xBC columns of ``d_zxBCdt``.  ``Mamba2FusedKernel`` saves only its inputs and recomputes conv,
softplus and scan in the backward (as the reference does, ``:352-367``); ``...WithCaching`` keeps the
intermediates (``:449-471``).

``mamba2_fused_prefill`` is the inference form of the same pipeline that also hands the sequence over to the
decode step: it leaves the SSM state after the last token and the last W conv inputs in the caller's cache
tensors, and continues from them when the cache already holds a prefix.  The reference has no such path
(``mamba2_mixer.py:220``: "cache not supported yet"); the layouts are those its ``step`` reads (``:270-276``).
"""
import torch

from . import _lib


def _forward_parts(zxBCdt, logA, D, conv_w, conv_b, dt_bias, norm_w, n_groups, d_state, d_inner, d_head, keep_states=False):
    """(norm_out, conv_out, scan_out, chunk states or None) of the core, outside autograd."""
    return _lib.native().forward_parts(zxBCdt, logA, D, conv_w, conv_b, dt_bias, norm_w, n_groups, d_state, d_inner, d_head, keep_states)


def _backward_parts(d_output, zxBCdt, logA, D, conv_w, conv_b, dt_bias, norm_w, conv_out, scan_out, states,
                    n_groups, d_state, d_inner, d_head):
    """The seven gradients of the core from what ``_forward_parts`` returned, outside autograd."""
    return _lib.native().backward_parts(d_output, zxBCdt, logA, D, conv_w, conv_b, dt_bias, norm_w, conv_out, scan_out, states,
                                        n_groups, d_state, d_inner, d_head)


class Mamba2FusedKernel(torch.autograd.Function):
    """Saves only the inputs; conv, softplus and scan are recomputed in the backward.  The node itself is C++ (csrc/binding.cpp)."""

    @staticmethod
    def apply(zxBCdt, logA, D, conv1d_weight, conv1d_bias, dt_bias, norm_weight, n_groups, ssm_state_size, intermediate_size, head_dim):
        return _lib.native().fused_core(zxBCdt, logA, D, conv1d_weight, conv1d_bias, dt_bias, norm_weight, n_groups, ssm_state_size,
                                        intermediate_size, head_dim, False)


class Mamba2FusedKernelWithCaching(torch.autograd.Function):
    """Keeps the conv output, the scan output and the chunk states for the backward."""

    @staticmethod
    def apply(zxBCdt, logA, D, conv1d_weight, conv1d_bias, dt_bias, norm_weight, n_groups, ssm_state_size, intermediate_size, head_dim):
        return _lib.native().fused_core(zxBCdt, logA, D, conv1d_weight, conv1d_bias, dt_bias, norm_weight, n_groups, ssm_state_size,
                                        intermediate_size, head_dim, True)


def mamba2_fused_kernel(zxBCdt, logA, D, conv1d_weight, conv1d_bias, dt_bias,
                        norm_weight, n_groups, ssm_state_size, intermediate_size,
                        head_dim):
    return Mamba2FusedKernel.apply(zxBCdt, logA, D, conv1d_weight, conv1d_bias, dt_bias,
                                   norm_weight, n_groups, ssm_state_size, intermediate_size,
                                   head_dim)


def mamba2_fused_kernel_with_caching(zxBCdt, logA, D, conv1d_weight, conv1d_bias, dt_bias,
                                     norm_weight, n_groups, ssm_state_size, intermediate_size,
                                     head_dim):
    return Mamba2FusedKernelWithCaching.apply(zxBCdt, logA, D, conv1d_weight, conv1d_bias, dt_bias,
                                              norm_weight, n_groups, ssm_state_size, intermediate_size,
                                              head_dim)


def mamba2_fused_prefill(zxBCdt, logA, D, conv1d_weight, conv1d_bias, dt_bias, norm_weight, n_groups, ssm_state_size,
                         intermediate_size, head_dim, conv_state, ssm_state, continuing=False):
    """Inference forward ``zxBCdt -> norm_out`` that updates the decode cache in place.

    ``conv_state`` (b, conv_dim, W), W in {k-1, k}: on return the last W rows of xBC (before the conv), oldest first.
    ``ssm_state`` (b, h, p, n) fp32: on return the scan's state after the last token.
    ``continuing``: the two tensors hold the state after an earlier prefix (prefill in pieces, or prefill after decode
    steps); otherwise they are taken as zero and only written."""
    return _lib.native().fused_prefill(zxBCdt, logA, D, conv1d_weight, conv1d_bias, dt_bias, _lib.f32_param(norm_weight), n_groups,
                                       ssm_state_size, intermediate_size, head_dim, conv_state, ssm_state, continuing)
