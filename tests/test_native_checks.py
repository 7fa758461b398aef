"""CPU: what the operators' host code refuses before it looks at a device: sizes that do not fit together are a ValueError, whatever
the tensors' device, and never an end of the process."""
import ctypes

import pytest
import torch


def _core_args(h, d, g, n, l=8):
    conv = d + 2 * g * n
    return (torch.zeros(1, l, d + conv + h), -torch.ones(h), torch.ones(h), torch.zeros(conv, 1, 4), torch.zeros(conv), torch.zeros(h), torch.ones(d))


@pytest.mark.parametrize("d,head_dim,g,message", [(96, 64, 1, "not a multiple of head_dim"), (64, 0, 1, "not a multiple of head_dim"),
                                                  (64, -64, 1, "not a multiple of head_dim"), (128, 64, 0, "not divisible by n_groups"),
                                                  (128, 64, 3, "not divisible by n_groups")])
def test_core_refuses_channels_that_are_no_whole_heads(d, head_dim, g, message):
    from mamba2 import _lib
    from mamba2.fused_kernel import mamba2_fused_kernel, mamba2_fused_kernel_with_caching, mamba2_fused_prefill
    h, n = d // head_dim if head_dim > 0 else 1, 64
    args = _core_args(h, d, g, n)
    for core in (mamba2_fused_kernel, mamba2_fused_kernel_with_caching):
        with pytest.raises(ValueError, match=message):
            core(*args, g, n, d, head_dim)
    with pytest.raises(ValueError, match=message):
        mamba2_fused_prefill(*args, g, n, d, head_dim, torch.zeros(1, d + 2 * g * n, 3), torch.zeros(1, h, 64, n))
    hidden, width = torch.zeros(1, 8, 32), 2 * d + 2 * g * n + h
    with pytest.raises(ValueError, match=message):
        _lib.native().mixer(hidden, torch.zeros(width, 32), args[1], args[2], args[5], args[3], args[6], torch.zeros(32, d), args[4], None, None,
                            g, n, d, head_dim, False)


def test_no_groups_is_an_error_and_not_a_division(lib):
    from mamba2 import _lib
    from mamba2.mamba2_kernel import mamba2_kernel
    with pytest.raises(ValueError, match="not divisible by n_groups"):
        mamba2_kernel(torch.zeros(1, 128, 2), torch.zeros(2), torch.zeros(1, 128, 2, 64), torch.zeros(1, 128, 0, 64), torch.zeros(1, 128, 0, 64), torch.zeros(2))
    p = _lib.SsdParams()
    p.batch, p.seqlen, p.nheads, p.headdim, p.dstate, p.ngroups = 1, 128, 2, 64, 64, 0
    assert lib.m2_ssd_bwd_workspace_bytes(ctypes.byref(p)) > 0
    assert lib.m2_ssd_bwd(ctypes.byref(p), None) == -1


def test_small_products_refuse_what_their_addressing_does_not_reach(lib):
    from mamba2 import _lib
    p = _lib.LinearParams(x=16, w=16, out=16, M=32, N=64, K=64, x_stride_row=1 << 26, out_stride_row=64, groups=1)
    assert lib.m2_linear_small(ctypes.byref(p), None) == -1 and b"32-bit" in lib.m2_last_error()
    p.x_stride_row, p.w = 64, 24
    assert lib.m2_linear_small(ctypes.byref(p), None) == -3


def test_every_struct_of_the_header_is_mirrored_and_reported(lib):
    """Each parameter struct that the header declares: its fields in the ctypes mirror, its size and offsets as the library was built."""
    import os
    import re

    from mamba2 import _lib
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    text = re.sub(r"/\*.*?\*/", "", open(os.path.join(root, "include", "mamba2_hip.h")).read(), flags=re.S)
    declared = re.findall(r"typedef struct (m2_\w+) \{(.*?)\} \1;", text, flags=re.S)
    mirrors = {"m2_conv1d_params": _lib.Conv1dParams, "m2_ssd_params": _lib.SsdParams, "m2_decode_params": _lib.DecodeParams,
               "m2_rmsnorm_params": _lib.RmsnormParams, "m2_linear_params": _lib.LinearParams, "m2_product_params": _lib.ProductParams}
    assert [name for name, _ in declared] == list(mirrors)
    for which, (name, body) in enumerate(declared):
        fields = [re.split(r"[\s*]+", f.strip())[-1] for decl in body.split(";") if decl.strip() for f in decl.split(",")]
        mirror = mirrors[name]
        assert fields == [f[0] for f in mirror._fields_], name
        buf = (ctypes.c_int64 * 128)()
        assert lib.m2_struct_layout(which, buf, 128) == 1 + len(fields), name
        assert buf[0] == ctypes.sizeof(mirror) and list(buf[1:1 + len(fields)]) == [getattr(mirror, f).offset for f in fields], name
    assert lib.m2_struct_layout(len(declared), (ctypes.c_int64 * 4)(), 4) == -1


@pytest.mark.parametrize("dtype,b,l,h,p,n,g,slices", [(1, 2, 4096, 128, 64, 128, 8, (1, 1)), (0, 3, 2048, 16, 128, 128, 8, (1, 1)), (1, 1, 17, 1, 64, 64, 1, (1, 1)),
                                                      (1, 4, 2048, 80, 64, 128, 1, (4, 4)), (0, 1, 256, 8, 64, 64, 1, (8, 8))])
def test_scan_backward_asks_for_what_its_kernels_write(lib, dtype, b, l, h, p, n, g, slices):
    """Workspace beside the buffer that the forward left, counted from the kernels: state gradients, per-token and per-chunk rows, and
    of dG, dB and dC a partial per slice and a sum only where there are several slices."""
    from mamba2 import _lib
    q = 128
    params = _lib.SsdParams(batch=b, seqlen=l, nheads=h, headdim=p, dstate=n, ngroups=g, dtype=dtype, dt_dtype=dtype, chunk_states=256)
    chunks, size, (s_g, s_b) = -(-l // q), 2 if dtype else 4, slices
    bhc, groups = b * (h * p // 64) * chunks, b * chunks * g
    want = bhc * 64 * n * size + bhc * 4 * (8 + 3 + 4 * q + 8) + (0 if dtype else bhc * 64 * n * 4)
    done = s_g == s_b == 1
    want += groups * q * q * 4 * ((0 if done and not dtype else s_g) + (s_g > 1)) + 2 * groups * q * n * 4 * ((0 if done else s_b) + (s_b > 1))
    got = lib.m2_ssd_bwd_workspace_bytes(ctypes.byref(params))
    assert want <= got <= want + 20 * 256, (got, want)


@pytest.mark.parametrize("chunks", [19, 20, 27, 28, 47, 48])
def test_scan_asks_for_segments_where_a_walk_goes_in_them(lib, chunks):
    """Few heads, many chunks: room for the segments' states from 20 chunks (a forward), 28 (one that keeps its states for the backward) and 48 (a backward)."""
    from mamba2 import _lib
    h, n, q = 8, 128, 128
    m = max(2, -(-chunks // 17))                       # 16 half heads: 16 sets of them on 256 CUs
    seg = (-(-chunks // m) - 1) * h * (64 * n + 1) * 4
    p = _lib.SsdParams(batch=1, seqlen=chunks * q, nheads=h, headdim=64, dstate=n, ngroups=h, dtype=1, dt_dtype=1)
    kept = lib.m2_ssd_chunk_states_bytes(ctypes.byref(p))
    assert 0 <= lib.m2_ssd_fwd_workspace_bytes(ctypes.byref(p)) - kept - (seg if chunks >= 20 else 0) <= 4 * 256
    p.chunk_states = 256
    assert 0 <= lib.m2_ssd_fwd_workspace_bytes(ctypes.byref(p)) - (seg if chunks >= 28 else 0) <= 4 * 256
    bhc = h * chunks
    want = bhc * 64 * n * 2 + bhc * 4 * (8 + 3 + 4 * q + 8) + bhc * q * q * 4 + (seg if chunks >= 48 else 0)      # a head a group: whole groups, one slice
    assert 0 <= lib.m2_ssd_bwd_workspace_bytes(ctypes.byref(p)) - want <= 20 * 256


@pytest.mark.parametrize("tokens,ins,outs,pays", [(500, 768, 3352, 1), (40, 2048, 1024, 1), (23291, 592, 296, 0), (15785, 736, 368, 0), (4395, 896, 448, 0)])
def test_product_pairs_leave_long_sums_to_products_that_split_them(lib, tokens, ins, outs, pays):
    from mamba2 import _lib
    x = _lib.ProductParams(M=tokens, N=ins, K=outs, a_k=1, b_k=0)
    w = _lib.ProductParams(M=outs, N=ins, K=tokens, a_k=0, b_k=0)
    assert lib.m2_product_pair_pays(x, w) == pays


def test_norm_checks_say_what_the_norms_refuse(lib):
    """Both checks, on the host alone: a group of over 8192 channels, an output off its vectors, and a gate off its vectors, which the core's takes."""
    from mamba2 import _lib
    plain, core = lib.m2_rmsnorm_gated_fwd_check, lib.m2_core_norm_fwd_check

    def params(channels=512, z=32, z_stride=512, out=48, out_stride=512, groups=1):
        return _lib.RmsnormParams(x=16, z=z, weight=4, out=out, rows=3, channels=channels, x_stride_row=channels, z_stride_row=z_stride, out_stride_row=out_stride,
                                  n_groups=groups, dtype=1, eps=1e-5)

    for p, wanted in ((params(), (0, 0)), (params(z=34), (-3, 0)), (params(z_stride=515), (-3, 0)), (params(out=50), (-3, -3)), (params(out_stride=516), (-3, -3)),
                      (params(channels=8256, z_stride=8256, out_stride=8256), (-1, -1)), (params(channels=8256, z_stride=8257, out_stride=8256, groups=3), (-3, 0)),
                      (params(z=0, out=0), (-6, -6))):
        assert (plain(ctypes.byref(p)), core(ctypes.byref(p))) == wanted
