"""GPU parity of the mixer glue kernels (m2_softplus_bias_*, m2_rmsnorm_gated_*) against the fp64 oracle
(oracle/mixer.py: softplus_ref, rmsnorm_gated_ref; backward = autograd through the oracle).

Shapes: the group widths of the reference's configurations (2.7B: 5120 channels in one group; 7B: 8192 in 8 groups of
1024; 370M-like 2048), ragged widths (not a multiple of 64 vectors), row counts that do not fill the last block, column
slices of a packed [z | xBC | dt] buffer, no gate.  Tolerances: fp32 1e-4 relative to RMS; bf16 2e-2 x RMS.
"""
import pytest
import torch

from conftest import rel_rms_err
from oracle.mixer import rmsnorm_gated_ref, softplus_ref

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
TOL = {torch.float32: 1e-4, torch.bfloat16: 2e-2}


def _rand(shape, dtype, seed, scale=1.0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(shape, generator=g) * scale).to(dtype)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("b,l,h", [(2, 100, 4), (4, 2048, 80), (1, 1, 128), (3, 77, 24)])
def test_softplus_bias_fwd_bwd(dtype, b, l, h):
    from mamba2 import glue
    # dt as the last h columns of a wider buffer (the packed projection output), values on both sides of the threshold
    width = 40 + h
    buf = _rand((b, l, width), dtype, 1, scale=6.0)
    bias = _rand((h,), torch.float32, 2)
    dt = buf.to(DEV)[..., 40:]
    out = glue.softplus_bias_hip(dt, bias.to(DEV))
    ref = softplus_ref(buf[..., 40:].double() + bias.double())
    assert out.shape == (b, l, h) and out.dtype == dtype and out.is_contiguous()
    assert rel_rms_err(out.cpu(), ref) < TOL[dtype]
    # backward into a column slice of a gradient buffer
    d_out = _rand((b, l, h), dtype, 3)
    gbuf = torch.full((b, l, width), 7.0, dtype=dtype, device=DEV)
    d_in, d_bias = glue.softplus_bias_bwd_hip(dt, bias.to(DEV), d_out.to(DEV), out_d_in=gbuf[..., 40:])
    v = (buf[..., 40:].double() + bias.double()).requires_grad_(True)
    softplus_ref(v).backward(d_out.double())
    # the kernel takes the derivative above the threshold as exactly 1 (sigmoid(10) = 1 - 4.5e-5)
    assert rel_rms_err(d_in.cpu(), v.grad) < TOL[dtype] + 1e-4
    assert rel_rms_err(d_bias.cpu(), v.grad.sum(dim=(0, 1))) < (1e-4 if dtype == torch.float32 else 2e-3)
    assert torch.equal(gbuf[..., :40], torch.full((b, l, 40), 7.0, dtype=dtype, device=DEV))      # neighbours untouched
    assert d_bias.dtype == torch.float32


NORM_SHAPES = [
    # rows (b, l), channels, groups
    ((2, 96), 5120, 1),        # 2.7B: one group of 5120 (four waves per row, 2.5 vectors per lane)
    ((1, 130), 8192, 8),       # 7B: eight groups of 1024 (one wave per row and group)
    ((2, 37), 2048, 1),        # one wave, four vectors per lane
    ((1, 50), 256, 2),         # groups of 128: 16 vectors, most lanes idle
    ((3, 5), 4160, 1),         # 520 vectors: ragged over 256 threads
    ((1, 3), 8192, 1),         # the widest supported group
]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,d,g", NORM_SHAPES)
@pytest.mark.parametrize("gated", [True, False])
def test_rmsnorm_gated_fwd_bwd(dtype, rows, d, g, gated):
    from mamba2 import glue
    eps = 1e-5
    x = _rand((*rows, d), dtype, 11)
    z = _rand((*rows, d), dtype, 12) if gated else None
    w = 1.0 + 0.2 * _rand((d,), torch.float32, 13)
    dout = _rand((*rows, d), dtype, 14)
    xg, wg, dg = x.to(DEV), w.to(DEV), dout.to(DEV)
    zg = z.to(DEV) if gated else None
    xd = x.double().requires_grad_(True)
    zd = z.double().requires_grad_(True) if gated else None
    wd = w.double().requires_grad_(True)
    ref = rmsnorm_gated_ref(xd, zd, wd, g, eps)
    ref.backward(dout.double())
    # fp32 output: nothing is rounded on the way out, so the bound is the fp32 one whatever the input type
    out32 = glue.rmsnorm_gated_hip(xg, zg, wg, g, eps, out_dtype=torch.float32)
    assert out32.dtype == torch.float32 and out32.shape == x.shape
    assert rel_rms_err(out32.cpu(), ref.detach()) < 1e-4
    # output in the input type: the same values, rounded once
    out = glue.rmsnorm_gated_hip(xg, zg, wg, g, eps, out_dtype=dtype)
    assert out.dtype == dtype and torch.equal(out, out32.to(dtype))
    dx, dw, dz = glue.rmsnorm_gated_bwd_hip(xg, zg, wg, dg, g, eps)
    # dx, dz are stored in the input type.  h = x silu(z) is heavy-tailed (elements beyond 10 RMS), and a bf16 value just
    # above a power of two is off by up to 2^-8 of itself from storage alone: roundings=2 discounts that worst case
    # instead of the 2^-9 best case, the arithmetic (fp32 throughout) must stay inside the tolerance
    assert rel_rms_err(dx.cpu(), xd.grad) < TOL[dtype]
    if gated:
        assert rel_rms_err(dz.cpu(), zd.grad) < TOL[dtype]
    else:
        assert dz is None
    # dw is an fp32 sum over the rows of products of the (bf16) inputs: the inputs are exact, the sum is not rounded to bf16
    assert rel_rms_err(dw.cpu(), wd.grad) < 1e-4 if dtype == torch.float32 else rel_rms_err(dw.cpu(), wd.grad) < 2e-3
    assert dw.dtype == torch.float32


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("width_pad", [0, 4])     # 4: rows of the packed buffer are not 16-byte aligned
def test_rmsnorm_gated_on_packed_views(dtype, width_pad):
    """z and dz as the first d columns of a packed (b, l, d + extra) buffer, as the fused mixer core passes them."""
    from mamba2 import glue
    b, l, d, g, eps = 2, 64, 512, 2, 1e-5
    extra = 136 + width_pad
    packed = _rand((b, l, d + extra), dtype, 21).to(DEV)
    z = packed[..., :d]
    x = _rand((b, l, d), dtype, 22).to(DEV)
    w = (1.0 + 0.1 * _rand((d,), torch.float32, 23)).to(DEV)
    dout = _rand((b, l, d), dtype, 24).to(DEV)
    out = glue.rmsnorm_gated_hip(x, z, w, g, eps, out_dtype=dtype)
    out_c = glue.rmsnorm_gated_hip(x, z.contiguous(), w, g, eps, out_dtype=dtype)
    assert torch.equal(out, out_c)
    gpacked = torch.full((b, l, d + extra), 3.0, dtype=dtype, device=DEV)
    dx, dw, dz = glue.rmsnorm_gated_bwd_hip(x, z, w, dout, g, eps, out_dz=gpacked[..., :d])
    dx_c, dw_c, dz_c = glue.rmsnorm_gated_bwd_hip(x, z.contiguous(), w, dout, g, eps)
    assert torch.equal(dx, dx_c) and torch.equal(dw, dw_c) and torch.equal(gpacked[..., :d], dz_c)
    assert torch.equal(gpacked[..., d:], torch.full((b, l, extra), 3.0, dtype=dtype, device=DEV))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,d", [(128, 2560), (3, 4096), (1, 8192), (130, 100), (5, 1028)])
def test_add_rmsnorm_in_place_residual(dtype, rows, d):
    """residual += delta; out = w * residual * rsqrt(mean(residual^2) + eps): against the fp64 oracle norm of the fp64 sum."""
    from mamba2 import glue
    eps = 1e-5
    res = _rand((rows, d), torch.float32, 31, scale=3.0)
    delta = _rand((rows, d), dtype, 32)
    w = 1.0 + 0.2 * _rand((d,), torch.float32, 33)
    rg = res.to(DEV)
    out = glue.add_rmsnorm_(rg, delta.to(DEV), w.to(DEV), eps, dtype)
    s = res.double() + delta.double()
    ref = rmsnorm_gated_ref(s, None, w.double(), 1, eps)
    assert out.dtype == dtype and out.shape == (rows, d)
    assert rel_rms_err(rg.cpu(), s) < 1e-6                     # the residual stream stays fp32
    assert rel_rms_err(out.cpu(), ref) < TOL[dtype]
    # nothing to add: the residual is left alone
    before = rg.clone()
    out2 = glue.add_rmsnorm_(rg, None, w.to(DEV), eps, dtype)
    assert torch.equal(rg, before) and torch.equal(out2, out)
    with pytest.raises(ValueError):
        glue.add_rmsnorm_(torch.zeros(2, 8200, device=DEV), None, torch.ones(8200, device=DEV), eps, dtype)


def test_glue_empty_and_errors():
    from mamba2 import glue
    x = torch.empty(0, 4, 512, dtype=torch.bfloat16, device=DEV)
    w = torch.ones(512, device=DEV)
    assert glue.rmsnorm_gated_hip(x, x, w, 1, 1e-5).shape == (0, 4, 512)
    dx, dw, dz = glue.rmsnorm_gated_bwd_hip(x, x, w, x, 1, 1e-5)
    assert dx.shape == x.shape and torch.equal(dw, torch.zeros(512, device=DEV))
    dt = torch.empty(0, 3, 8, dtype=torch.bfloat16, device=DEV)
    d_in, d_bias = glue.softplus_bias_bwd_hip(dt, torch.zeros(8, device=DEV), dt)
    assert torch.equal(d_bias, torch.zeros(8, device=DEV))
    with pytest.raises(ValueError):      # group wider than the kernels hold in registers
        glue.rmsnorm_gated_hip(torch.zeros(2, 16384, dtype=torch.bfloat16, device=DEV), None, torch.ones(16384, device=DEV), 1, 1e-5)
    with pytest.raises(ValueError):      # channels per group not a multiple of the vector width
        glue.rmsnorm_gated_hip(torch.zeros(2, 36, dtype=torch.bfloat16, device=DEV), None, torch.ones(36, device=DEV), 3, 1e-5)
    with pytest.raises(RuntimeError):    # no CPU path
        glue.rmsnorm_gated_hip(torch.zeros(2, 64), None, torch.ones(64), 1, 1e-5)


@pytest.mark.parametrize("norm_rows,channels,norm_dtype", [(0, 40, torch.float32), (1, 33, torch.bfloat16), (3, 64, torch.float32), (257, 132, torch.bfloat16), (5, 0, torch.float32)])
@pytest.mark.parametrize("slots,conv_channels,conv_dtype", [(0, 7, torch.float32), (1, 9, torch.bfloat16), (6, 130, torch.float32)])
@pytest.mark.parametrize("heads,times_A,dtypes", [(0, True, (torch.float32,) * 3), (5, False, (torch.bfloat16, torch.float32, torch.bfloat16)), (1500, True, (torch.float32, torch.bfloat16, torch.float32))])
def test_param_sums(norm_rows, channels, norm_dtype, slots, conv_channels, conv_dtype, heads, times_A, dtypes):
    """Each part of the joint launch against fp64 sums of the same partials, at the edges of its workgroups; parts that are absent."""
    from mamba2 import _lib
    lib = _lib.load()
    torch.manual_seed(norm_rows + slots + heads)
    r = lambda *shape: torch.randn(*shape, device="cuda")
    rows, conv = r(max(norm_rows, 1), max(channels, 1)), r(max(slots, 1), conv_channels, 5)
    A, dA, dD, db = (r(max(heads, 1)) for _ in range(4))
    new = lambda n, dtype: torch.full((max(n, 1),), 7.0, device="cuda", dtype=dtype)
    o_norm, o_w, o_b = new(channels, norm_dtype), new(conv_channels * 4, conv_dtype), new(conv_channels, conv_dtype)
    o_A, o_D, o_db = (new(heads, t) for t in dtypes)
    code, ptr = _lib.dtype_code, _lib.ptr
    _lib.check(lib.m2_param_sums(ptr(rows), norm_rows, channels, ptr(o_norm), code(norm_dtype), ptr(conv), slots, conv_channels, ptr(o_w), ptr(o_b),
                                 code(conv_dtype), heads, ptr(A) if times_A else None, ptr(dA), ptr(dD), ptr(db), ptr(o_A), code(dtypes[0]), ptr(o_D),
                                 code(dtypes[1]), ptr(o_db), code(dtypes[2]), _lib.stream_ptr()), "param_sums")

    def close(got, want, terms):
        # fp32 sums: half an ulp of the largest partial sum per addition; bf16 results: half an ulp of the value on top
        bound = terms * 2.0 ** -24 * (want.abs().max() + 4 * terms ** 0.5) + (2.0 ** -8 * want.abs() if got.dtype == torch.bfloat16 else 0.0)
        assert ((got.double() - want).abs() <= bound).all()

    if channels:
        close(o_norm[:channels], rows[:norm_rows].double().sum(0), max(norm_rows, 1))
    if slots:
        s = conv.double().sum(0)
        close(o_w, s[:, :4].reshape(-1), slots)
        close(o_b, s[:, 4], slots)
    else:
        assert (o_w == 7).all() and (o_b == 7).all()
    if heads:
        close(o_A, dA.double() * (A.double() if times_A else 1.0), 1)
        close(o_D, dD.double(), 1)
        close(o_db, db.double(), 1)
    else:
        assert (o_A == 7).all()


@pytest.mark.parametrize("heads,channels,with_D,types", [(24, 1536, True, (torch.bfloat16,) * 4), (5, 33, False, (torch.float32, torch.bfloat16, torch.bfloat16, torch.float32))])
def test_mixer_params_and_their_gradients(heads, channels, with_D, types):
    """The small parameters into fp32 and their gradients back into the parameters' types: products and casts, one rounding each."""
    from mamba2 import _lib
    lib, code, ptr = _lib.load(), _lib.dtype_code, _lib.ptr
    torch.manual_seed(heads)
    A_log, D, dt_bias, norm = (torch.randn(n, device=DEV).to(t) for n, t in zip((heads, heads, heads, channels), types))
    out = torch.full((3 * heads + channels,), 7.0, device=DEV)
    _lib.check(lib.m2_mixer_params(ptr(A_log), code(types[0]), ptr(D) if with_D else None, code(types[1]), ptr(dt_bias), code(types[2]), ptr(norm),
                                   code(types[3]), ptr(out), heads, channels, _lib.stream_ptr()), "mixer_params")
    A, D32, bias32, norm32 = out.split((heads, heads, heads, channels))
    assert ((A.double() + A_log.double().exp()).abs() <= 2.0 ** -21 * A.double().abs()).all()      # expf: a few ulp
    assert torch.equal(bias32, dt_bias.float()) and torch.equal(norm32, norm.float())
    assert torch.equal(D32, D.float()) if with_D else (D32 == 7).all()
    dA, dD, db, dn = (torch.randn(n, device=DEV) for n in (heads, heads, heads, channels))
    got = [torch.full((n,), 7.0, device=DEV, dtype=t) for n, t in zip((heads, heads, heads, channels), types)]
    _lib.check(lib.m2_mixer_params_grads(ptr(A), ptr(dA), ptr(dD) if with_D else None, ptr(db), ptr(dn), ptr(got[0]), code(types[0]), ptr(got[1]) if with_D else None,
                                         code(types[1]), ptr(got[2]), code(types[2]), ptr(got[3]), code(types[3]), heads, channels, _lib.stream_ptr()), "mixer_params_grads")
    for name, a, want in zip(("A_log", "D", "dt_bias", "norm"), got, (A * dA, dD, db, dn)):
        assert torch.equal(a, want.to(a.dtype)) if name != "D" or with_D else (a == 7).all(), name


# rows per workgroup: one, two and four workgroups per CU, one row each, a last workgroup (or its last waves) with fewer rows or none
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,d,g", [(1029, 2048, 1), (7003, 1024, 1), (301, 8192, 8), (5001, 512, 1), (641, 4096, 8), (1100, 4096, 1), (1101, 5120, 1), (3001, 2560, 1),
                                      (515, 7168, 1)])
def test_rmsnorm_gated_rows_per_workgroup(dtype, rows, d, g):
    test_rmsnorm_gated_fwd_bwd(dtype, (1, rows), d, g, True)


# groups that share a wave: eight, four and two of them, with idle lanes in each, spare lanes behind the last group, fewer groups than a wave
# could take, and 32 vectors against 33
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,d,g", [(2003, 512, 8), (5, 2048, 32), (77, 576, 3), (130, 384, 2), (33, 40, 5), (1, 128, 2), (9, 1024, 4), (9, 1056, 4), (9, 544, 4)])
@pytest.mark.parametrize("gated", [True, False])
def test_rmsnorm_gated_groups_that_share_a_wave(dtype, rows, d, g, gated):
    test_rmsnorm_gated_fwd_bwd(dtype, (1, rows), d, g, gated)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,d,g,extra,first", [(131, 512, 8, 13, 0), (70, 2048, 1, 1, 3), (33, 5120, 1, 7, 1), (1, 896, 1, 271, 0), (40, 4096, 1, 2, 5)])
def test_core_norm_reads_the_gate_on_any_element(dtype, rows, d, g, extra, first):
    """z in rows of a width that is no multiple of a vector, from any element on: the values of an aligned copy, forward and backward."""
    import ctypes
    from mamba2 import _lib
    lib, ptr = _lib.load(), _lib.ptr
    packed = _rand((rows * (d + extra) + first,), dtype, 41).to(DEV)
    z = packed[first:].view(rows, d + extra)[:, :d]
    x, dout, w = _rand((rows, d), dtype, 42).to(DEV), _rand((rows, d), dtype, 43).to(DEV), (1 + 0.1 * _rand((d,), torch.float32, 44)).to(DEV)
    need = lib.m2_rmsnorm_gated_bwd_workspace_bytes(rows, d, g, _lib.dtype_code(dtype))

    def call(gate):
        out, dx, dz, ws = torch.zeros_like(x), torch.zeros_like(x), torch.zeros_like(x), torch.zeros(need // 4, device=DEV)
        p = _lib.RmsnormParams(x=ptr(x), z=ptr(gate), weight=ptr(w), out=ptr(out), d_out=ptr(dout), dx=ptr(dx), dz=ptr(dz), workspace=ptr(ws), workspace_bytes=need, rows=rows,
                               channels=d, x_stride_row=d, z_stride_row=gate.stride(0), out_stride_row=d, d_out_stride_row=d, dx_stride_row=d, dz_stride_row=d, n_groups=g,
                               dtype=_lib.dtype_code(dtype), eps=1e-5)
        n = ctypes.c_int64(-1)
        _lib.check(lib.m2_core_norm_fwd(ctypes.byref(p), _lib.stream_ptr()), "core_norm_fwd")
        _lib.check(lib.m2_core_norm_bwd_partial(ctypes.byref(p), ctypes.byref(n), _lib.stream_ptr()), "core_norm_bwd_partial")
        refused = lib.m2_rmsnorm_gated_fwd(ctypes.byref(p), _lib.stream_ptr()) != 0
        return (out, dx, dz, ws[:n.value * d]), refused

    whole = z.clone(memory_format=torch.contiguous_format)
    for a, b in zip(call(z)[0], call(whole)[0]):
        assert torch.equal(a, b)
    assert call(z)[1] and not call(whole)[1]      # the plain entry asks for whole vectors, as before


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,d,g", [(5, 512, 8), (3, 512, 1), (4, 2560, 1), (2, 1088, 1)])
def test_rmsnorm_gated_weight_on_any_element(dtype, rows, d, g):
    """The weights come in 16-byte pieces: from a tensor that starts on any element the same bits, forward and backward."""
    from mamba2 import glue
    x, z, dout = (_rand((rows, d), dtype, s).to(DEV) for s in (51, 52, 53))
    w = (1 + 0.2 * _rand((d,), torch.float32, 54)).to(DEV)
    odd = torch.empty(d + 1, device=DEV)[1:].copy_(w)
    assert odd.data_ptr() % 16 == 4
    got = [(glue.rmsnorm_gated_hip(x, z, v, g, 1e-5), *glue.rmsnorm_gated_bwd_hip(x, z, v, dout, g, 1e-5)) for v in (w, odd)]
    assert all(torch.equal(a, b) for a, b in zip(*got))


# rows per workgroup: a row each and chains of two in one launch shape's range, five rows per CU and one more, idle lanes with few and many rows, a vector
# and a quarter a lane
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,d,g", [(513, 8192, 8), (3700, 1024, 1), (4500, 512, 1), (1280, 4096, 1), (1281, 4096, 1), (257, 2560, 1), (1537, 2560, 1), (2600, 640, 2), (400, 1536, 8)])
def test_rmsnorm_gated_workgroups_per_cu(dtype, rows, d, g):
    test_rmsnorm_gated_fwd_bwd(dtype, (1, rows), d, g, True)
