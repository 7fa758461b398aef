"""GPU: the conv kernels at the edges of their pieces, in both layouts: rows shorter than a vector, one past it, rows that start
anywhere (odd channel or token counts), several splits per channel, each activation."""
import pytest
import torch

from conftest import rel_err, rel_rms_err
from oracle.conv import conv1d_grads_ref, make_conv_inputs

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("channels_last,b,l,C,act", [
    (False, 1, 1, 3, "silu"), (False, 2, 15, 5, None), (False, 1, 16, 700, "silu"), (False, 3, 17, 8, "relu"),
    (False, 2, 333, 40, "silu"), (False, 1, 4099, 3, "silu"), (False, 5, 2048, 64, "silu"),
    (True, 2, 70, 9, "silu"), (True, 1, 33, 131, "relu"), (True, 3, 129, 1025, None), (True, 1, 5, 1, "silu")])
def test_conv_layout_edges(dtype, channels_last, b, l, C, act):
    from mamba2.conv1d_grouped import conv1d_backward, conv1d_forward
    d = make_conv_inputs(b, l, C, seed=l + C, dtype=dtype)
    if not channels_last:
        d["x"], d["dy"] = (d[k].transpose(1, 2).contiguous() for k in ("x", "dy"))
    ref = conv1d_grads_ref(*(d[k].double() for k in ("x", "w", "bias", "dy")), act, channels_last=channels_last)
    x, w, bias, dy = (d[k].to(DEV) for k in ("x", "w", "bias", "dy"))
    got = (conv1d_forward(x, w, bias, act, channels_last=channels_last),
           *conv1d_backward(x, w, bias, dy, act, channels_last=channels_last))
    tol, metric = (1e-4, rel_err) if dtype == torch.float32 else (2e-2, rel_rms_err)
    for name, a, r in zip(("y", "dx", "dw", "db"), got, ref):
        assert metric(a, r) < tol, name


@pytest.mark.parametrize("l1,l2,k,W", [(5, 1, 4, 4), (1, 2, 4, 3), (16, 17, 4, 4), (130, 3, 4, 4), (7, 40, 2, 3), (2, 1, 3, 5)])
@pytest.mark.parametrize("dtype,state_dtype", [(torch.bfloat16, torch.bfloat16), (torch.bfloat16, torch.float32), (torch.float32, torch.float32)])
@pytest.mark.parametrize("strided", [False, True])
def test_prefill_in_two_pieces(l1, l2, k, W, dtype, state_dtype, strided):
    """The conv with the cache in front of it, and what it leaves there, against one pass over the whole sequence."""
    from mamba2.fused_kernel import mamba2_fused_prefill
    torch.manual_seed(l1 * 100 + l2)
    b, h, p, n, g = 2, 8, 64, 64, 1
    d, c, l = h * p, h * p + 2 * g * n, l1 + l2
    zx = (torch.randn(b, l, d + c + h, device="cuda") * 0.5).to(dtype)
    A, D, dt_bias = -torch.rand(h, device="cuda") - 0.5, torch.randn(h, device="cuda"), torch.randn(h, device="cuda")
    conv_w, conv_b = (torch.randn(c, 1, k, device="cuda") * 0.3).to(dtype), torch.randn(c, device="cuda").to(dtype)
    norm_w = torch.rand(d, device="cuda") + 0.5

    def states():
        if strided:
            return (torch.empty(b, c, 2 * W, device="cuda", dtype=state_dtype)[..., ::2], torch.empty(b, h, n, p, device="cuda").transpose(2, 3))
        return torch.empty(b, c, W, device="cuda", dtype=state_dtype), torch.empty(b, h, p, n, device="cuda")

    def run(part, st, continuing):
        return mamba2_fused_prefill(part, A, D, conv_w, conv_b, dt_bias, norm_w, g, n, d, p, *st, continuing=continuing)

    one, two = states(), states()
    whole = run(zx, one, False)
    pieces = torch.cat([run(zx[:, :l1], two, False), run(zx[:, l1:], two, True)], 1)
    tail = torch.nn.functional.pad(zx[:, :, d:d + c], (0, 0, W, 0))[:, l:].transpose(1, 2)
    assert torch.equal(one[0].float(), tail.float()) and torch.equal(two[0].float(), tail.float())
    tol = 2e-2 if dtype == torch.bfloat16 else 2e-4
    torch.testing.assert_close(pieces.float(), whole.float(), rtol=tol, atol=tol)
    torch.testing.assert_close(two[1], one[1], rtol=tol, atol=tol)


@pytest.mark.parametrize("C", [8, 12, 9, 64, 257, 260])                     # whole vectors, shared last vectors, more than one block
@pytest.mark.parametrize("W,l", [(3, 1), (3, 2), (4, 3), (5, 4), (5, 1), (8, 3), (8, 6), (11, 40), (4, 16), (4, 129)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("continuing", [0, 1])
def test_prefill_leaves_the_last_inputs(C, W, l, dtype, continuing):
    """The cache after a prefill is, bit for bit, the end of (what it held | the sequence); the outputs those of the conv over both."""
    import ctypes
    from mamba2 import _lib
    from mamba2.conv1d_grouped import conv1d_forward
    lib, b = _lib.load(), 2
    torch.manual_seed(C * 100 + W * 10 + l)
    x = torch.randn(b, l, C, device=DEV).to(dtype)
    w, bias = torch.randn(C, 1, 4, device=DEV).to(dtype), torch.randn(C, device=DEV).to(dtype)
    state = torch.randn(b, C, W, device=DEV).to(dtype)
    before = state.clone() if continuing else torch.zeros_like(state)
    joined = torch.cat([before, x.transpose(1, 2)], 2)
    y = torch.empty_like(x)
    p = _lib.Conv1dParams(x=x.data_ptr(), w=w.data_ptr(), bias=bias.data_ptr(), y=y.data_ptr(), batch=b, seqlen=l, channels=C, k=4,
                          x_stride_b=l * C, x_stride_l=C, x_stride_c=1, y_stride_b=l * C, y_stride_l=C, y_stride_c=1,
                          dtype=_lib.dtype_code(dtype), param_dtype=_lib.dtype_code(dtype), activation=1)
    _lib.check(lib.m2_conv1d_prefill(ctypes.byref(p), _lib.ptr(state), W, continuing, _lib.stream_ptr()), "prefill")
    assert torch.equal(state, joined[:, :, -W:])
    ref = conv1d_forward(joined.transpose(1, 2).contiguous(), w, bias, "silu", channels_last=True)[:, W:]
    assert torch.equal(y, ref)      # the same sums in the same order


@pytest.mark.parametrize("b,l,C", [(1, 3, 64), (1, 9, 130), (1, 800, 1024), (1, 3000, 1024), (2, 4090, 1024), (1, 2060, 4100), (3, 4100, 6000),
                                   (2, 4130, 1024), (1, 12299, 128), (1, 2097125, 4)])
def test_conv_segment_lengths(b, l, C):
    """Sizes on both sides of the rules for the tokens per thread (4, 8, and 16 where the grid needs it, forward; 8, 16, 32 backward,
    the last one also for few channels and for many partial rows), ends inside a segment."""
    from mamba2.conv1d_grouped import conv1d_backward, conv1d_forward
    torch.manual_seed(l)
    x, dy = (torch.randn(b, l, C, device=DEV).bfloat16() for _ in range(2))
    w, bias = torch.randn(C, 1, 4, device=DEV).bfloat16(), torch.randn(C, device=DEV).bfloat16()
    xd, wd, bd = (t.float().requires_grad_(True) for t in (x, w, bias))
    ref = torch.nn.functional.silu(torch.nn.functional.conv1d(xd.transpose(1, 2), wd, bd, padding=3, groups=C)[..., :l]).transpose(1, 2)
    grads = torch.autograd.grad(ref, (xd, wd, bd), dy.float())
    got = (conv1d_forward(x, w, bias, "silu", channels_last=True), *conv1d_backward(x, w, bias, dy, "silu", channels_last=True))
    for name, a, r in zip(("y", "dx", "dw", "db"), got, (ref.detach(), *grads)):
        # one bf16 rounding of the result (2^-9 of it; heavy tails count against the tensor's norm) behind fp32 sums
        assert (a.float() - r).norm() / r.norm() < 2.0 ** -8, name


# channel-major backward: the splits of a channel inside a workgroup (two, four) and in several partial rows; a last workgroup that is not full
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("b,l,C,act", [(1, 2048, 3075, "silu"), (2, 2050, 2049, None), (2, 4100, 1023, "silu")])
def test_conv_channel_major_splits(dtype, b, l, C, act):
    test_conv_layout_edges(dtype, False, b, l, C, act)


# channel-major: every way a row can end inside its last pieces, several channels to a wave and (few channels, long rows) partial rows of sums
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("b,l,C", [(2, l, 37) for l in (2, 4, 7, 8, 9, 10, 11, 12, 13, 15, 18, 19, 20, 22, 24, 27, 29, 31, 34)] +
                         [(3, 160, 70), (9, 115, 65), (2, 5001, 9), (9, 8190, 3)])
def test_conv_channel_major_row_ends(dtype, b, l, C):
    test_conv_layout_edges(dtype, False, b, l, C, "silu")


# channel-major: a channel's rounds over three of a workgroup's four waves, over several workgroups with one round a wave and with more, and the last of
# them without work
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("b,l,C", [(3, 1000, 5), (17, 795, 20), (2, 70001, 2), (5, 2600, 300)])
def test_conv_channel_major_rounds(dtype, b, l, C):
    test_conv_layout_edges(dtype, False, b, l, C, "silu")
