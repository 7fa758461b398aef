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
