"""GPU: heads of 128 channels run as pairs of 64-channel kernel heads; x, dy and dx with heads further apart than their width."""
import pytest
import torch

from conftest import rel_err, rel_rms_err
from oracle.ssd import make_ssd_inputs, ssd_grads_ref

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("b,l,h,n,g", [(1, 130, 1, 128, 1), (2, 257, 9, 64, 3)])
def test_wide_heads_far_apart(dtype, b, l, h, n, g):
    from mamba2.mamba2_kernel import ssd_backward, ssd_forward
    d = make_ssd_inputs(b, l, h, 128, n, g, seed=l, dtype=dtype)
    ref = ssd_grads_ref(*(d[k].double() for k in ("dt", "A", "X", "B", "C", "D", "dy")), chunk=64)
    v = {k: t.to(DEV) for k, t in d.items()}

    def apart(t):
        wide = torch.zeros(b, l, h, 160, dtype=dtype, device=DEV)
        wide[..., 16:144] = t
        return wide[..., 16:144]

    X, dy, dX = apart(v["X"]), apart(v["dy"]), apart(torch.zeros_like(v["X"]))
    y, S = ssd_forward(v["dt"], v["A"], X, v["B"], v["C"], v["D"], want_final_state=True)
    ddt, dA, _, dB, dC, dD, _ = ssd_backward(v["dt"], v["A"], X, v["B"], v["C"], v["D"], dy, out_dX=dX)
    tol, metric = (1e-4, rel_err) if dtype == torch.float32 else (2e-2, rel_rms_err)
    for name, got in (("y", y), ("final_state", S), ("dX", dX), ("ddt", ddt), ("dA", dA), ("dB", dB), ("dC", dC), ("dD", dD)):
        assert metric(got, ref[name]) < tol, name


@pytest.mark.parametrize("l", [1, 129, 384])
@pytest.mark.parametrize("b,h", [(2, 104), (1, 257), (2, 128)])
def test_whole_heads_per_workgroup(b, h, l):
    """The state passes at head counts on either side of where a workgroup takes a whole head, over one, two and three chunks."""
    from mamba2.mamba2_kernel import ssd_backward, ssd_forward
    d = make_ssd_inputs(b, l, h, 64, 128, 1, seed=l + h, dtype=torch.bfloat16)
    v = {k: t.to(DEV) for k, t in d.items()}
    some = [0, h // 2, h - 1]      # heads are independent up to dB and dC, which sum over them
    X, dy, dt = (d[k][:, :, some].double() for k in ("X", "dy", "dt"))
    ref = ssd_grads_ref(dt, d["A"][some].double(), X, d["B"].double(), d["C"].double(), d["D"][some].double(), dy, chunk=64)
    y, _ = ssd_forward(v["dt"], v["A"], v["X"], v["B"], v["C"], v["D"])
    ddt, dA, dX, dB, dC, dD, _ = ssd_backward(v["dt"], v["A"], v["X"], v["B"], v["C"], v["D"], v["dy"])
    for name, got in (("y", y[:, :, some]), ("dX", dX[:, :, some]), ("ddt", ddt[:, :, some]), ("dA", dA[some]), ("dD", dD[some])):
        assert rel_rms_err(got, ref[name]) < 2e-2, name
    assert torch.isfinite(dB.float()).all() and torch.isfinite(dC.float()).all()
