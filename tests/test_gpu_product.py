"""GPU: the products of a layer's projections on few tokens, in the storage forms of a linear layer's forward and backward, at the
edges of their tiles and k splits, against fp64 on the CPU."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _taken(M, K, a_k, b_k):
    """What the storage asks for: the contiguous extent of each operand (k, or the rows of a transposed A) in eights."""
    return not ((a_k or b_k) and K % 8) and (a_k or not M % 8)


SIZES = [(1, 8, 8), (8, 8, 1), (64, 64, 64), (65, 72, 72), (72, 200, 1000), (40, 64, 5), (200, 2560, 520), (136, 264, 2056), (1000, 1544, 136)]
FORMS = [(*s, *f) for s in SIZES for f in ((1, 1), (1, 0), (0, 0), (0, 1))]


@pytest.mark.parametrize("M,N,K,a_k,b_k", [f for f in FORMS if _taken(f[0], f[2], f[3], f[4])])
@pytest.mark.parametrize("pad", [0, 8])
def test_product(M, N, K, a_k, b_k, pad):
    from mamba2 import _lib
    lib = _lib.load()
    assert lib.m2_product_fits(M, N, K, a_k, b_k)
    gen = torch.Generator().manual_seed(M + N + K)
    a, b = (torch.randn(r, K, generator=gen).bfloat16() for r in (M, N))
    bias = torch.randn(N, generator=gen).bfloat16()
    ref = a.double() @ b.double().T + bias.double()

    def stored(t, k):      # rows of the operand as it lies in memory, NaN behind their ends
        t = t if k else t.T
        buf = torch.full((t.shape[0], -(-t.shape[1] // 8) * 8 + pad), float("nan"), dtype=t.dtype)
        buf[:, :t.shape[1]] = t
        return buf.to(DEV)

    ad, bd, biasd = stored(a, a_k), stored(b, b_k), bias.to(DEV)
    out = torch.full((M, N + pad), 7.0, dtype=torch.bfloat16, device=DEV)
    n = lib.m2_product_workspace_bytes(M, N, K)
    ws = torch.empty(max(n, 1), dtype=torch.uint8, device=DEV)
    p = _lib.ProductParams(a=_lib.ptr(ad), b=_lib.ptr(bd), bias=_lib.ptr(biasd), out=_lib.ptr(out), workspace=_lib.ptr(ws), workspace_bytes=n, M=M, N=N, K=K,
                           lda=ad.stride(0), ldb=bd.stride(0), ldo=N + pad, a_k=a_k, b_k=b_k)
    _lib.check(lib.m2_product(p, _lib.stream_ptr()), "m2_product")
    got = out.double().cpu()
    assert ((got[:, :N] - ref).norm() / ref.norm()).item() < 4e-3
    assert (got[:, N:] == 7.0).all()


# tiles and splits whose count is no multiple of the XCDs: six and five splits of the small tile, several of the large one
@pytest.mark.parametrize("M,N,K", [(65, 136, 3200), (264, 1288, 3336), (136, 2568, 4104), (200, 2568, 5128), (192, 4104, 1032)])
@pytest.mark.parametrize("a_k,b_k", [(1, 1), (1, 0), (0, 0)])
def test_product_shares(M, N, K, a_k, b_k):
    if _taken(M, K, a_k, b_k):
        test_product(M, N, K, a_k, b_k, 0)


@pytest.mark.parametrize("M,N,K,a_k,b_k", [f for f in FORMS if not _taken(f[0], f[2], f[3], f[4])] + [(64, 12, 64, 1, 1), (0, 64, 64, 1, 1)])
def test_product_refuses_other_storage(M, N, K, a_k, b_k):
    from mamba2 import _lib
    lib = _lib.load()
    assert not lib.m2_product_fits(M, N, K, a_k, b_k)
    t = torch.zeros(1 << 14, dtype=torch.bfloat16, device=DEV)          # refused before any of it is read
    p = _lib.ProductParams(a=_lib.ptr(t), b=_lib.ptr(t), out=_lib.ptr(t), M=M, N=N, K=K, lda=8, ldb=8, ldo=8, a_k=a_k, b_k=b_k)
    with pytest.raises(ValueError, match="is not taken"):
        _lib.check(lib.m2_product(p, _lib.stream_ptr()), "m2_product")


# both products of a linear layer's backward in one launch: single and ragged tiles, either chain the longer one, dx split over k
@pytest.mark.parametrize("tokens,outs,ins", [(1, 8, 8), (64, 64, 64), (65, 72, 200), (1000, 72, 136), (500, 3352, 264), (40, 4104, 64)])
@pytest.mark.parametrize("pad", [0, 8])
def test_product_pair(tokens, outs, ins, pad):
    from mamba2 import _lib
    lib = _lib.load()
    gen = torch.Generator().manual_seed(tokens + outs)
    dy, w, x = (torch.randn(r, c, generator=gen).bfloat16() for r, c in ((tokens, outs), (outs, ins), (tokens, ins)))

    def stored(t):      # NaN behind the rows' ends
        buf = torch.full((t.shape[0], t.shape[1] + pad), float("nan"), dtype=t.dtype)
        buf[:, :t.shape[1]] = t
        return buf.to(DEV)

    dyd, wd, xd = stored(dy), stored(w), stored(x)
    dx, dw = (torch.full((r, ins + pad), 7.0, dtype=torch.bfloat16, device=DEV) for r in (tokens, outs))
    px = _lib.ProductParams(a=_lib.ptr(dyd), b=_lib.ptr(wd), out=_lib.ptr(dx), M=tokens, N=ins, K=outs, lda=outs + pad, ldb=ins + pad, ldo=ins + pad, a_k=1, b_k=0)
    pw = _lib.ProductParams(a=_lib.ptr(dyd), b=_lib.ptr(xd), out=_lib.ptr(dw), M=outs, N=ins, K=tokens, lda=outs + pad, ldb=ins + pad, ldo=ins + pad, a_k=0, b_k=0)
    n = lib.m2_product_pair_workspace_bytes(px, pw)
    ws = torch.empty(max(n, 1), dtype=torch.uint8, device=DEV)
    px.workspace, px.workspace_bytes = _lib.ptr(ws), n
    _lib.check(lib.m2_product_pair(px, pw, _lib.stream_ptr()), "m2_product_pair")
    for out, ref in ((dx, dy.double() @ w.double()), (dw, dy.double().T @ x.double())):
        got = out.double().cpu()
        assert ((got[:, :ins] - ref).norm() / ref.norm()).item() < 4e-3      # one rounding to bf16: 2^-9 at most per value
        assert (got[:, ins:] == 7.0).all()
    if n:
        px.workspace_bytes = n - 1
        with pytest.raises(RuntimeError, match="workspace too small"):
            _lib.check(lib.m2_product_pair(px, pw, _lib.stream_ptr()), "m2_product_pair")
