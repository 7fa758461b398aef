"""GPU: the small products and the three-launch decode step of a layer, at the edges of their tiles (rows and outputs that are no
multiple of 16, fewer k steps than waves, one and two column tiles, shapes that fall back), against fp64 on the CPU."""
import pytest
import torch

from oracle.decode import decode_step_ref
from oracle.mixer import rmsnorm_gated_ref, softplus_ref

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _rel(got, ref):
    return ((got.double().cpu() - ref).norm() / ref.norm()).item()


@pytest.mark.parametrize("M,N,K,groups", [(1, 5, 64, 1), (3, 16, 192, 1), (9, 40, 320, 1), (16, 33, 1024, 4), (17, 100, 2560, 8), (32, 4384, 1024, 1), (8, 20000, 256, 2),
                                          (2, 256, 5120, 8)])
@pytest.mark.parametrize("normed,out_kind", [(False, 0), (True, 1), (True, 2)])
def test_linear_small(M, N, K, groups, normed, out_kind):
    from mamba2 import _lib
    lib = _lib.load()
    assert lib.m2_linear_small_fits(M, N, K, groups)
    gen = torch.Generator().manual_seed(M + N)
    w = (torch.randn(N, K, generator=gen) / K ** 0.5).bfloat16().to(DEV)
    bias = torch.randn(N, generator=gen).bfloat16().to(DEV)
    next_w = (1 + 0.1 * torch.randn(N, generator=gen)).to(DEV)
    x = torch.randn(M, K, generator=gen).bfloat16().to(DEV)
    sq = torch.rand(M, groups * 3, generator=gen).to(DEV) * K / 3 / groups
    base = torch.randn(M, N, generator=gen)
    out = base.bfloat16().to(DEV) if out_kind == 0 else base.to(DEV)
    nx, nsq = torch.empty(M, N, dtype=torch.bfloat16, device=DEV), torch.empty(M, -(-N // 16), device=DEV)
    p = _lib.LinearParams()
    p.x, p.w, p.bias, p.out = (_lib.ptr(t) for t in (x, w, bias, out))
    p.M, p.N, p.K, p.x_stride_row, p.out_stride_row, p.groups, p.out_kind, p.eps = M, N, K, K, N, groups, out_kind, 1e-5
    if normed:
        p.sq, p.nsq = _lib.ptr(sq), groups * 3
    if out_kind == 2:
        p.next_weight, p.next_x, p.next_sq = _lib.ptr(next_w), _lib.ptr(nx), _lib.ptr(nsq)
    _lib.check(lib.m2_linear_small(p, _lib.stream_ptr()), "m2_linear_small")
    xd = x.double().cpu().view(M, groups, K // groups)
    if normed:
        xd = xd * torch.rsqrt(sq.double().cpu().view(M, groups, 3).sum(-1, keepdim=True) * groups / K + 1e-5)
    ref = xd.reshape(M, K) @ w.double().cpu().T + bias.double().cpu() + (base.double() if out_kind == 2 else 0)
    assert _rel(out, ref) < 5e-3
    if out_kind == 2:
        assert _rel(nx, ref * next_w.double().cpu()) < 5e-3 and _rel(nsq.sum(1), ref.pow(2).sum(1)) < 1e-3


@pytest.mark.parametrize("b,h,p,n,g,W,groups_norm", [(1, 8, 64, 128, 1, 4, True), (3, 6, 64, 64, 2, 3, True), (16, 4, 128, 64, 1, 4, False),
                                                     (17, 8, 128, 128, 8, 4, True), (5, 24, 64, 128, 8, 4, False), (33, 8, 64, 128, 1, 3, True)])
@pytest.mark.parametrize("block", [False, True])
def test_layer_step_against_oracle(b, h, p, n, g, W, groups_norm, block):
    from mamba2.configuration_mamba2 import Mamba2Config
    from mamba2.mamba2_mixer import Mamba2Cache
    from mamba2.modeling_mamba2 import Mamba2Block
    d, hidden = h * p, h * p // 2
    cfg = Mamba2Config(num_heads=h, head_dim=p, hidden_size=hidden, state_size=n, n_groups=g, num_hidden_layers=1, rmsnorm_within_groups=groups_norm)
    torch.manual_seed(b + h)
    blk = Mamba2Block(cfg, 0).bfloat16().to(DEV)
    cache = Mamba2Cache(cfg, b, dtype=torch.bfloat16, device=DEV, conv_width=W)
    for t in (cache.conv_states[0], cache.ssm_states[0]):
        t.normal_(0, 0.5)
    x = torch.randn(b, 1, hidden, device=DEV)
    m = blk.mixer
    f = lambda t: t.detach().double().cpu()
    xin = f(x) if block else f(x.bfloat16())
    u = f(blk.norm.weight) * xin * torch.rsqrt(xin.pow(2).mean(-1, keepdim=True) + blk.norm.variance_epsilon) if block else xin
    zx = u @ f(m.in_proj.weight).T
    cx = d + 2 * g * n
    y, cs, S = decode_step_ref(zx[..., d:d + cx], f(cache.conv_states[0]), f(m.conv1d.weight).squeeze(1), f(m.conv1d.bias), f(cache.ssm_states[0]),
                               softplus_ref(zx[..., d + cx:] + f(m.dt_bias)), -torch.exp(f(m.A_log)), f(m.D), n_groups=g)
    ref = rmsnorm_gated_ref(y, zx[..., :d], f(m.norm.weight), g if groups_norm else 1, m.norm.eps) @ f(m.out_proj.weight).T
    with torch.no_grad():
        got = blk.step(x, cache_params=cache) if block else m.step(x.bfloat16(), cache_params=cache)
    assert _rel(got, ref + xin if block else ref) < 2e-2
    assert _rel(cache.conv_states[0], cs) < 5e-3 and _rel(cache.ssm_states[0], S) < 1e-2
    # the same block inside a model's residual stream, chained into itself
    if block:
        from mamba2 import _lib
        c2, c3 = (Mamba2Cache(cfg, b, dtype=torch.bfloat16, device=DEV, conv_width=W) for _ in range(2))
        with torch.no_grad():
            stream = _lib.native().residual_stream(x)
            for _ in range(2):
                m._step(c2, stream=stream, block_norm=blk.norm, next_norm=blk.norm)
            got = _lib.native().stream_norm(stream, _lib.f32_param(blk.norm.weight), blk.norm.variance_epsilon, torch.bfloat16)
            want = blk.norm(blk.step(blk.step(x, cache_params=c3), cache_params=c3))
        assert _rel(got.view(b, 1, hidden), want.double().cpu()) < 1e-2
        assert _rel(c2.ssm_states[0], c3.ssm_states[0].double().cpu()) < 1e-2


# few rows kept in LDS beside the ring: padded to 1, 2 or 4, step counts that do not divide by the waves, one and several tiles per workgroup,
# and rows too long for that
@pytest.mark.parametrize("M,N,K,groups", [(1, 33, 128, 1), (2, 16, 64, 1), (3, 4100, 320, 1), (4, 20000, 256, 2), (3, 50, 1088, 1), (4, 40, 16384, 1), (1, 9000, 2560, 4)])
def test_linear_small_few_rows(M, N, K, groups):
    for normed, out_kind in ((False, 0), (True, 2)):
        test_linear_small(M, N, K, groups, normed, out_kind)


@pytest.mark.parametrize("W", [5, 8])
def test_layer_step_conv_widths(W):
    test_layer_step_against_oracle(3, 8, 64, 64, 1, W, True, False)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,channels,offset", [(1, 64, 0), (3, 1030, 0), (8, 1024, 0), (5, 2048, 1), (33, 7, 0)])      # offset: a table on no vector
def test_embed_rows(rows, channels, offset, dtype):
    from mamba2 import _lib
    lib, gen = _lib.load(), torch.Generator().manual_seed(channels)
    vocab = 11
    table = torch.randn(vocab * channels + offset, generator=gen).to(DEV, dtype)[offset:].view(vocab, channels)
    ids = torch.randint(0, vocab, (rows,), generator=gen)
    ids[0] = vocab                                  # outside the table
    ids, w = ids.to(DEV), torch.rand(channels, generator=gen).to(DEV) + 0.5
    res, x, sq = torch.empty(rows, channels, device=DEV), torch.empty(rows, channels, device=DEV, dtype=torch.bfloat16), torch.empty(rows, 1, device=DEV)
    rc = lib.m2_embed_rows(table.data_ptr(), _lib.M2_F32 if dtype == torch.float32 else _lib.M2_BF16, vocab, ids.data_ptr(), res.data_ptr(), w.data_ptr(),
                           x.data_ptr(), sq.data_ptr(), rows, channels, torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    assert res[0].isnan().all() and x[0].isnan().all() and sq[0].isnan().all()
    want = table[ids[1:]].float()
    assert torch.equal(res[1:], want) and torch.equal(x[1:], (want * w).bfloat16())
    # fp32 sums of `channels` squares in another order: at most channels roundings of 2^-24 each
    assert torch.allclose(sq[1:, 0], want.pow(2).sum(1), rtol=channels * 2.0 ** -24, atol=0.0)


def test_embed_rows_the_residual_alone():
    from mamba2 import _lib
    lib = _lib.load()
    table = torch.randn(7, 130, device=DEV)
    ids = torch.tensor([3, 7, 0], device=DEV)
    res = torch.empty(3, 130, device=DEV)
    args = (table.data_ptr(), _lib.M2_F32, 7, ids.data_ptr(), res.data_ptr())
    assert lib.m2_embed_rows(*args, None, None, None, 3, 130, torch.cuda.current_stream().cuda_stream) == 0
    assert torch.equal(res[[0, 2]], table[[3, 0]]) and res[1].isnan().all()
    assert lib.m2_embed_rows(*args, table.data_ptr(), None, None, 3, 130, None) == -6      # weight, x and sq together
