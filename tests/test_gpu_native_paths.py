"""GPU: calls that the native step and layer take or leave to the modules: parameters of other types and alignments, hooks and
overrides, a prefill that fails.  The reference is the same work block by block, module by module."""
import pytest
import torch

from conftest import rel_err

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _rel(got, ref):
    return ((got.double() - ref.double()).norm() / ref.double().norm()).item()


def _model(layers=2, dtype=torch.bfloat16, **kw):
    from mamba2.configuration_mamba2 import Mamba2Config
    from mamba2.modeling_mamba2 import Mamba2ForCausalLM
    cfg = Mamba2Config(num_heads=8, head_dim=64, hidden_size=256, state_size=64, n_groups=2, num_hidden_layers=layers, vocab_size=320, expand=2,
                       residual_in_fp32=True, **kw)
    torch.manual_seed(0)
    return cfg, Mamba2ForCausalLM(cfg).to(DEV).to(dtype).eval()


def _cache(cfg, b, dtype=torch.bfloat16, seed=1):
    from mamba2.mamba2_mixer import Mamba2Cache
    cache = Mamba2Cache(cfg, b, dtype=dtype, device=DEV)
    gen = torch.Generator(device=DEV).manual_seed(seed)
    for t in cache.conv_states + cache.ssm_states:
        t.normal_(0, 0.3, generator=gen)
    return cache


@torch.no_grad()
def _blockwise(m, ids, cache):
    x = m.backbone.embeddings(ids).float()
    for blk in m.backbone.layers:
        x = x + blk.mixer.step(blk.norm(x).to(blk.mixer.in_proj.weight.dtype), cache)
    return m.backbone.norm_f(x).double() @ m.lm_head.weight.double().T


@pytest.mark.parametrize("b", [5, 33])
@pytest.mark.parametrize("layers,head,table", [("bfloat16", "float32", "bfloat16"), ("float32", "bfloat16", "float32"), ("bfloat16", "float16", "bfloat16"),
                                               ("bfloat16", "bfloat16", "float16")])
def test_step_of_a_model_with_a_head_of_another_dtype(b, layers, head, table):
    cfg, m = _model(dtype=getattr(torch, layers))
    m.lm_head.to(getattr(torch, head))
    m.backbone.embeddings.to(getattr(torch, table))
    ids = torch.randint(0, cfg.vocab_size, (b, 1), generator=torch.Generator().manual_seed(2)).to(DEV)
    c1, c2 = (_cache(cfg, b, getattr(torch, layers)) for _ in range(2))
    for _ in range(2):
        with torch.no_grad():
            got = m.step(ids, c1)
        assert got.dtype == torch.float32 and _rel(got, _blockwise(m, ids, c2)) < 1e-2      # bf16 rows and layers
    assert _rel(c1.ssm_states[1], c2.ssm_states[1]) < 1e-2


@pytest.mark.parametrize("b", [5, 33])
def test_step_through_layers_of_two_dtypes(b):
    """What a bf16 layer leaves to be added in front of an fp32 one goes into the stream as it is."""
    from mamba2 import _lib
    cfg, m = _model()
    blocks = list(m.backbone.layers)
    blocks[1].float()
    c = _cache(cfg, b)
    c.conv_states[1] = c.conv_states[1].float()
    c2 = _cache(cfg, b)
    c2.conv_states[1] = c2.conv_states[1].float()
    x = torch.randn(b, 1, cfg.hidden_size, generator=torch.Generator().manual_seed(3)).to(DEV)
    with torch.no_grad():
        stream = _lib.native().residual_stream(x)
        for i, blk in enumerate(blocks):
            blk.mixer._step(c, stream=stream, block_norm=blk.norm)
        got = _lib.native().stream_sum(stream).view(x.shape)
        want = x
        for blk in blocks:
            want = want + blk.mixer.step(blk.norm(want).to(blk.mixer.in_proj.weight.dtype), c2)
    assert rel_err(got, want) < 1e-2


def _views_of_one_buffer(module, offset):
    """Every parameter a contiguous view into one flat buffer per dtype, `offset` elements off the allocation's alignment."""
    for dtype in {p.dtype for p in module.parameters()}:
        ps = [p for p in module.parameters() if p.dtype == dtype]
        flat = torch.empty(sum(p.numel() + 8 for p in ps) + offset, dtype=dtype, device=DEV)
        at = offset
        for p in ps:
            p.data = flat[at:at + p.numel()].copy_(p.detach().reshape(-1)).view(p.shape)
            at += -(-p.numel() // 8) * 8
    return module


@pytest.mark.parametrize("b", [3, 33])
@pytest.mark.parametrize("offset", [1, 4])
def test_weights_that_start_anywhere(b, offset):
    """Views into a flat buffer of parameters: contiguous, but on no 16-byte boundary."""
    cfg, m = _model()
    ids = torch.randint(0, cfg.vocab_size, (b, 1), generator=torch.Generator().manual_seed(2)).to(DEV)
    c1, c2, c3 = (_cache(cfg, b) for _ in range(3))
    with torch.no_grad():
        want = m.step(ids, c1)
        for block in m.backbone.layers:
            block.norm.float()
        _views_of_one_buffer(m, offset)
        assert m.lm_head.weight.data_ptr() % 16 and m.lm_head.weight.is_contiguous()
        got = m.step(ids, c2)
        x = m.backbone.embeddings(ids).float()
        block = m.backbone.layers[0]
        assert _rel(block.step(x, c3), x + block.mixer.step(block.norm(x).bfloat16(), _cache(cfg, b))) < 1e-2
    assert _rel(got, want) < 1e-2 and _rel(c2.ssm_states[1], c1.ssm_states[1]) < 1e-2
    assert torch.equal(c2.conv_states[0][..., :-1], c1.conv_states[0][..., :-1])


@pytest.mark.parametrize("b", [3, 33])
def test_layer_step_on_rows_of_any_stride(b):
    """The last token of a longer tensor, a column slice that starts anywhere, a transposed and an expanded one."""
    cfg, m = _model(1)
    mixer, d = m.backbone.layers[0].mixer, cfg.hidden_size
    gen = torch.Generator().manual_seed(4)
    x = torch.randn(b, 1, d, generator=gen).bfloat16().to(DEV)
    long, wide = torch.zeros(b, 7, d, dtype=x.dtype, device=DEV), torch.zeros(b, 1, d + 5, dtype=x.dtype, device=DEV)
    long[:, -1:], wide[..., 3:3 + d] = x, x
    far = torch.empty(b, (1 << 26) // d + 1, d, dtype=x.dtype, device=DEV)[:, -1:]      # rows more than 2^26 elements apart
    far.copy_(x)
    forms = {"last": long[:, -1:], "columns": wide[..., 3:3 + d], "transposed": x[:, 0].T.contiguous().T[:, None], "far": far}
    forms["expanded"] = x[:1].expand(b, 1, d)
    for name, form in forms.items():
        c1, c2 = (_cache(cfg, b) for _ in range(2))
        with torch.no_grad():
            want, got = mixer.step(form.contiguous(), c1), mixer.step(form, c2)
        # up to 32 rows one kernel takes them all; above, some forms go to the library's product, which sums in another order
        for a, e in ((got, want), (c2.ssm_states[0], c1.ssm_states[0])):
            assert torch.equal(a, e) if b <= 32 else _rel(a, e) < 1e-2, name


def test_tuned_step_lets_the_library_try_the_projections():
    """GraphedStep(tune_gemms=True) above 32 sequences: the projections' shapes are among those that TunableOp timed, and while it is
    off they run in this library's kernel (bit for bit the untuned step's logits)."""
    import torch.cuda.tunable as tunable
    from mamba2.modeling_mamba2 import GraphedStep
    cfg, m = _model()
    b = 56
    ids = torch.randint(0, cfg.vocab_size, (b, 1), generator=torch.Generator().manual_seed(2)).to(DEV)
    c1, c2, c3 = (_cache(cfg, b) for _ in range(3))
    with torch.no_grad():
        before = m.step(ids, c1)
    limits = tunable.get_max_tuning_duration(), tunable.get_max_tuning_iterations()
    try:
        tunable.set_max_tuning_duration(1)
        tunable.set_max_tuning_iterations(1)
        step = GraphedStep(m, c2, b, tune_gemms=True)
    finally:
        tunable.set_max_tuning_duration(limits[0])
        tunable.set_max_tuning_iterations(limits[1])
    shapes = " ".join(r[1] for r in tunable.get_results())
    mixer = m.backbone.layers[0].mixer
    for proj in (mixer.in_proj, mixer.out_proj):
        assert f"{proj.out_features}_{b}_{proj.in_features}" in shapes, shapes
    assert _rel(step(ids), before) < 1e-2
    with torch.no_grad():
        assert torch.equal(m.step(ids, c3), before)


def _hook(m, calls):
    m.register_forward_hook(lambda *_: calls.append(1))


def _replaced(m, calls):
    forward = m.forward

    def wrapper(*args, **kwargs):
        calls.append(1)
        return forward(*args, **kwargs)

    m.forward = wrapper


def _own_step(m, calls):
    class Other(type(m)):
        def step(self, *args, **kwargs):
            calls.append(1)
            return super().step(*args, **kwargs)

    m.__class__ = Other


@pytest.mark.parametrize("change,where", [(c, w) for c in (_hook, _replaced) for w in ("norm", "mixer.norm", "mixer.in_proj", "mixer.out_proj")]
                         + [(_own_step, "mixer"), (_own_step, "")])
def test_step_calls_what_a_user_put_there(change, where):
    """A hook, a replaced forward and a step of one's own run once per token, in a layer's, a block's and a model's step, and change
    nothing else."""
    cfg, m = _model()
    b = 3
    ids = torch.randint(0, cfg.vocab_size, (b, 1), generator=torch.Generator().manual_seed(2)).to(DEV)
    calls = []
    block = m.backbone.layers[1]
    with torch.no_grad():
        x = m.backbone.embeddings(ids)
        want = m.step(ids, _cache(cfg, b)), block.step(x.float(), _cache(cfg, b)), block.mixer.step(x, _cache(cfg, b))
        change(block.get_submodule(where), calls)
        got = m.step(ids, _cache(cfg, b)), block.step(x.float(), _cache(cfg, b))
        assert len(calls) == 2
        if where.startswith("mixer"):
            got += (block.mixer.step(x, _cache(cfg, b)),)
            assert len(calls) == 3
    for g, w in zip(got, want):
        assert _rel(g, w) < 1e-2


@pytest.mark.parametrize("change,where", [(_hook, "backbone.norm_f"), (_replaced, "backbone.norm_f"), (_hook, "lm_head"), (_replaced, "lm_head"), (_own_step, "backbone")])
def test_model_step_calls_what_a_user_put_there(change, where):
    cfg, m = _model()
    ids = torch.randint(0, cfg.vocab_size, (3, 1), generator=torch.Generator().manual_seed(2)).to(DEV)
    calls = []
    with torch.no_grad():
        want = m.step(ids, _cache(cfg, 3))
        change(m.get_submodule(where), calls)
        assert _rel(m.step(ids, _cache(cfg, 3)), want) < 1e-2 and len(calls) == 1


@pytest.mark.parametrize("change", [_hook, _replaced])
@pytest.mark.parametrize("where", ["in_proj", "out_proj"])
def test_forward_and_prefill_call_what_a_user_put_there(change, where):
    cfg, m = _model(1)
    mixer, calls = m.backbone.layers[0].mixer, []
    x = torch.randn(2, 40, cfg.hidden_size, generator=torch.Generator().manual_seed(5)).bfloat16().to(DEV)

    def passes():
        out = mixer(x)
        grad, = torch.autograd.grad(out.float().pow(2).sum(), mixer.A_log)
        with torch.no_grad():
            return out.detach(), grad, mixer(x, cache_params=_cache(cfg, 2))

    want = passes()
    change(mixer.get_submodule(where), calls)
    for g, w in zip(passes(), want):
        assert _rel(g, w) < 2e-2
    assert len(calls) == 2


def test_model_of_other_blocks_is_stepped_through_their_own_step():
    class Own(torch.nn.Module):
        def __init__(self, inner):
            super().__init__()
            self.inner = inner

        def step(self, *args, **kwargs):
            return self.inner.step(*args, **kwargs)

    cfg, m = _model()
    ids = torch.randint(0, cfg.vocab_size, (3, 1), generator=torch.Generator().manual_seed(2)).to(DEV)
    with torch.no_grad():
        want = m.step(ids, _cache(cfg, 3))
        m.backbone.layers[0].mixer = Own(m.backbone.layers[0].mixer)
        m.backbone.layers[0].mixer.in_proj = m.backbone.layers[0].mixer.inner.in_proj      # whose dtype the block's norm is cast to
        m.backbone.layers[1] = Own(m.backbone.layers[1])
        m.backbone.layers[0].mixer.inner.norm.register_forward_hook(lambda *_: None)
        assert _rel(m.step(ids, _cache(cfg, 3)), want) < 1e-2


@pytest.mark.parametrize("types", [(torch.float64, torch.float16, torch.float64, torch.float16), (torch.float16, torch.float32, torch.bfloat16, torch.float64)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_layer_takes_small_parameters_of_any_type(types, dtype):
    """A_log, D, dt_bias and the norm's weight in types that the casting kernel does not read: as the modules one by one take them."""
    cfg, m = _model(1, dtype)
    mixer = m.backbone.layers[0].mixer
    for owner, name, t in zip((mixer, mixer, mixer, mixer.norm), ("A_log", "D", "dt_bias", "weight"), types):
        setattr(owner, name, torch.nn.Parameter(getattr(owner, name).detach().to(t)))
    x = torch.randn(2, 140, cfg.hidden_size, generator=torch.Generator().manual_seed(5)).to(dtype).to(DEV)

    def passes():
        mixer.zero_grad()
        out = mixer(x)
        out.float().pow(2).sum().backward()
        return out.detach(), {k: p.grad.clone() for k, p in mixer.named_parameters()}

    got = passes()
    _hook(mixer.in_proj, [])          # the same layer, module by module
    want = passes()
    bar = 1e-2 if dtype == torch.bfloat16 else 2e-3          # fp16 gradients of the small parameters: 2^-11 each
    assert _rel(got[0], want[0]) < bar
    for k, p in mixer.named_parameters():
        assert got[1][k].dtype == p.dtype and _rel(got[1][k], want[1][k]) < bar, k


@pytest.mark.parametrize("continuing", [False, True])
@pytest.mark.parametrize("h,head_dim,n,message", [(4, 32, 64, "headdim"), (4, 64, 32, "dstate"), (136, 64, 64, "8192")])
def test_prefill_that_is_refused_leaves_the_cache(continuing, h, head_dim, n, message):
    """Heads or states that the scan does not take, a group wider than the norm takes: neither state has moved."""
    from mamba2.fused_kernel import mamba2_fused_prefill
    d, g, b, l = h * head_dim, 1, 2, 40
    cx = d + 2 * g * n
    gen = torch.Generator(device=DEV).manual_seed(6)
    rand = lambda *s: torch.randn(*s, device=DEV, generator=gen)
    conv_state, ssm_state = rand(b, cx, 4).bfloat16(), rand(b, h, head_dim, n)
    before = conv_state.clone(), ssm_state.clone()
    with pytest.raises(ValueError, match=message):
        mamba2_fused_prefill(rand(b, l, d + cx + h).bfloat16(), -torch.ones(h, device=DEV), torch.ones(h, device=DEV), rand(cx, 1, 4).bfloat16(),
                             rand(cx).bfloat16(), rand(h), torch.ones(d, device=DEV), g, n, d, head_dim, conv_state, ssm_state, continuing=continuing)
    assert torch.equal(conv_state, before[0]) and torch.equal(ssm_state, before[1])


@pytest.mark.parametrize("b", [3, 33])
def test_biases_that_broadcast_and_biases_that_do_not_fit(b):
    """A bias of one value is added to every output, as nn.Linear does; one of another length or on the host is an error."""
    cfg, m = _model(1, use_bias=True)
    mixer = m.backbone.layers[0].mixer
    x = torch.randn(b, 1, cfg.hidden_size, generator=torch.Generator().manual_seed(4)).bfloat16().to(DEV)
    long = torch.randn(2, 20, cfg.hidden_size, generator=torch.Generator().manual_seed(5)).bfloat16().to(DEV)

    def passes():
        with torch.no_grad():
            return mixer.step(x, _cache(cfg, b)), mixer(long), mixer(long, cache_params=_cache(cfg, 2)), m.lm_head(x)

    full = {}
    for p in (mixer.in_proj, mixer.out_proj):
        p.bias = torch.nn.Parameter(torch.full((1,), 0.25, dtype=torch.bfloat16, device=DEV))
        full[p] = torch.nn.Parameter(p.bias.detach().repeat(p.out_features))
    got = passes()
    for p, bias in full.items():
        p.bias = bias
    for g, w in zip(got, passes()):
        assert _rel(g, w) < 1e-2
    for bias in (torch.zeros(mixer.out_proj.out_features - 1, dtype=torch.bfloat16, device=DEV), torch.zeros(mixer.out_proj.out_features, dtype=torch.bfloat16)):
        mixer.out_proj.bias = torch.nn.Parameter(bias)
        for call in (lambda: mixer.step(x, _cache(cfg, b)), lambda: mixer(long), lambda: mixer(long, cache_params=_cache(cfg, 2))):
            with torch.no_grad(), pytest.raises(RuntimeError):
                call()
    mixer.out_proj.bias = full[mixer.out_proj]
    for bias in (torch.zeros(8, dtype=torch.bfloat16, device=DEV), torch.zeros(mixer.conv_dim, device=DEV)):
        mixer.conv1d.bias = torch.nn.Parameter(bias)
        with torch.no_grad(), pytest.raises(ValueError, match="conv bias"):
            mixer.step(x, _cache(cfg, b))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("b", [3, 33])
def test_layer_takes_parameters_that_are_strided_views(b, dtype):
    """Every parameter a view with a stride of two into a wider one: step, training pass and prefill as with parameters of their own."""
    cfg, m = _model(1, dtype)
    mixer = m.backbone.layers[0].mixer
    x = torch.randn(b, 1, cfg.hidden_size, generator=torch.Generator().manual_seed(4)).to(dtype).to(DEV)
    long = torch.randn(2, 40, cfg.hidden_size, generator=torch.Generator().manual_seed(5)).to(dtype).to(DEV)

    def passes():
        out = mixer(long)
        grads = torch.autograd.grad(out.float().pow(2).sum(), list(mixer.parameters()))
        with torch.no_grad():
            return [mixer.step(x, _cache(cfg, b, dtype)), mixer(long, cache_params=_cache(cfg, 2, dtype)), out.detach(), *grads]

    want = passes()
    for owner in (mixer, mixer.conv1d, mixer.norm, mixer.in_proj, mixer.out_proj):
        for name, p in list(owner._parameters.items()):
            if p is not None:
                wide = torch.stack((p.detach(), torch.full_like(p, float("nan"))), dim=-1)
                setattr(owner, name, torch.nn.Parameter(wide[..., 0]))
    assert not mixer.D.is_contiguous() and not mixer.in_proj.weight.is_contiguous()
    for g, w in zip(passes(), want):
        assert _rel(g, w) < 2e-2


def _one_token(x, layout):
    """x (b, 1, width), its values in another layout; every row lies inside the tensor's own memory."""
    b, _, width = x.shape
    if layout == "time first":
        form = torch.empty(1, b, width, dtype=x.dtype, device=DEV).copy_(x.transpose(0, 1)).transpose(0, 1)
        assert form.is_contiguous() and form.stride() == (width, b * width, 1)
    elif layout == "last of five":
        form = x.repeat(1, 5, 1)[:, -1:]
    else:
        form = torch.cat([x, x], 2)[..., :width]
    return form


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("b,h", [(1, 8), (2, 8), (5, 8), (3, 5)])      # rows on 16 bytes and (5 heads) rows that are not
@pytest.mark.parametrize("layout", ["time first", "last of five", "padded"])
def test_core_on_one_token_of_any_layout(layout, b, h, dtype):
    """The stride of the token dimension says nothing where that has one entry: forward, backward and prefill, bit for bit as on
    contiguous rows."""
    from mamba2.fused_kernel import mamba2_fused_kernel, mamba2_fused_kernel_with_caching, mamba2_fused_prefill
    p, n, g = 64, 64, 1
    d, c = h * p, h * p + 2 * g * n
    gen = torch.Generator(device=DEV).manual_seed(7)
    rand = lambda *s: torch.randn(*s, device=DEV, generator=gen)
    x, dy = rand(b, 1, d + c + h).to(dtype), rand(b, 1, d).to(dtype)
    params = [-rand(h).abs(), rand(h), rand(c, 1, 4).to(dtype), rand(c).to(dtype), rand(h), rand(d)]
    states = rand(b, c, 4).to(dtype), rand(b, h, p, n)

    def passes(form):
        out = []
        for core in (mamba2_fused_kernel, mamba2_fused_kernel_with_caching):
            leaves = [t.detach().requires_grad_(True) for t in (form, *params)]
            y = core(*leaves, g, n, d, p)
            out += [y.detach(), *torch.autograd.grad(y, leaves, dy)]
        for continuing in (False, True):
            moved = [t.clone() for t in states]
            with torch.no_grad():
                out += [mamba2_fused_prefill(form, *params, g, n, d, p, *moved, continuing=continuing), *moved]
        return out

    for got, want in zip(passes(_one_token(x, layout)), passes(x)):
        assert torch.equal(got, want)
