"""The work that users of this package have it do, as cases that can be timed and compared: training (the scan, the conv, the
fused mixer core and a whole mixer layer, forward and backward), prefill (a prompt into the decode cache) and decode (one
layer's operator, one layer's step, a whole model's captured step).  Every case goes through the public entry points.

``listed()`` names the cases, ``draw(rng)`` gives others of the same ranges, ``prepare(case, seed)`` makes what a program holds
before the call, ``run(state)`` is one pass, ``work(case)`` the bytes and operations a pass cannot do without and
``tolerance(case)`` how far another correct implementation at the same precision may be off.
"""
import math
import os
import sys

import torch

_PACKAGE = os.path.join(os.getcwd(), "state-space-models-neuron_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(1, _PACKAGE)

from mamba2.configuration_mamba2 import Mamba2Config  # noqa: E402
from mamba2.conv1d_grouped import nki_conv1d  # noqa: E402
from mamba2.fused_kernel import mamba2_fused_kernel, mamba2_fused_kernel_with_caching, mamba2_fused_prefill  # noqa: E402
from mamba2.mamba2_kernel import mamba2_kernel  # noqa: E402
from mamba2.mamba2_kernel_inference import mamba2_kernel_inference  # noqa: E402
from mamba2.mamba2_mixer import Mamba2Cache, Mamba2Mixer  # noqa: E402
from mamba2.modeling_mamba2 import GraphedStep, Mamba2ForCausalLM  # noqa: E402

DEV = "cuda:0"
DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}
CONV_K = 4
CHUNK = 128


def _ssd(b, l, h, p, n, g, dtype):
    return {"path": "ssd", "b": b, "l": l, "h": h, "p": p, "n": n, "g": g, "dtype": dtype}


def _conv(b, l, c, channels_last, dtype):
    return {"path": "conv", "b": b, "l": l, "c": c, "channels_last": channels_last, "dtype": dtype}


def _core(b, l, h, p, n, g, caching, dtype):
    return {"path": "core", "b": b, "l": l, "h": h, "p": p, "n": n, "g": g, "caching": caching, "dtype": dtype}


def _layer(b, l, h, p, n, g):
    return {"path": "layer", "b": b, "l": l, "h": h, "p": p, "n": n, "g": g, "dtype": "bf16"}


def _prefill(b, l, h, p, n, g, projections, continuing):
    return {"path": "prefill", "b": b, "l": l, "h": h, "p": p, "n": n, "g": g, "projections": projections, "continuing": continuing,
            "dtype": "bf16"}


def _decode(b, h, p, n, g, width, dtype):
    return {"path": "decode", "b": b, "h": h, "p": p, "n": n, "g": g, "width": width, "dtype": dtype}


def _step(b, h, p, n, g):
    return {"path": "step", "b": b, "h": h, "p": p, "n": n, "g": g, "width": 4, "dtype": "bf16"}


def _model(b, h, p, n, g, layers, vocab):
    return {"path": "model", "b": b, "h": h, "p": p, "n": n, "g": g, "width": 4, "layers": layers, "vocab": vocab, "dtype": "bf16"}


def listed():
    def named(name, case):
        return dict(case, name=name)

    return [
        # the scan operator in training at the 2.7B layer's shape, one full batch: what a caller with a mixer of its own uses
        named("ssd-train-2.7B", _ssd(4, 2048, 80, 64, 128, 1, "bf16")),
        # the same in fp32 with wide heads and eight groups: the 370M layer of the integration test, as one debugs or fine-tunes it
        named("ssd-train-370M-fp32", _ssd(3, 2048, 16, 128, 128, 8, "fp32")),
        # the conv operator in its default (batch, channels, length) layout, training, 2.7B width
        named("conv-train-2.7B-bcl", _conv(4, 2048, 5376, False, "bf16")),
        # the fused mixer core in training at the 7B layer's shape, activations kept: the largest case
        named("core-train-7B", _core(2, 4096, 128, 64, 128, 8, True, "bf16")),
        # the fused core with recompute on a smaller layer and sequences that are no multiple of the chunk
        named("core-train-recompute-ragged", _core(3, 1111, 32, 64, 128, 1, False, "bf16")),
        # a whole small mixer layer in training on one short sequence: launches and host work count
        named("layer-train-small", _layer(1, 500, 24, 64, 128, 1)),
        # a short prompt through one 2.7B layer into the decode cache: time to the first token
        named("prefill-prompt-200", _prefill(1, 200, 80, 64, 128, 1, True, False)),
        # one long document through the core at the 2.7B width: a single sequence, many chunks
        named("prefill-core-16k", _prefill(1, 16384, 80, 64, 128, 1, False, False)),
        # prompts taken up in pieces behind a cached prefix, a batch of them
        named("prefill-core-continue", _prefill(8, 333, 80, 64, 128, 1, False, True)),
        # the decode operator of one 2.7B layer at a serving batch
        named("decode-op-b128", _decode(128, 80, 64, 128, 1, 3, "bf16")),
        # one layer's decode step for a single user, called eagerly: the smallest call
        named("decode-layer-b1", _step(1, 80, 64, 128, 1)),
        # token by token through a whole small model as one captured step, a few users
        named("decode-model-b8", _model(8, 32, 64, 128, 1, 24, 32768)),
    ]


def _log(rng, lo, hi):
    """A whole number from lo to hi, spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _dims(rng, lo, hi, by=1):
    """(heads, head width, state size, groups): heads from lo to hi channels of 64, in the multiples that the groups need, and
    of `by` (the heads of a whole layer come in eights, as in every configuration; the operators take any number)."""
    g = rng.choice((1, 1, 1, 2, 8))
    p = rng.choice((64, 64, 64, 128))
    n = rng.choice((128, 128, 64))
    by = max(by, g)
    h = max(1, _log(rng, lo, hi) * 64 // p // by) * by
    return h, p, n, g


def _batch_len(rng, per_token, most, lmin, lmax, bmax=16):
    """A batch and a length whose tokens, at per_token channels each, stay within `most` values."""
    l = _log(rng, lmin, max(lmin, min(lmax, most // per_token)))
    return _log(rng, 1, max(1, min(bmax, most // (per_token * l)))), l


def draw(rng):
    path = rng.choice(("ssd", "conv", "core", "layer", "prefill", "prefill", "decode", "step", "model"))
    dtype = rng.choice(("bf16", "bf16", "fp32"))
    if path == "ssd":
        h, p, n, g = _dims(rng, 8, 128)
        b, l = _batch_len(rng, h * p, 4 * 2048 * 5120 if dtype == "bf16" else 3 * 2048 * 2048, 64, 8192)
        return _ssd(b, l, h, p, n, g, dtype)
    if path == "conv":
        c = 8 * _log(rng, 32, 1280) + rng.choice((0, 0, 0, 4, 1))
        b, l = _batch_len(rng, c, 4 * 2048 * 5376 // (1 if dtype == "bf16" else 2), 16, 8192)
        return _conv(b, l, c, rng.random() < 0.5, dtype)
    if path == "core":
        h, p, n, g = _dims(rng, 8, 128)
        b, l = _batch_len(rng, h * p, 2 * 4096 * 8192 if dtype == "bf16" else 3 * 2048 * 2048, 64, 8192)
        return _core(b, l, h, p, n, g, rng.random() < 0.7, dtype)
    if path == "layer":
        h, p, n, g = _dims(rng, 8, 64, 8)
        b, l = _batch_len(rng, h * p, 2048 * 1792, 32, 2048)
        return _layer(b, l, h, p, n, g)
    if path == "prefill":
        projections = rng.random() < 0.5
        h, p, n, g = _dims(rng, 8, 96, 8 if projections else 1)
        b, l = _batch_len(rng, h * p, 1024 * 5120 if projections else 16384 * 5120, 5, 1024 if projections else 16384)
        return _prefill(b, l, h, p, n, g, projections, rng.random() < 0.4)
    if path == "decode":
        h, p, n, g = _dims(rng, 8, 128)
        return _decode(_log(rng, 1, max(1, min(256, 128 * 80 * 64 // (h * p)))), h, p, n, g, rng.choice((3, 4)), dtype)
    h, p, n, g = _dims(rng, 8, 80, 8)
    if path == "step":
        return _step(_log(rng, 1, 64), h, p, n, g)
    h, p, n, g = _dims(rng, 8, 32, 8)
    return _model(_log(rng, 1, 32), h, p, n, g, rng.randint(4, 24), 8 * rng.randint(1000, 4096))


# ------------------------------------------------------------------------------------------------ what a program holds
def _decay(h, gen):
    """A as trained layers have it: -exp(U(log 1, log 16))."""
    return -torch.exp(torch.empty(h, device=DEV).uniform_(0.0, math.log(16.0), generator=gen))


def _dt_bias(h, gen):
    """The inverse softplus of step sizes log-uniform in [1e-3, 1e-1], as the layers are initialised."""
    dt = torch.exp(torch.empty(h, device=DEV).uniform_(math.log(1e-3), math.log(1e-1), generator=gen))
    return dt + torch.log(-torch.expm1(-dt))


def _randn(gen, *shape):
    return torch.randn(*shape, device=DEV, generator=gen)


def _half(gen, *shape):
    return torch.rand(*shape, device=DEV, generator=gen) - 0.5


def _packed(case, l, gen):
    """[z | x | B | C | dt] as the input projection leaves it."""
    h, p, n, g = (case[k] for k in "hpng")
    d = h * p
    zx = _randn(gen, case["b"], l, 2 * d + 2 * g * n + h)
    zx[..., 2 * d:2 * d + 2 * g * n] /= math.sqrt(n)
    return zx.to(DTYPES[case["dtype"]])


def _core_params(case, gen):
    h, p, n, g = (case[k] for k in "hpng")
    d = h * p
    t = DTYPES[case["dtype"]]
    return [_decay(h, gen), torch.ones(h, device=DEV), _half(gen, d + 2 * g * n, 1, CONV_K).to(t), _half(gen, d + 2 * g * n).to(t),
            _dt_bias(h, gen), 1 + 0.1 * _randn(gen, d)]


def _config(case, layers=1, vocab=64):
    h, p, n, g = (case[k] for k in "hpng")
    return Mamba2Config(num_heads=h, head_dim=p, hidden_size=h * p // 2, state_size=n, n_groups=g, num_hidden_layers=layers, expand=2,
                        vocab_size=vocab)


def _trained(mixer, gen):
    """The decay, step and conv values of a trained layer in place of the constructor's."""
    with torch.no_grad():
        mixer.A_log.copy_(torch.log(-_decay(mixer.num_heads, gen)))
        mixer.dt_bias.copy_(_dt_bias(mixer.num_heads, gen))
        mixer.norm.weight.add_(0.1 * _randn(gen, mixer.intermediate_size))
        mixer.in_proj.weight.normal_(0.0, 0.02, generator=gen)
        mixer.out_proj.weight.normal_(0.0, 0.02, generator=gen)


def _mixer(case, gen):
    with torch.device(DEV):
        mixer = Mamba2Mixer(_config(case), 0)
    with torch.no_grad():
        mixer.conv1d.weight.copy_(_half(gen, *mixer.conv1d.weight.shape))
        mixer.conv1d.bias.copy_(_half(gen, *mixer.conv1d.bias.shape))
    _trained(mixer, gen)
    return mixer.to(DTYPES[case["dtype"]])


def _cache(case, gen, layers=1, width=CONV_K):
    """A decode cache in mid-sequence."""
    cache = Mamba2Cache(_config(case, layers), case["b"], dtype=DTYPES[case["dtype"]], device=DEV, conv_width=width)
    for conv, ssm in zip(cache.conv_states, cache.ssm_states):
        conv.copy_(_randn(gen, *conv.shape))
        ssm.copy_(0.1 * _randn(gen, *ssm.shape))
    return cache


def prepare(case, seed):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    path, b, t = case["path"], case["b"], DTYPES[case["dtype"]]
    s = {"case": case}
    if path == "ssd":
        l, h, p, n, g = (case[k] for k in "lhpng")
        dt = torch.exp(torch.empty(b, l, h, device=DEV).uniform_(math.log(1e-3), math.log(1e-1), generator=gen)).to(t)
        s["leaves"] = [dt, _decay(h, gen), _randn(gen, b, l, h, p).to(t), (_randn(gen, b, l, g, n) / math.sqrt(n)).to(t),
                       (_randn(gen, b, l, g, n) / math.sqrt(n)).to(t), torch.ones(h, device=DEV)]
        s["dout"] = _randn(gen, b, l, h, p).to(t)
    elif path == "conv":
        l, c = case["l"], case["c"]
        shape = (b, l, c) if case["channels_last"] else (b, c, l)
        s["leaves"] = [_randn(gen, *shape).to(t), _half(gen, c, 1, CONV_K).to(t), _half(gen, c).to(t)]
        s["dout"] = _randn(gen, *shape).to(t)
    elif path == "core":
        s["leaves"] = [_packed(case, case["l"], gen)] + _core_params(case, gen)
        s["dout"] = _randn(gen, b, case["l"], case["h"] * case["p"]).to(t)
    elif path == "layer":
        s["mixer"] = _mixer(case, gen)
        hidden = _randn(gen, b, case["l"], s["mixer"].hidden_size).to(t)
        s["leaves"] = [hidden] + list(s["mixer"].parameters())
        s["dout"] = _randn(gen, *hidden.shape).to(t)
    elif path == "prefill":
        s["cache"] = _cache(case, gen)
        s["cache"].seqlen_offset = 64 if case["continuing"] else 0
        if case["projections"]:
            s["mixer"] = _mixer(case, gen)
            s["hidden"] = _randn(gen, b, case["l"], s["mixer"].hidden_size).to(t)
        else:
            s["packed"], s["params"] = _packed(case, case["l"], gen), _core_params(case, gen)
    elif path == "decode":
        h, p, n, g = (case[k] for k in "hpng")
        c = h * p + 2 * g * n
        xBC = _randn(gen, b, 1, c)
        xBC[..., h * p:] /= math.sqrt(n)
        dt = torch.exp(torch.empty(b, 1, h, device=DEV).uniform_(math.log(1e-3), math.log(1e-1), generator=gen)).to(t)
        s["args"] = [xBC.to(t), _randn(gen, b, c, case["width"]).to(t), _half(gen, c, CONV_K).to(t), _half(gen, c).to(t),
                     0.1 * _randn(gen, b, h, p, n), dt, _decay(h, gen), torch.ones(h, device=DEV), g]
    elif path == "step":
        s["mixer"], s["cache"] = _mixer(case, gen), _cache(case, gen, width=case["width"])
        s["hidden"] = _randn(gen, b, 1, s["mixer"].hidden_size).to(t)
    else:
        config = _config(case, case["layers"], case["vocab"])
        torch.manual_seed(seed)
        with torch.device(DEV):
            model = Mamba2ForCausalLM(config)
        for block in model.backbone.layers:
            _trained(block.mixer, gen)
        model = model.to(t).eval()
        s["cache"] = _cache(case, gen, case["layers"], case["width"])
        s["step"] = GraphedStep(model, s["cache"], b)
        s["ids"] = torch.randint(0, case["vocab"], (b, 1), device=DEV, generator=gen)
    for leaf in s.get("leaves", ()):
        leaf.requires_grad_(True)
    return s


# --------------------------------------------------------------------------------------------------------------- a pass
def run(state):
    case = state["case"]
    path = case["path"]
    if path in ("ssd", "conv", "core", "layer"):
        leaves = state["leaves"]
        if path == "ssd":
            out = mamba2_kernel(*leaves)
        elif path == "conv":
            out = nki_conv1d(*leaves, activation="silu", channels_last=case["channels_last"])
        elif path == "core":
            core = mamba2_fused_kernel_with_caching if case["caching"] else mamba2_fused_kernel
            out = core(*leaves, case["g"], case["n"], case["h"] * case["p"], case["p"])
        else:
            out = state["mixer"](leaves[0])
        return [out.detach(), *torch.autograd.grad(out, leaves, state["dout"])]
    with torch.no_grad():
        if path == "decode":
            return mamba2_kernel_inference(*state["args"])
        if path == "model":
            return [state["step"](state["ids"]), *state["cache"].conv_states, *state["cache"].ssm_states]
        cache = state["cache"]
        if path == "step":
            out = state["mixer"].step(state["hidden"], cache)
        elif case["projections"]:
            out = state["mixer"](state["hidden"], cache_params=cache)
        else:
            out = mamba2_fused_prefill(state["packed"], *state["params"], case["g"], case["n"], case["h"] * case["p"], case["p"],
                                       cache.conv_states[0], cache.ssm_states[0], continuing=case["continuing"])
        return [out, cache.conv_states[0], cache.ssm_states[0]]


# ------------------------------------------------------------------------------------------- what a pass cannot do without
def _scan_flops(case, tokens):
    """The chunked scan, forward: per token and head the causal half of the chunk's products with x, the state's build-up and
    its reading; per token and group the causal half of C B^T."""
    h, p, n, g = (case[k] for k in "hpng")
    q = min(CHUNK, case["l"])
    return tokens * (h * (q * p + 4 * n * p) + g * q * n)


def work(case):
    path, b, e = case["path"], case["b"], 4 if case["dtype"] == "fp32" else 2
    if path == "conv":
        tokens, c = b * case["l"], case["c"]
        # read x, dy and write y, dx; two passes of k multiply-adds, and one for the weights' gradient
        return {"bytes": e * (4 * tokens * c + 2 * c * (CONV_K + 1)), "flops": 3 * 2 * CONV_K * tokens * c}
    h, p, n, g = (case[k] for k in "hpng")
    d, gn = h * p, g * n
    conv_dim = d + 2 * gn
    packed, hidden = d + conv_dim + h, d // 2
    small = e * conv_dim * (CONV_K + 1) + 4 * (3 * h + d)
    if path in ("ssd", "core", "layer", "prefill"):
        tokens, scan = b * case["l"], _scan_flops(case, b * case["l"])
    if path == "ssd":
        # read x, B, C, dt, dy; write y and the gradients of x, B, C, dt
        return {"bytes": e * tokens * (4 * d + 4 * gn + 2 * h) + 16 * h, "flops": 3 * scan}
    if path == "core":
        return {"bytes": e * tokens * (2 * packed + 2 * d) + 2 * small, "flops": 3 * (scan + 2 * CONV_K * tokens * conv_dim + 8 * tokens * d)}
    projections = hidden * packed + d * hidden
    if path == "layer":
        return {"bytes": e * (4 * tokens * hidden + 2 * projections) + 2 * small,
                "flops": 3 * (2 * tokens * projections + scan + 2 * CONV_K * tokens * conv_dim + 8 * tokens * d)}
    if path == "prefill":
        states = b * (4 * d * n + e * CONV_K * conv_dim) * (2 if case["continuing"] else 1)
        inner = scan + 2 * CONV_K * tokens * conv_dim + 8 * tokens * d
        if case["projections"]:
            return {"bytes": e * (2 * tokens * hidden + projections) + states + small, "flops": inner + 2 * tokens * projections}
        return {"bytes": e * tokens * (packed + d) + states + small, "flops": inner}
    # one token: every state is read and written, every weight read
    states, token = 2 * b * (4 * d * n + e * case["width"] * conv_dim), b * (6 * d * n + 2 * CONV_K * conv_dim)
    if path == "decode":
        return {"bytes": states + e * b * (conv_dim + h + d) + small, "flops": token}
    if path == "step":
        return {"bytes": states + e * (2 * b * hidden + projections) + small, "flops": token + 2 * b * projections}
    layers, head = case["layers"], hidden * case["vocab"]
    return {"bytes": layers * (states + e * projections + small) + e * head + b * (4 * case["vocab"] + e * hidden),
            "flops": layers * (token + 2 * b * projections) + 2 * b * head}


def tolerance(case):
    if case["dtype"] == "fp32":
        return {"rel": 2e-5}        # 32-bit products and sums over thousands of terms
    if case["path"] in ("layer", "model"):
        return {"rel": 2e-2}        # a chain of bf16 tensors, each rounded where it is handed over
    return {"rel": 1e-2}            # bf16 results of bf16 operands
