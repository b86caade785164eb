"""Timed workloads of the analog SigmaMoE layer: what a program that trains or serves it asks of this package.

A case names a layer (d_model D, experts E, expert size F, heads k), a token count T, the element type and the analog
options; it either runs the whole layer at inference (router, top-k, expert feed-forward) or one training step of it
(forward, backward and, where the case says so, the weight clip that follows the optimizer).  The layer, its weights and
the batch are in GPU memory before a pass, as in a training loop or a serving process.

Every training step returns its output and all gradients.  The output noise of a training forward is drawn in the
kernels from the layer's own step counter, which starts at zero in every new state.
"""
import math
import random

import torch

from analog_moe_amd import config as rpu
from analog_moe_amd.moe_layer import AnalogSigmaMoELayer, AnalogSigmaMoELayerAIHWKIT

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}

# What a case says, and what it means if it does not say it.
DEFAULTS = dict(
    train=True,           # a training step; False: inference under no_grad, in eval mode
    router=False,         # the pass starts at layer(x), router included; False: the routing decision is given
    routing="router",     # how a given decision is drawn: "router" (sigmoid top-k of a random projection),
                          # "even" (experts loaded T*k/E +- a few percent), "zipf" (load follows Zipf(1.2))
    mis=-1,               # max_input_size: K-tiles of at most this many features, -1: one tile
    adc=True,             # 8-bit output quantiser, bound 12
    noise=0.04,           # output noise of a training forward, in units of max |W|
    modifier="NONE",      # weight modifier of a training forward
    clip=False,           # Gaussian weight clip after the backward pass
    flavour="plain",      # "plain": the fused layer; "bias": with expert and output biases (the layer is then composed
                          # of single projections); "abs_max": the other flavour, rows scaled by their abs-max and noise
                          # per channel
)


def _case(name, T, D, E, F, k, dtype, **options):
    return dict(DEFAULTS, name=name, T=T, D=D, E=E, F=F, k=k, dtype=dtype, **options)


def listed():
    return [
        # one sequence generating: the smallest call, launches and host time
        _case("decode_1_bf16", 1, 1024, 64, 256, 8, "bf16", train=False, router=True),
        # a batch of sequences generating together
        _case("decode_48_bf16", 48, 1024, 64, 256, 8, "bf16", train=False, router=True),
        # a prompt of odd length through a layer with two analog tiles per column
        _case("prefill_1717_bf16", 1717, 1024, 64, 256, 8, "bf16", train=False, router=True, mis=512),
        # evaluating the small language model in single precision
        _case("eval_2048_f32", 2048, 412, 16, 128, 4, "f32", train=False, router=True),
        # a unit-test sized training step: latency
        _case("train_tiny_f32", 256, 128, 8, 64, 2, "f32", noise=0.0),
        # the small language model (rows of 412 elements: no multiple of a vector or a K step), both precisions
        _case("train_412_bf16", 8192, 412, 16, 128, 4, "bf16"),
        _case("train_412_f32", 8192, 412, 16, 128, 4, "f32"),
        # the 64-expert layer with two analog tiles per column, the benchmark's default workload with a router's spread
        _case("train_64e_bf16", 16384, 1024, 64, 256, 8, "bf16", mis=512, routing="even"),
        # 128 experts under a skewed load: the largest call
        _case("train_128e_zipf_bf16", 32768, 2048, 128, 512, 4, "bf16", routing="zipf"),
        # the whole hardware-aware step of a decoder's layer: router, weight modifier, noise, weight clip
        _case("train_hwa_f16", 4096, 1024, 64, 256, 8, "f16", router=True,
              modifier="DISCRETIZE_ADD_NORMAL_PER_CHANNEL", clip=True),
        # layers the fused path does not take
        _case("train_bias_bf16", 3000, 512, 32, 128, 4, "bf16", flavour="bias"),
        _case("train_absmax_f32", 1500, 512, 32, 128, 4, "f32", flavour="abs_max", adc=False),
    ]


def _spread(rng: random.Random, lo: int, hi: int) -> int:
    """An integer of [lo, hi], its logarithm evenly spread."""
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def draw(rng: random.Random):
    train = rng.random() < 0.6
    dtype = rng.choice(("bf16", "bf16", "f16", "f32"))
    # model sizes: mostly multiples of 64, now and then only of 4 (such as 412)
    step_d, step_f = rng.choice((64, 64, 4)), rng.choice((64, 64, 16))
    D = max(128, _spread(rng, 128, 2048) // step_d * step_d)
    F = max(64, _spread(rng, 64, 512) // step_f * step_f)
    E, k = rng.choice((8, 16, 32, 64, 128)), rng.choice((1, 2, 4, 8))
    T = _spread(rng, 64, 32768) if train else _spread(rng, 1, 8192)
    # no more work than the largest listed case; single precision has a sixteenth of the matrix rate
    most = 131072 * 2048 * 512 // (16 if dtype == "f32" else 1)
    T = max(1, min(T, most // (k * D * F), 131072 * 2048 // (k * D)))
    c = dict(DEFAULTS, T=T, D=D, E=E, F=F, k=k, dtype=dtype, train=train)
    c["mis"] = rng.choice((-1, -1, 512))
    c["adc"] = rng.random() < 0.7
    if train:
        c["noise"] = rng.choice((0.0, 0.04, 0.04))
        c["flavour"] = rng.choice(("plain",) * 6 + ("bias", "abs_max"))
        c["routing"] = rng.choice(("router", "even", "zipf"))
        if c["flavour"] == "plain" and rng.random() < 0.2:
            c["modifier"] = rng.choice(("DISCRETIZE", "ADD_NORMAL", "DISCRETIZE_ADD_NORMAL_PER_CHANNEL"))
    else:
        c["router"] = True
        c["flavour"] = rng.choice(("plain",) * 6 + ("bias",))
    return c


def _rpu_config(c):
    r = rpu.AIHWKITTorchInferenceRPUConfig() if c["flavour"] == "abs_max" else rpu.TorchInferenceRPUConfig()
    r.forward.inp_res = 2 ** 8 - 2
    r.forward.out_noise = c["noise"]
    if c["adc"]:
        r.forward.out_res, r.forward.out_bound = 2 ** 8 - 2, 12.0
    if c["flavour"] == "abs_max":
        r.forward.noise_management = rpu.NoiseManagementType.ABS_MAX
        r.remap.type = rpu.WeightRemapType.CHANNELWISE_SYMMETRIC
    r.mapping.max_input_size = c["mis"]
    ir = r.pre_post.input_range
    ir.enable, ir.learn_input_range, ir.init_value, ir.decay = True, True, 3.0, 0.01
    r.modifier.type = rpu.WeightModifierType[c["modifier"]]
    r.modifier.std_dev, r.modifier.res = 0.02, 2 ** 8 - 2
    if c["clip"]:
        r.clip.type, r.clip.sigma = rpu.WeightClipType.LAYER_GAUSSIAN, 2.5
    return r


def _routing(c, x, g):
    """Gate values and expert ids [T, k] of a routing decision made before the pass."""
    T, E, k = c["T"], c["E"], c["k"]
    if c["routing"] == "even":
        base = torch.arange(T * k, device="cuda").reshape(T, k)
        idx = (base + torch.randint(0, E, (T, 1), generator=g, device="cuda")) % E
        return torch.rand(T, k, generator=g, device="cuda") * 0.5 + 0.25, idx
    if c["routing"] == "zipf":
        p = torch.arange(1, E + 1, dtype=torch.float32, device="cuda") ** -1.2
        logits = torch.randn(T, E, generator=g, device="cuda") + torch.log(p / p.sum())
    else:
        logits = x @ (torch.randn(c["D"], E, generator=g, device="cuda") / c["D"] ** 0.5)
    return torch.sigmoid(logits).topk(k, dim=-1, sorted=False)


def prepare(case, seed):
    c = dict(DEFAULTS, **case)
    dt = DTYPES[c["dtype"]]
    g = torch.Generator(device="cuda").manual_seed(seed)

    def normal(*shape):
        return torch.randn(*shape, generator=g, device="cuda")

    torch.manual_seed(seed)
    cls = AnalogSigmaMoELayerAIHWKIT if c["flavour"] == "abs_max" else AnalogSigmaMoELayer
    with torch.device("cuda"):
        layer = cls(_rpu_config(c), d_model=c["D"], n_experts=c["E"], expert_size=c["F"], k=c["k"],
                    bias=c["flavour"] == "bias")
    with torch.no_grad():
        layer.keys.copy_(normal(*layer.keys.shape) / c["D"] ** 0.5)
        layer.values.copy_(normal(*layer.values.shape) / c["F"] ** 0.5)
        layer.expert_sel.weight.copy_(normal(*layer.expert_sel.weight.shape) / c["D"] ** 0.5)
        if c["flavour"] == "bias":
            layer.bias.copy_(0.1 * normal(*layer.bias.shape))
            layer.o_bias.copy_(0.1 * normal(*layer.o_bias.shape))
    layer = layer.to(dt)
    layer.train(c["train"])
    x = normal(1, c["T"], c["D"])
    s = dict(c, layer=layer)
    if c["train"]:
        layer.use_device_noise_counter()
        if not c["router"]:
            gate, idx = _routing(c, x[0], g)
            s["gate"], s["idx"] = gate.to(dt)[None].requires_grad_(), idx[None].contiguous()
        s["dy"] = normal(1, c["T"], c["D"]).to(dt)
    s["x"] = x.to(dt).requires_grad_(c["train"])
    return s


def run(s):
    layer, x = s["layer"], s["x"]
    if not s["train"]:
        with torch.no_grad():
            return layer(x)[0]
    wrt = {"x": x, "keys": layer.keys, "values": layer.values, "input_range": layer.input_range}
    if s["router"]:
        wrt["router"], wrt["router_input_range"] = layer.expert_sel.weight, layer.expert_sel.input_range
    else:
        wrt["gate"] = s["gate"]
    if s["flavour"] == "bias":
        wrt["bias"], wrt["o_bias"] = layer.bias, layer.o_bias
    for p in wrt.values():
        p.grad = None
    if s["router"]:
        y, reg = layer(x)
        torch.autograd.backward((y, 0.01 * reg), (s["dy"], None))
    else:
        y = layer.forward_selected(x, s["gate"], s["idx"])
        y.backward(s["dy"])
    out = {"y": y.detach(), **{n: p.grad for n, p in wrt.items()}}
    if s["clip"]:
        layer.post_update_step()
        out["clipped_keys"], out["clipped_values"] = layer.keys.detach(), layer.values.detach()
    return out


def work(case):
    c = dict(DEFAULTS, **case)
    T, D, E, F, k = (c[n] for n in "TDEFk")
    M, b = T * k, DTYPES[c["dtype"]].itemsize
    if not c["train"]:
        # every token in and out once, the weights of the experts that get tokens once
        return {"bytes": b * (2 * T * D + 2 * min(E, M) * D * F + D * E), "flops": 4 * M * D * F + 2 * T * D * E}
    # x, dy in; y, grad_x out; the hidden activation and its gradient once each way; weights in (both directions),
    # weight gradients out; the selection
    w = {"bytes": b * (4 * T * D + 4 * M * F + 6 * min(E, M) * D * F) + 24 * M, "flops": 12 * M * D * F}
    if c["router"]:
        w["bytes"] += b * (3 * D * E + 2 * T * E)
        w["flops"] += 6 * T * D * E
    if c["clip"]:
        w["bytes"] += b * 4 * E * D * F
    return w


def tolerance(case):
    # Measured on the listed cases and eight drawn ones, each run again with the features of x and of the first
    # projection's weights in another order (the same products, summed otherwise) and, without noise, as two single
    # projections instead of the fused pair (one rounding of the down-projection's result more).  Another order moves a
    # few hidden values across a step of the quantisers: up to 7.3e-4 of the norm and 0.17 of a single value.  The extra
    # rounding is 2.8e-3 of the norm in bf16, 4.4e-4 in fp16.  Four times that:
    return {"rel": 3e-3 if dict(DEFAULTS, **case)["dtype"] == "f32" else 1e-2, "max": 0.7}
