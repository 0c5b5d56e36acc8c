"""The work that programs have this framework do on one GPU, as cases that can be prepared, run and compared.

Every case goes through public entry points: the neuron modules (``IFNode``, ``LIFNode``, ``ParametricLIFNode`` with
``backend="hip"``), the spike compression functions, ``SpikingSelfAttention`` and ``SpikformerConv2dBNLIF``.  ``listed()`` holds
fixed ones, ``draw(rng)`` more of the same ranges.  Five kinds:

``train``      forward and backward of one multi-step neuron layer, ``[T, B, C, H, W]``
``step``       the same kind of layer called one time step at a time, inference only
``bits``       inference of an IF layer whose spikes are bit-packed for storage and unpacked again
``attention``  the spiking self-attention block ``[T, B, D, tokens]``, training or inference
``conv``       kernel-size-1 convolution + batch norm + LIF (a layer of a spiking MLP) on spike input, forward and backward
"""

import math

import torch

from spikingjelly_amd import configure
from spikingjelly_amd.activation_based import functional, layer, neuron, surrogate
from spikingjelly_amd.activation_based.hip_kernel.compress import bit_spike_compress, bit_spike_decompress
from spikingjelly_amd.activation_based.model.spikformer import SpikformerConv2dBNLIF

_DTYPES = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}


def _train(name, node, dtype, T, B, C, H, W, v_seq, soft=False, mode="torch"):
    """``mode``: what 16-bit storage means, every op rounded ("torch") or fp32 state ("fp32_state")."""
    return {"name": name, "kind": "train", "node": node, "dtype": dtype, "T": T, "B": B, "C": C, "H": H, "W": W,
            "v_seq": v_seq, "soft": soft, "mode": mode}


def _attention(name, train, T, B, D, heads, tokens):
    return {"name": name, "kind": "attention", "train": train, "T": T, "B": B, "D": D, "heads": heads, "tokens": tokens}


def listed():
    return [
        # a fully connected layer of a small classifier: 8192 neurons, the time is the calls and not the data
        _train("lif_f32_small", "lif", "f32", 4, 64, 128, 1, 1, False),
        # the early layer of a large convolutional network at a training batch that fills the memory system
        _train("lif_f32_large", "lif", "f32", 16, 256, 128, 32, 32, True),
        # the last, incomplete batch of an epoch over feature maps with an odd side: rows of an odd number of elements
        _train("lif_f32_ragged", "lif", "f32", 8, 61, 67, 27, 27, False),
        # learnable time constant in bf16 with fp32 state, the mixed-precision training of a mid layer
        _train("plif_bf16", "plif", "bf16", 8, 128, 256, 16, 16, True, True, "fp32_state"),
        # half-precision training of an odd-sized map, bit-identical to the torch backend on half tensors
        _train("lif_f16_ragged", "lif", "f16", 6, 33, 129, 29, 29, False),
        # event streams: many time steps, few neurons
        _train("lif_f32_long", "lif", "f32", 128, 32, 32, 32, 32, False),
        # a layer driven one step at a time (closed-loop or streaming inference)
        {"name": "lif_f32_steps", "kind": "step", "dtype": "f32", "T": 8, "B": 32, "C": 128, "H": 16, "W": 16},
        # converted networks: integrate-and-fire on rate-coded half inputs, spikes stored as bits and read back
        {"name": "if_f16_bits", "kind": "bits", "dtype": "f16", "T": 32, "B": 64, "C": 512, "H": 14, "W": 14, "fused": False},
        # one training step of an attention block at a usual batch
        _attention("attention_train", True, 4, 64, 384, 12, 196),
        # the same block answering a single request
        _attention("attention_infer", False, 4, 1, 384, 12, 196),
        # an attention block over 7 x 7 positions: token counts are not always a multiple of four
        _attention("attention_ragged", True, 4, 16, 256, 8, 49),
        # the widening layer of a spiking MLP
        {"name": "mlp_train", "kind": "conv", "T": 4, "B": 32, "Cin": 384, "Cout": 1536, "H": 14, "W": 14},
    ]


def _log_uniform(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _layer_shape(rng, neurons):
    """``(B, C, H, W)`` of about ``neurons`` neurons: powers of two, or any sizes (odd ones among them)."""
    if rng.random() < 0.5:
        side = rng.choice([1, 4, 8, 16, 32])
        C = rng.choice([32, 64, 128, 256])
    else:
        side = rng.choice([1, 3, 5, 7, 9, 13, 14, 27, 28, 29])
        C = rng.randint(10, 260)
    while side > 1 and side * side * C > neurons:
        side //= 2
    return max(1, neurons // (C * side * side)), C, side, side


def draw(rng):
    kind = rng.choice(["train", "train", "train", "step", "bits", "attention", "attention", "conv"])
    if kind == "train":
        T = rng.choice([1, 2, 4, 4, 6, 8, 8, 10, 16, 20, 32, 64, 128])
        dtype = rng.choice(["f32", "f32", "f16", "bf16"])
        steps = _log_uniform(rng, 3e4, 2e8)  # neurons x time steps
        B, C, H, W = _layer_shape(rng, max(64, steps // T))
        case = _train("", rng.choice(["lif", "lif", "plif", "if"]), dtype, T, B, C, H, W, rng.random() < 0.5,
                      rng.random() < 0.3, "torch" if dtype == "f32" else rng.choice(["torch", "fp32_state"]))
    elif kind == "step":
        B, C, H, W = _layer_shape(rng, _log_uniform(rng, 8e3, 4e6))
        case = {"kind": "step", "dtype": rng.choice(["f32", "f16"]), "T": rng.randint(4, 16), "B": B, "C": C, "H": H, "W": W}
    elif kind == "bits":
        T = rng.choice([4, 8, 16, 32])
        B, C, H, W = _layer_shape(rng, max(64, _log_uniform(rng, 1e5, 2e8) // T))
        whole = (B * C * H * W) % 8 == 0  # rows that start on a byte can be packed by the neuron itself
        case = {"kind": "bits", "dtype": rng.choice(["f32", "f16"]), "T": T, "B": B, "C": C, "H": H, "W": W,
                "fused": whole and rng.random() < 0.5}
    elif kind == "attention":
        heads, per_head = rng.choice([4, 6, 8, 12]), rng.choice([32, 32, 48, 64])
        train = rng.random() < 0.6
        case = _attention("", train, rng.choice([2, 4, 4, 6]), _log_uniform(rng, 1, 32), heads * per_head, heads,
                          rng.choice([49, 64, 81, 100, 144, 196]))
    else:
        side = rng.choice([7, 8, 10, 14])
        case = {"kind": "conv", "T": rng.choice([2, 4, 4, 6]), "B": _log_uniform(rng, 1, 32), "Cin": 32 * rng.randint(3, 16),
                "Cout": 32 * rng.randint(3, 48), "H": side, "W": side}
    case.pop("name", None)
    return case


# ------------------------------------------------------------------------------------------------------------------------------
def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _normal(shape, mean, std, dtype, g):
    return torch.randn(shape, generator=g, device="cuda").mul_(std).add_(mean).to(dtype)


def _node(case):
    reset = None if case.get("soft") else 0.0
    common = dict(v_reset=reset, step_mode="m", backend="hip", store_v_seq=bool(case["v_seq"]))
    if case["node"] == "if":
        return neuron.IFNode(surrogate_function=surrogate.ATan(2.0), **common)
    if case["node"] == "plif":
        return neuron.ParametricLIFNode(init_tau=2.0, surrogate_function=surrogate.Sigmoid(4.0), **common)
    return neuron.LIFNode(tau=2.0, surrogate_function=surrogate.ATan(2.0), **common)


def _initialise(conv, bn, fan_in, g):
    with torch.no_grad():
        conv.weight.uniform_(-1.0, 1.0, generator=g).mul_(fan_in ** -0.5)
        bn.weight.uniform_(0.8, 1.6, generator=g)
        bn.bias.uniform_(0.0, 0.4, generator=g)


def prepare(case, seed):
    g = _generator(seed)
    kind = case["kind"]
    configure.hip_half_precision_mode = case.get("mode", "torch")
    s = {"kind": kind, "case": case}
    if kind == "attention":
        T, B, D, tokens = case["T"], case["B"], case["D"], case["tokens"]
        # weights as the layers initialise them (uniform within 1 / sqrt(fan in)); batch norm as training leaves it, with
        # scales and offsets that make the neurons behind it fire at rates between a few and some twenty per cent
        block = layer.SpikingSelfAttention(D, case["heads"], backend="hip").cuda()
        for conv, bn, variance in ((block.qkv_conv_bn[0], block.qkv_conv_bn[1], 1 / 3), (block.proj_conv_bn[0], block.proj_conv_bn[1], 0.06)):
            _initialise(conv, bn, D, g)
            bn.running_var.fill_(variance)
        block.train(case["train"])
        s["block"], s["x"] = block, _normal((T, B, D, tokens), 0.0, 1.0, torch.float32, g)
        if case["train"]:
            s["x"].requires_grad_()
            s["grad"] = _normal((T, B, D, tokens), 0.0, 1.0, torch.float32, g)
        return s
    if kind == "conv":
        T, B, Cin, Cout, H, W = (case[k] for k in ("T", "B", "Cin", "Cout", "H", "W"))
        block = SpikformerConv2dBNLIF(Cin, Cout, kernel_size=1, backend="hip").cuda()
        _initialise(block.conv_bn.block[0], block.conv_bn.block[1], Cin, g)
        # what a residual stream carries into such a layer: the sum of the spikes of two branches
        x = (torch.rand((T, B, Cin, H, W), generator=g, device="cuda") < 0.15).float()
        x += torch.rand((T, B, Cin, H, W), generator=g, device="cuda") < 0.1
        s["block"], s["x"] = block, x.requires_grad_()
        s["grad"] = _normal((T, B, Cout, H, W), 0.0, 1.0, torch.float32, g)
        return s
    dtype = _DTYPES[case["dtype"]]
    shape = tuple(case[k] for k in ("T", "B", "C", "H", "W"))
    if kind == "bits":
        s["x"] = (torch.rand(shape, generator=g, device="cuda") * 0.25).to(dtype)
        s["node"] = neuron.IFNode(v_threshold=1.0, v_reset=None, step_mode="m", backend="hip").cuda().eval()
        s["v0"] = torch.zeros(shape[1:], dtype=dtype, device="cuda")
        return s
    if kind == "step":
        s["x"] = _normal(shape, 0.5, 1.0, dtype, g)
        s["node"] = neuron.LIFNode(tau=2.0, step_mode="s", backend="hip").cuda().eval()
        return s
    s["x"] = _normal(shape, 0.3, 0.8, dtype, g).requires_grad_()
    s["grad"] = _normal(shape, 0.0, 1.0, dtype, g)
    if case["v_seq"]:
        s["grad_v"] = _normal(shape, 0.0, 0.1, dtype, g)
    s["node"] = _node(case).cuda()
    return s


def run(s):
    kind, x = s["kind"], s["x"]
    if kind == "train":
        node = s["node"]
        x.grad = None
        for p in node.parameters():
            p.grad = None
        spikes = node(x)
        if node.store_v_seq:
            v_seq = node.v_seq
            torch.autograd.backward([spikes, v_seq], [s["grad"], s["grad_v"]])
        else:
            v_seq = None
            spikes.backward(s["grad"])
        v = node.v
        functional.reset_net(node)
        return [spikes.detach(), v.detach(), None if v_seq is None else v_seq.detach(), x.grad] + [p.grad for p in node.parameters()]
    if kind == "step":
        node = s["node"]
        with torch.no_grad():
            spikes = [node(x[t]) for t in range(x.shape[0])]
        v = node.v
        functional.reset_net(node)
        return spikes + [v]
    if kind == "bits":
        with torch.no_grad():
            if s["case"]["fused"]:
                packed, v, _ = functional.if_multi_step_hip_packed(x, s["v0"], 1.0, None)
                return [packed, v, bit_spike_decompress(packed, x.shape, dtype=x.dtype)]
            node = s["node"]
            spikes = node(x)
            packed = bit_spike_compress(spikes)
            v = node.v
            functional.reset_net(node)
            return [packed, v, bit_spike_decompress(packed, spikes.shape, dtype=x.dtype)]
    # Blocks of convolutions, batch norms and neurons.  Their spikes leave as bits, as a program that keeps them for later
    # stores them.
    block = s["block"]
    if kind == "attention" and not s["case"]["train"]:
        with torch.no_grad():
            spikes = block(x)
        functional.reset_net(block)
        return [bit_spike_compress(spikes)]
    x.grad = None
    for p in block.parameters():
        p.grad = None
    spikes = block(x)
    spikes.backward(s["grad"])
    functional.reset_net(block)
    return [bit_spike_compress(spikes.detach()), x.grad] + [p.grad for p in block.parameters()]


def work(case):
    kind = case["kind"]
    if kind == "attention":
        T, B, D, L = case["T"], case["B"], case["D"], case["tokens"]
        columns, heads = T * B * L, case["heads"]
        per_head = D // heads
        act = columns * D
        products = 2.0 * columns * D * 4 * D                         # both convolutions, forward
        contraction = 2.0 * T * B * heads * 2 * per_head * per_head * L  # V K^T and its product with Q
        if not case["train"]:
            return {"bytes": 4.0 * act + 4.0 * 4 * D * D + 4.0 * act, "flops": products + contraction}
        # in: input, gradient of the output, weights; out: spikes, gradient of the input and of the weights
        return {"bytes": 4.0 * (2 * act + 4 * D * D) + 4.0 * (2 * act + 4 * D * D), "flops": 3.0 * products + 3.0 * contraction}
    if kind == "conv":
        T, B, Cin, Cout, H, W = (case[k] for k in ("T", "B", "Cin", "Cout", "H", "W"))
        columns = T * B * H * W
        return {"bytes": 4.0 * (2 * columns * Cin + 2 * columns * Cout + 2 * Cin * Cout), "flops": 3.0 * 2.0 * columns * Cin * Cout}
    n = case["B"] * case["C"] * case["H"] * case["W"]
    size = 4 if case["dtype"] == "f32" else 2
    tn = case["T"] * n
    if kind == "step":
        return {"bytes": float(2 * tn * size + n * size), "flops": 8.0 * tn}
    if kind == "bits":  # x in, bits out and in again, spikes out, state in and out
        return {"bytes": float(2 * tn * size + tn // 4 + 2 * n * size), "flops": 6.0 * tn}
    tensors = 6 if case["v_seq"] else 4  # x, spike gradient (, state gradient) in; spikes (, states), input gradient out
    return {"bytes": float(tensors * tn * size + n * size), "flops": 30.0 * tn}


def tolerance(case):
    """Spikes, states and bits are defined bit for bit; gradients carry the rounding of their type.

    Measured with this framework's own alternatives, stated about four times that: fp32 gradients with the sums of the
    parametric neuron's dL/dk in another order 2e-6; 16-bit gradients whose membrane potentials were stored in the 16-bit
    type between forward and backward instead of recomputed in fp32, bf16: 2.9e-3 (largest single difference 0.05), dL/dk
    2.5e-2 (its terms cancel); blocks with convolutions split into other terms, or run by the library: up to 5.9e-3, because
    1.4e-5 of the spikes (1.1e-4 of their bytes) fall on the other side of their threshold with another order of a
    convolution's sums, and single gradients behind such a spike are off by 0.76."""
    kind = case["kind"]
    if kind in ("attention", "conv"):
        return {"rel": 2.4e-2, "max": 0.99, "differ": 5e-4}
    if kind != "train":
        return "exact"
    plif = case["node"] == "plif"
    if case["dtype"] == "f32":
        return {"rel": 1e-5 if plif else 4e-6, "max": 1e-4}
    fine = case["dtype"] == "f16"  # three more bits of fraction
    if case["mode"] == "torch":
        # the recurrence's values are those of the 16-bit type itself: only the last rounding of a gradient is free
        return {"rel": 1e-3 if fine else 8e-3, "max": 4e-3 if fine else 3e-2}
    if plif:
        return {"rel": 4e-3 if fine else 3e-2, "max": 2.5e-2 if fine else 0.2}
    return {"rel": 1.5e-3 if fine else 1.2e-2, "max": 2.5e-2 if fine else 0.2}
