"""The passes that a program built on minml_amd runs, as plain cases: which they are, what they start from, how one pass is made.

A case names a kind of pass and its sizes:

  resnet   minml_amd.resnet.ResNet.forward: stem, residual blocks of 3x3 Winograd layers, 1x1 policy head, fp16 or fp32
  int8     minml_amd.resnet.QuantizedResNet.forward: the same network on int8 activations and weights, fp32 logits
  conv     minml_amd.conv2d.Conv2D.forward: one layer on the implicit-GEMM path (1x1 through gemm_ex), bias, ReLU and a residual
  hybrid   minml_amd.hybridnet.HybridNet.forward: residual trunk, then attention half-blocks
  experts  one mixture-of-experts half-block of that network on activations in hand: normalisation, router, expert-choice routing, gather,
           the two expert layers, scatter (apart from the network's other layers, whose last bit decides which of two equally good tokens
           an expert takes, so that results could not be compared)

`issue` says how the program issues a network's pass: "recorded" replays a recorded pass (core.Graph) as programs with few positions in
flight do, "calls" makes the library calls one by one, and "layers" (resnet) does so with three calls per 3x3 layer, as the reference's
own Conv2D issues them. Everything here is inference: the library has no backward path.
"""
import math

import numpy as np
import torch

from minml_amd import core as ml
from minml_amd.conv2d import IMPLICIT_GEMM, Conv2D
from minml_amd.hybridnet import EXPERTS, HIDDEN, HybridNet, get_capacity, make_hybrid_parameters
from minml_amd.resnet import QuantizedResNet, ResNet, calibrate_activations, he_normal_weights, make_input, make_parameters

PLANES = 32  # binary input planes of the networks
SIZE = {"float16": 2, "float32": 4}


def listed():
    return [
        # one position at a time: a program that plays against a person, or the last positions of a search
        dict(name="resnet_fp16_b1", kind="resnet", dtype="float16", batch=1, board=15, channels=256, blocks=20, issue="recorded"),
        # the leaves that a tree search collects before it evaluates them
        dict(name="resnet_fp16_b16", kind="resnet", dtype="float16", batch=16, board=15, channels=256, blocks=20, issue="recorded"),
        # several games in one process, a count that fills no tile evenly
        dict(name="resnet_fp16_b101", kind="resnet", dtype="float16", batch=101, board=15, channels=256, blocks=20, issue="calls"),
        # the throughput workload: self-play or analysis with a full batch
        dict(name="resnet_fp16_b1024", kind="resnet", dtype="float16", batch=1024, board=15, channels=256, blocks=20, issue="calls"),
        # an unchanged caller of the reference's layers on the large board: every Winograd stage a call of its own
        dict(name="resnet_fp16_layers_b203", kind="resnet", dtype="float16", batch=203, board=19, channels=128, blocks=10, issue="layers"),
        # full precision, the configuration that the reference also runs on its CPU
        dict(name="resnet_fp32_b256", kind="resnet", dtype="float32", batch=256, board=15, channels=128, blocks=10, issue="calls"),
        # the quantised network with a full batch, and with the few positions of an interactive program
        dict(name="int8_b1024", kind="int8", batch=1024, board=15, channels=256, blocks=20, issue="calls"),
        dict(name="int8_b9", kind="int8", batch=9, board=15, channels=128, blocks=10, issue="recorded"),
        # single layers of networks with other kernel sizes: 5x5 and 3x3 on wide layers, and a 1x1 layer on a ragged batch
        dict(name="conv5x5_c256_b512", kind="conv", dtype="float16", batch=512, board=19, channels=256, kernel=5, residual=True),
        dict(name="conv1x1_c384_b77", kind="conv", dtype="float16", batch=77, board=19, channels=384, kernel=1, residual=True),
        # the convolution + attention network with the few positions of an interactive program, and the half-block that it adds to every
        # attention half-block where it has experts, with a full batch
        dict(name="hybrid_b6", kind="hybrid", batch=6, board=15, channels=256, blocks=10, attention=4, heads=8, issue="recorded"),
        dict(name="experts_b256", kind="experts", batch=256, board=15, channels=256),
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    """A case of the same ranges: batches and blocks over their logarithm, boards from 9x9 to 20x20, layer widths from 64 to 384."""
    kind = rng.choice(("resnet", "resnet", "resnet", "int8", "conv", "hybrid", "experts"))
    board = rng.choice((15, 15, 19, rng.randint(9, 20)))
    channels = rng.choice((64, 96, 128, 192, 256, 256, 384))
    if kind == "conv":
        case = dict(kind=kind, dtype=rng.choice(("float16", "float16", "float32")), batch=_log_int(rng, 1, 512), board=board, channels=channels,
                    kernel=rng.choice((1, 3, 5)), residual=rng.random() < 0.5)
    elif kind == "hybrid":
        channels = rng.choice((128, 256))
        case = dict(kind=kind, batch=_log_int(rng, 1, 256), board=board, channels=channels, blocks=_log_int(rng, 2, 10), attention=rng.randint(1, 4),
                    heads=channels // 32, issue="recorded")
    elif kind == "experts":
        case = dict(kind=kind, batch=_log_int(rng, 1, 256), board=board, channels=rng.choice((128, 256)))
    else:
        case = dict(kind=kind, batch=_log_int(rng, 1, 1024), board=board, channels=channels, blocks=_log_int(rng, 2, 20), issue="recorded")
        if kind == "resnet":
            case["dtype"] = rng.choice(("float16", "float16", "float32"))
            case["issue"] = rng.choice(("recorded", "calls", "layers"))
    if case.get("issue") == "recorded" and case["batch"] > 64:
        case["issue"] = "calls"
    # no dearer than the full batch of the largest listed network (fp32 and the widest kernels counted at their own rates)
    most = 0.5 * work(listed()[3])["flops"] / (8 if case.get("dtype") == "float32" else 1)
    while work(case)["flops"] > most and case["batch"] > 1:
        case["batch"] = max(1, case["batch"] * 2 // 3)
    return case


# ---- what a program has in hand -------------------------------------------------------------------------------------------------

_context = None


def _the_context():
    global _context
    if _context is None:
        _context = ml.Context(0)
    return _context


def _half(a):
    return np.ascontiguousarray(a, np.float32).astype(np.float16).view(np.uint16)


def _storage(dtype):
    return _half if dtype == "float16" else (lambda a: np.ascontiguousarray(a, np.float32))


class _State:
    """A network or a layer with its inputs, and one pass of it."""

    def __init__(self, owner, forward, outputs, graph=None):
        self.owner, self.forward, self.outputs, self.graph = owner, forward, outputs, graph


class _DeviceArray:
    """The memory of a minml_amd tensor as torch may look at it; keeps the owner alive."""

    def __init__(self, tensor, owner):
        self.owner = (tensor, owner)
        kind = {ml.dtype_of("float16"): "<f2", ml.dtype_of("float32"): "<f4", ml.dtype_of("int8"): "|i1"}[tensor.dtype]
        self.__cuda_array_interface__ = {"shape": tensor.shape, "typestr": kind, "data": (tensor.ptr, False), "version": 2}


def _as_torch(tensor, owner):
    return torch.as_tensor(_DeviceArray(tensor, owner), device="cuda:0")


def _network_state(case, net, forward, tensors):
    """tensors(net): the tensors that hold the pass's results, known after one pass."""
    graph = None
    if case["issue"] == "recorded":
        forward()  # the ordinary pass that must precede a recording
        graph = ml.Graph.record(_the_context(), forward)
    return _State(net, forward, tensors, graph)


def prepare(case, seed):
    ctx = _the_context()
    kind = case["kind"]
    if kind == "resnet":
        to = _storage(case["dtype"])
        params = make_parameters(seed, PLANES, case["channels"], case["blocks"])
        net = ResNet(ctx, case["batch"], case["board"], PLANES, case["channels"], case["blocks"], case["dtype"], params, to, fused=case["issue"] != "layers")
        net.setInput(to(make_input(seed, case["batch"], case["board"], PLANES)))
        return _network_state(case, net, net.forward, lambda: [net.output, net.trunk_output()])
    if kind == "int8":
        params = make_parameters(seed, PLANES, case["channels"], case["blocks"])
        ranges = calibrate_activations(ctx, params, case["board"], PLANES, case["channels"], case["blocks"], batches=3, seed=seed)
        net = QuantizedResNet(ctx, case["batch"], case["board"], PLANES, case["channels"], case["blocks"], params, ranges)
        net.setInput(make_input(seed, case["batch"], case["board"], PLANES))
        return _network_state(case, net, net.forward, lambda: [net.output])
    if kind == "hybrid":
        params = make_hybrid_parameters(seed, PLANES, case["channels"], case["blocks"], case["attention"], case["heads"], case["board"])
        net = HybridNet(ctx, case["batch"], case["board"], PLANES, case["channels"], case["blocks"], case["heads"], "float16", params, _half)
        net.setInput(_half(make_input(seed, case["batch"], case["board"], PLANES)))
        return _network_state(case, net, net.forward, lambda: [net.output, net.last])
    if kind == "experts":
        return _prepare_experts(ctx, case, seed)
    rng = np.random.default_rng(seed)
    to = _storage(case["dtype"])
    c, k = case["channels"], case["kernel"]
    shape = (case["batch"], case["board"], case["board"], c)
    layer = Conv2D(ctx, shape, c, k, "relu", True, case["dtype"], algorithm=IMPLICIT_GEMM if k > 1 else None)
    layer.setWeights(to(he_normal_weights(rng, (c, k, k, c))), to(rng.standard_normal(c) * 0.1))
    inputs = _normal(seed, [shape] * (2 if case["residual"] else 1), case["dtype"])
    out = ml.Tensor(shape, case["dtype"])
    return _State((layer, inputs), lambda: layer.forward(inputs, out), lambda: [out])


def _normal(seed, shapes, dtype):
    """Activations in hand: N(0, 1), made on the device."""
    draws = torch.Generator(device="cuda:0")
    draws.manual_seed(seed)
    tensors = [ml.Tensor(shape, dtype) for shape in shapes]
    for t in tensors:
        _as_torch(t, None).normal_(generator=draws)
    torch.cuda.synchronize()
    return tensors


def _prepare_experts(ctx, case, seed):
    """The feed-forward half-block as HybridNet.forward issues it; weights N(0, 0.02), biases N(0, 0.01) as there."""
    batch, board, c = case["batch"], case["board"], case["channels"]
    rows, k = batch * board * board, get_capacity(2.0, board * board, EXPERTS)
    rng = np.random.default_rng(seed)
    dev = lambda shape, sigma, mean=0.0: ml.toDevice(ctx, _half(mean + sigma * rng.standard_normal(shape, np.float32)), "float16")
    gamma, w_router, b_router = dev((c,), 0.02, 1.0), dev((EXPERTS, c), 0.02), dev((EXPERTS,), 0.01)
    w_1, b_1, w_2, b_2 = dev((EXPERTS, HIDDEN, c), 0.02), dev((EXPERTS, HIDDEN), 0.01), dev((EXPERTS, c, HIDDEN), 0.02), dev((EXPERTS, c), 0.01)
    x, = _normal(seed, [(batch, board, board, c)], "float16")
    new = lambda *shape: ml.Tensor(shape, "float16")
    normed, scores, table, out = new(batch, board, board, c), new(batch, board, board, EXPERTS), new(batch, 2, EXPERTS, k), new(batch, board, board, c)
    gathered, hidden, slots = new(batch, k, EXPERTS, c), new(batch, k, EXPERTS, HIDDEN), new(batch, k, EXPERTS, c)

    def forward():
        ml.rmsnormForward(ctx, x, normed, gamma)
        ml.gemm_ex(ctx, scores.view((rows, EXPERTS)), 1.0, "n", normed.view((rows, c)), "t", w_router, 0.0, None, b_router, "linear")
        ml.expertChoiceRoutingForward(ctx, scores, table)
        ml.gatherTokensForward(ctx, normed, table, 0.0, gathered)
        ml.moeForward(ctx, gathered, w_1, b_1, 0.0, hidden, "relu")
        ml.moeForward(ctx, hidden, w_2, b_2, 0.0, slots, "linear")
        ml.scatterTokensForward(ctx, slots, table, 0.0, out)

    return _State(None, forward, lambda: [out])


def run(state):
    if state.graph is not None:
        state.graph.launch()
    else:
        state.forward()
    return [_as_torch(t, state) for t in state.outputs()]


# ---- what a pass cannot do without ----------------------------------------------------------------------------------------------

def _tiles(case):
    return case["batch"] * ((case["board"] + 3) // 4) ** 2


def work(case):
    """Bytes: inputs, parameters and results once each (activations between layers not counted). Flops: what the algorithm of the path
    multiplies, i.e. 36 products per 4x4 tile in the Winograd layers, k x k taps elsewhere."""
    pixels, c = case["batch"] * case["board"] ** 2, case["channels"]
    kind = case["kind"]
    if kind == "conv":
        s = SIZE[case["dtype"]]
        weights = case["kernel"] ** 2 * c * c
        return {"bytes": float(s * ((3 if case["residual"] else 2) * pixels * c + weights + c)), "flops": 2.0 * pixels * weights}
    if kind == "experts":
        slots = case["batch"] * EXPERTS * get_capacity(2.0, case["board"] ** 2, EXPERTS)
        weights = EXPERTS * (c + 1 + 2 * c * HIDDEN + HIDDEN + c) + c
        return {"bytes": 2.0 * (2 * pixels * c + weights), "flops": 2.0 * pixels * c * EXPERTS + 4.0 * slots * c * HIDDEN}
    blocks = case["blocks"]
    trunk_weights = 9 * c * (PLANES + 2 * blocks * c)
    if kind == "int8":
        return {"bytes": float(pixels * (PLANES + 4) + trunk_weights + c), "flops": 2.0 * pixels * (trunk_weights + c)}
    s = SIZE[case.get("dtype", "float16")]
    flops = 2.0 * 36 * _tiles(case) * c * (PLANES + 2 * blocks * c) + 2.0 * pixels * c
    values = pixels * (PLANES + 1 + c) + trunk_weights + c
    if kind == "hybrid":
        flops += case["attention"] * (2.0 * pixels * 4 * c * c + 4.0 * pixels * case["board"] ** 2 * c)
        values += case["attention"] * 4 * c * c
    return {"bytes": float(s * values), "flops": flops}


def tolerance(case):
    """About four times what the same pass shows with its sums in another order: the networks with their channels permuted (fp16: 1e-3 to
    1.4e-2 at the logits, the more the smaller their norm, 3e-3 to 4e-3 in the trunk, largest difference 0.08; fp32: 1e-5 and 5e-5), single
    layers and the experts against a 64-bit evaluation (fp16: 4.2e-4 and 1.5e-3, largest 1e-3 and 3.6e-3; fp32: 1.1e-6 and 1.4e-5). fp16
    results are rounded towards zero at every store, so errors of a whole unit in the last place are ordinary."""
    kind = case["kind"]
    if kind == "int8":
        return "exact"  # int32 accumulators, a requantisation without fused operations, one fp32 head in a fixed order
    if kind == "conv":
        return {"rel": 1.5e-3, "max": 4e-3} if case["dtype"] == "float16" else {"rel": 4e-6, "max": 6e-5}
    if kind == "experts":
        return {"rel": 6e-3, "max": 1.5e-2}
    return {"rel": 3e-2, "max": 0.3} if case.get("dtype") != "float32" else {"rel": 4e-5, "max": 2e-4}
