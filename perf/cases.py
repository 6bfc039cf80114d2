"""Workloads of the Clebsch-Gordan layers for timing and comparison, through the package's public modules.

A case is a dict of plain values:

    kind      "product"  CG_woFilter_cuda alone (the CG product)
              "mixing"   MyBatchNormWeightMM_cuda alone (fragment norm + weight mixing on a given product tensor)
              "layer"    one CGBN_cuda layer
              "stack"    SphericalCNN with its l=0 embedding and a linear head of ten classes
              "net"      MNIST_Net, the classifier
    lmax      degrees l = 0..lmax
    tau_type, tau   channels per degree as model.define_taus gives them: 1 constant, 2 ~ tau/(2l+1), 3 ~ tau/sqrt(2l+1)
    batch     samples
    mst       True: minimum-spanning-tree triples (``sparse_flag``), False: every l2 <= l1
    train     True: forward in training mode and backward, False: evaluation mode without gradients
    layers, tau_in  (stacks and nets) number of layers, channels of the input in every degree

All arithmetic is single precision, the only data type of these modules.
"""
import math

import numpy as np
import torch

from cgnet_amd import CG_layers, CGNet, CGutils, model


def listed():
    return [
        # the smallest call: one CG product of a toy model; launches and the host path count, nothing else
        {"name": "product_L3_tau2_B4", "kind": "product", "lmax": 3, "tau_type": 1, "tau": 2, "batch": 4, "mst": False, "train": False},
        # a training step of the smallest layer: ten launches and autograd around them
        {"name": "layer_L3_tau2_B4_train", "kind": "layer", "lmax": 3, "tau_type": 1, "tau": 2, "batch": 4, "mst": False, "train": True},
        # a layer with few channels in evaluation (spherical-MNIST-shaped fragments, validation pass)
        {"name": "layer_L11_tau5_B32_eval", "kind": "layer", "lmax": 11, "tau_type": 1, "tau": 5, "batch": 32, "mst": False, "train": False},
        # the headline workload: one layer, forward and backward, of a training step
        {"name": "layer_L11_tau12_B100_train", "kind": "layer", "lmax": 11, "tau_type": 1, "tau": 12, "batch": 100, "mst": False, "train": True},
        # the same layer where a trained model is evaluated
        {"name": "layer_L11_tau12_B100_eval", "kind": "layer", "lmax": 11, "tau_type": 1, "tau": 12, "batch": 100, "mst": False, "train": False},
        # the CG product as an operator of its own, forward and backward, at a high degree
        {"name": "product_L15_tau16_B64_train", "kind": "product", "lmax": 15, "tau_type": 1, "tau": 16, "batch": 64, "mst": False, "train": True},
        # the same with the reduced set of triples
        {"name": "product_mst_L15_tau16_B64_train", "kind": "product", "lmax": 15, "tau_type": 1, "tau": 16, "batch": 64, "mst": True, "train": True},
        # fragment norm and mixing as an operator of their own (callers that chain the two modules)
        {"name": "mixing_L11_tau12_B50_train", "kind": "mixing", "lmax": 11, "tau_type": 1, "tau": 12, "batch": 50, "mst": False, "train": True},
        # the largest: four layers at degree 20 on real signals, 12 GB of product tensors, one training step
        {"name": "stack_L20_tau16_B32_train", "kind": "stack", "lmax": 20, "tau_type": 1, "tau": 16, "batch": 32, "mst": False, "train": True, "layers": 4, "tau_in": 1},
        # reduced triples, six input signals, ragged channels (16, 10, 8, 7, 6, 5, ... 4) and an odd batch
        {"name": "stack_mst_L13_tau16r_B27_train", "kind": "stack", "lmax": 13, "tau_type": 3, "tau": 16, "batch": 27, "mst": True, "train": True, "layers": 3, "tau_in": 6},
        # a training step of the spherical-MNIST classifier: five layers, channels 12, 7, 6, 5, 4, ... 3
        {"name": "net_L10_tau12r_B100_train", "kind": "net", "lmax": 10, "tau_type": 3, "tau": 12, "batch": 100, "mst": False, "train": True, "layers": 5, "tau_in": 1},
        # the classifier asked for one image at a time
        {"name": "net_L10_tau12r_B1_eval", "kind": "net", "lmax": 10, "tau_type": 3, "tau": 12, "batch": 1, "mst": False, "train": False, "layers": 5, "tau_in": 1},
    ]


def _log_int(rng, low, high):
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    """One more case: degrees up to 20, up to 16 channels in constant or falling numbers, 1 to 128 samples."""
    kind = rng.choice(["product", "mixing", "layer", "layer", "stack", "net"])
    case = {"kind": kind, "lmax": rng.randint(2, 20), "tau_type": rng.choice([1, 1, 2, 3]), "tau": _log_int(rng, 1, 16),
            "batch": _log_int(rng, 1, 128), "mst": rng.random() < 0.3, "train": rng.random() < 0.65}
    if kind in ("stack", "net"):
        case["layers"] = rng.randint(2, 5)
        case["tau_in"] = rng.choice([1, 1, 2, 6]) if kind == "stack" else 1
    limit = max(_cost(c) for c in listed())
    while _cost(case) > limit and case["batch"] > 1:
        case["batch"] = (case["batch"] + 1) // 2
    while _cost(case) > limit:
        case["layers"] -= 1
    return case


# --------------------------------------------------------------------------- sizes and work
def _taus(case):
    return model.define_taus(case["tau_type"], case["tau"], case["lmax"])


def _layer_taus(case):
    """Channels per degree entering the first layer and leaving every layer."""
    taus = _taus(case)
    if case["kind"] in ("stack", "net"):
        return [[case["tau_in"]] * (case["lmax"] + 1)] + [taus] * case["layers"]
    return [taus, taus]


def _triples(lmax, mst):
    pairs = (CGutils.SparseLtuples.compute_mst_ltuples(lmax) if mst else CGutils.SparseLtuples.compute_default_ltuples(lmax))
    return [(l, l1, l2) for l in range(lmax + 1) for l1, l2 in pairs[l]]


def _sizes(case, taus_in, taus_out):
    """Of one layer: entries per sample of F, FF and O, of W, channels of FF, multiply-adds of the product per sample."""
    lmax = case["lmax"]
    t_ff, macs, table = [0] * (lmax + 1), 0, 0
    for l, l1, l2 in _triples(lmax, case["mst"]):
        channels = taus_in[l1] * taus_in[l2]
        t_ff[l] += channels
        macs += channels * sum(max(0, min(l2, m + l1) - max(-l2, m - l1) + 1) for m in range(-l, l + 1))
        table += (2 * l + 1) * (2 * l2 + 1)
    entries = lambda taus: sum(t * (2 * l + 1) for l, t in enumerate(taus))  # noqa: E731
    return {"F": entries(taus_in), "FF": entries(t_ff), "O": entries(taus_out), "channels": sum(t_ff), "table": table,
            "W": sum(a * b for a, b in zip(t_ff, taus_out)), "product": macs,
            "mix": sum(a * b * (2 * l + 1) for l, (a, b) in enumerate(zip(t_ff, taus_out)))}


def work(case):
    """Complex numbers have 8 bytes, a complex multiply-add 8 operations.  The product tensor counts where it crosses the
    caller's boundary ("product": it is the result, "mixing": the input); inside a layer it need not exist."""
    B, kind, train = case["batch"], case["kind"], case["train"]
    taus = _layer_taus(case)
    nbytes = flops = 0
    for i in range(len(taus) - 1):
        s = _sizes(case, taus[i], taus[i + 1])
        grad_in = train and (i > 0 or kind not in ("stack", "net"))     # the first layer of a model reads data
        product, mix = 8 * B * s["product"], 8 * B * s["mix"]
        if kind == "product":
            flops += product * (3 if train else 1)
            nbytes += 8 * B * (s["F"] + s["FF"]) * (2 if train else 1) + 4 * s["table"]
        elif kind == "mixing":
            flops += mix * (3 if train else 1)
            nbytes += 8 * (B * (s["FF"] + s["O"]) + s["W"]) * (2 if train else 1) + 4 * s["channels"] * (2 if train else 1)
        else:
            flops += product * (3 if grad_in else 1) + mix * (1 + train + grad_in)
            # activations between the layers of a model need not leave the chip any more than FF does
            ends = B * ((s["F"] if i == 0 else 0) + (s["O"] if kind == "layer" else 0)) * (2 if train and kind == "layer" else 1)
            nbytes += 8 * (ends + s["W"] * (2 if train else 1)) + 4 * (s["table"] + s["channels"] * (2 if train else 1))
    if kind in ("stack", "net"):
        width = 2 * sum(t[0] for t in taus)
        head = width * 10 if kind == "stack" else width * 256 + 2560
        flops += 2 * B * head * (3 if train else 1)
        nbytes += 4 * head * (2 if train else 1) + 4 * 10 * B
    return {"bytes": nbytes, "flops": flops}


def _cost(case):
    """Time is spent on operations and on the product tensors that the modules hold: the dearer of the two."""
    taus = _layer_taus(case)
    ff = sum(_sizes(case, taus[i], taus[i + 1])["FF"] for i in range(len(taus) - 1))
    return max(work(case)["flops"] / 20, 8 * case["batch"] * ff * (5 if case["train"] else 2))


def tolerance(case):
    """About four times what the package's own routes differ by on the same inputs (matrix cores or vector units, backward
    in one or two kernels, folded or full diagonal triples): 4.2e-7 / 2.9e-6 for a single layer, 4.2e-5 / 4.9e-3 for
    several, where every layer squares the relative error of what comes in and divides small channels by small stds."""
    if case["kind"] in ("stack", "net"):
        return {"rel": 2e-4, "max": 0.02}
    return {"rel": 2e-6, "max": 2e-5}


# --------------------------------------------------------------------------- inputs
def _gaussian(taus, batch, gen):
    """Straight fragments, i.i.d. with variance 1/(2l+1)."""
    return torch.cat([torch.randn(batch, t * (2 * l + 1), 2, generator=gen, device="cuda") / math.sqrt(2 * l + 1)
                      for l, t in enumerate(taus)], dim=1)


def _real_signal(channels, lmax, batch, gen):
    """Straight coefficients of real signals: f_l^{-m} = (-1)^m conj(f_l^m), variance 1/(2l+1)."""
    parts = []
    for l in range(lmax + 1):
        pos = torch.randn(batch, channels, l + 1, 2, generator=gen, device="cuda") / math.sqrt(2 * l + 1)
        pos[:, :, 0, 1] = 0.
        sign = torch.tensor([(-1.) ** m for m in range(l, 0, -1)], device="cuda").reshape(1, 1, l, 1)
        neg = pos[:, :, 1:].flip(2) * sign * torch.tensor([1., -1.], device="cuda")
        parts.append(torch.cat([neg, pos], dim=2).reshape(batch, -1, 2))
    return torch.cat(parts, dim=1)


def _set_weights(mixing, gen):
    """Weights of variance ~ 1/(product channels) per degree."""
    with torch.no_grad():
        for l in range(mixing.lmax + 1):
            a, b = int(mixing.cumu_tm_W[l]), int(mixing.cumu_tm_W[l + 1])
            if b > a:
                mixing.W[a:b] = torch.randn(b - a, 2, generator=gen, device="cuda") * (0.5 / math.sqrt(2 * int(mixing.t_FF[l])))


def _train_a_little(net, x):
    """Running stds as after some training: nine tenths of a batch's, one tenth of the random start (what keeps channels
    that vanish by symmetry away from zero); the count of a later step."""
    mixings = [m for m in net.modules() if isinstance(m, CG_layers.MyBatchNormWeightMM_cuda)]
    norms = [m for m in net.modules() if isinstance(m, torch.nn.BatchNorm1d)]
    for m in mixings:
        m.bn_cnt = 1. / 9.
    for m in norms:
        m.momentum = 1.
    with torch.no_grad():
        net.train()(x)
    for m in mixings:
        m.bn_cnt = 10.
    for m in norms:
        m.momentum = 0.1


def prepare(case, seed):
    """The module with its weights, the batch and, for operators, the gradient that comes from above."""
    torch.manual_seed(seed)
    np.random.seed(seed % (1 << 31))
    gen = torch.Generator(device="cuda").manual_seed(seed)
    kind, lmax, B = case["kind"], case["lmax"], case["batch"]
    taus = _taus(case)
    state = {"kind": kind, "train": case["train"]}
    if kind == "product":
        net = CG_layers.CG_woFilter_cuda(lmax, taus, lll_mode="mst" if case["mst"] else None)
        x = _gaussian(taus, B, gen)
        outputs = net.t_FF
    elif kind == "mixing":
        t_ff = [0] * (lmax + 1)
        for l, l1, l2 in _triples(lmax, case["mst"]):
            t_ff[l] += taus[l1] * taus[l2]
        net = CG_layers.MyBatchNormWeightMM_cuda(lmax, t_ff, taus)
        _set_weights(net, gen)
        x = _gaussian(t_ff, B, gen)
        outputs = taus
        net.bn_cnt = 10.
    elif kind == "layer":
        net = CG_layers.CGBN_cuda(lmax, taus, taus, sparse_flag=case["mst"])
        _set_weights(net.bnWMM, gen)
        net.bnWMM.bn_cnt = 10.
        x = _gaussian(taus, B, gen)
        outputs = taus
    else:
        if kind == "stack":
            net = CGNet.SphericalCNN(lmax, _layer_taus(case), sparse_flag=case["mst"])
            state["head"] = torch.nn.Linear(net.output_length, 10, device="cuda")
            cnn = net
        else:
            net = model.MNIST_Net(lmax, tau_type=case["tau_type"], tau_man=case["tau"], nlayers=case["layers"], dropout=None, sparse=case["mst"])
            cnn = net.SphericalCNN
        for layer in cnn.cgs:
            _set_weights(layer.bnWMM, gen)
        _train_a_little(net, _real_signal(case["tau_in"], lmax, max(8, min(32, B)), gen))
        x = _real_signal(case["tau_in"], lmax, B, gen)
        state["labels"] = torch.randint(0, 10, (B,), generator=gen, device="cuda")
        outputs = None
    net.train(case["train"])
    if outputs is not None and case["train"]:
        state["grad"] = torch.randn(B, sum(int(t) * (2 * l + 1) for l, t in enumerate(outputs)), 2, generator=gen, device="cuda")
        x.requires_grad_(True)
    state.update(net=net, x=x)
    return state


def run(state):
    """One pass: the forward in evaluation mode, or forward and backward of a training step."""
    net, x, kind = state["net"], state["x"], state["kind"]
    call = (lambda: net(x)) if kind in ("mixing", "stack", "net") else (lambda: net(x, straight_output=True))
    if not state["train"]:
        with torch.no_grad():
            out = call()
            return state["head"](out) if kind == "stack" else out
    net.zero_grad(set_to_none=True)
    result = {}
    if kind in ("stack", "net"):
        if kind == "stack":
            state["head"].zero_grad(set_to_none=True)
            out = torch.log_softmax(state["head"](call()), dim=1)
            result["head"] = list(state["head"].parameters())
        else:
            out = call()
        loss = torch.nn.functional.nll_loss(out, state["labels"])
        loss.backward()
        result["head"] = [p.grad for p in result.get("head", ())]
    else:
        x.grad = None
        out = call()
        out.backward(state["grad"])
        result["grad_input"] = x.grad
    result["out"] = out.detach()
    result["grads"] = {name: p.grad for name, p in net.named_parameters() if p.requires_grad}
    result["stds"] = {name: p.detach() for name, p in net.named_parameters() if name.endswith("bn_stds")}
    return result
