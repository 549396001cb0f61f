"""The work that users of this framework have it do, as cases that can be timed and compared.

Every case is a forward pass through the public entry points: a graph of ``eddl_amd.models`` or of the layer factories,
``Net.build`` on the device and one call of ``Net.forward``, ``Net.predict`` or ``Net.predict_batches``.  A case names

  model   conv (one Conv2D), block (Conv-BN-ReLU-MaxPool), vgg16, resnet50 or unet
  batch, size, width    images of a call and their height and width (the graphs of the three networks take square images)
  channels, filters, kernel, stride    of the single convolution and the block
  mode    forward (input and output stay on the device), predict (host arrays in and out, one blocking call) or
          stream (four host batches through predict_batches)
  fuse    the fused plan, or the layer walk: one call per layer, as the reference's own forward makes them
  search  launch plans searched when the plan is first run (the benchmark and the C++ host do so), or the planner's own

Weights, batch-norm statistics and inputs have the distributions that the benchmark's configurations use (He-normal
filters, running variances in 0.5 ... 1.5), drawn from the seed.
"""
import math

import numpy as np
import torch

import eddl_amd
from eddl_amd import models
from eddl_amd import net as L

NETWORKS = {"vgg16": models.vgg16, "resnet50": models.resnet50, "unet": models.unet}


def _case(name, model, batch, size, mode="forward", fuse=True, search=True, **more):
    return dict(dict(name=name, model=model, batch=batch, size=size, mode=mode, fuse=fuse, search=search), **more)


def listed():
    return [
        # the smallest call anyone makes: one convolution of a CIFAR-sized batch, bound by launches and host time
        _case("conv_3x32x32_b8", "conv", 8, 32, width=32, channels=3, filters=32, kernel=3, stride=1),
        # one stage of a network, the unit that the reference's users stack: 64 images of 56x56
        _case("block_64x56x56_b64", "block", 64, 56, channels=64, filters=64),
        # the headline: throughput of an image classifier with large 3x3 layers and a heavy dense head
        _case("vgg16_b32", "vgg16", 32, 224),
        # one image at a time, as a service answers a request: few tiles, the dense head reads its weights for one row
        _case("vgg16_b1", "vgg16", 1, 224),
        # CIFAR-sized images in a large batch: tiny planes behind the second pool
        _case("vgg16_32px_b128", "vgg16", 128, 32),
        # throughput of a deep residual network: most layers are short 1x1 convolutions with batch norm and residual
        _case("resnet50_b64", "resnet50", 64, 224),
        # the same for one image: more than fifty dependent launches
        _case("resnet50_b1", "resnet50", 1, 224),
        # an odd batch of ragged planes (125, 63, 32, 16, 8 pixels wide), with the planner's own launch plans
        _case("resnet50_250px_b7_planner", "resnet50", 7, 250, search=False),
        # layer by layer, as a program written for the reference runs before it asks for a fused plan: batch norm, ReLU,
        # addition and pooling are launches of their own
        _case("resnet50_walk_b32", "resnet50", 32, 224, fuse=False),
        # host arrays in, host arrays out, one blocking call: the reference's predict
        _case("resnet50_predict_b16", "resnet50", 16, 224, mode="predict"),
        # segmentation at training resolution: encoder, decoder, skip connections; the largest tensors
        _case("unet_512px_b4", "unet", 4, 512),
        # one image of a ragged size through the same network
        _case("unet_368px_b1", "unet", 1, 368),
    ]


def _flops(case):
    """Multiplications and additions of the convolutions and dense layers, direct form."""
    return _work(case)["flops"]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _drawn(rng):
    kind = rng.choice(("conv", "conv", "block", "vgg16", "resnet50", "resnet50", "unet"))
    search = rng.random() < 0.75
    if kind == "conv":
        kernel = rng.choice((1, 1, 3, 3, 3, 5, 7))
        return dict(model="conv", batch=_log(rng, 1, 64), size=_log(rng, 7, 256), width=_log(rng, 7, 256), channels=_log(rng, 1, 512),
                    filters=_log(rng, 8, 512), kernel=kernel, stride=rng.choice((1, 1, 1, 2)), mode="forward", fuse=True, search=search)
    if kind == "block":
        return dict(model="block", batch=_log(rng, 1, 96), size=2 * _log(rng, 7, 112), channels=_log(rng, 16, 256), filters=_log(rng, 16, 256),
                    mode="forward", fuse=True, search=search)
    mode = rng.choice(("forward", "forward", "forward", "predict", "stream"))
    fuse = mode != "forward" or rng.random() < 0.75
    if kind == "unet":
        return dict(model="unet", batch=_log(rng, 1, 4), size=16 * _log(rng, 6, 32), mode=mode, fuse=fuse, search=search)
    if kind == "vgg16":
        return dict(model="vgg16", batch=_log(rng, 1, 48), size=32 * _log(rng, 1, 8), mode=mode, fuse=fuse, search=search)
    return dict(model="resnet50", batch=_log(rng, 1, 64), size=_log(rng, 64, 320), mode=mode, fuse=fuse, search=search)


def draw(rng):
    while True:
        case = _drawn(rng)
        batches = 4 if case["mode"] == "stream" else 1
        if _flops(case) <= 1.2e12 and batches * case["batch"] * case["size"] * case.get("width", case["size"]) * 3 * 4 <= 1 << 28:
            return case


def _graph(case):
    batch, size = case["batch"], case["size"]
    if case["model"] == "conv":
        x = L.Input([case["channels"], size, case["width"]], batch)
        k, s = case["kernel"], case["stride"]
        pads = [k // 2] * 4  # symmetric: "same" of a strided layer would not be, and the layer refuses that
        return L.Net([x], [L.Conv2D(x, case["filters"], [k, k], [s, s], "custom", use_bias=True, pads=pads)])
    if case["model"] == "block":
        return models.conv_bn_relu_pool_block(batch, case["channels"], size, case["filters"])
    return NETWORKS[case["model"]](batch=batch, size=size)


_device = None


def _backend():
    global _device
    if _device is None:
        _device = eddl_amd.Backend(0)
    return _device


def _fill(hip, net, seed):
    """Parameters drawn on the device, layer by layer, with the deviations of the He-normal initialiser."""
    for k, layer in enumerate(net.layers):
        p = net.dparams[id(layer)]
        at = (seed * 1000003 + k * 101) & 0x7FFFFFFF
        if layer.kind == "conv2d":
            _, c, r, s = p["K"].shape
            hip.rand_normal(p["K"], 0.0, math.sqrt(2.0 / (c * r * s)), at)
            hip.rand_normal(p["bias"], 0.0, 0.05, at + 1)
        elif layer.kind == "dense":
            hip.rand_normal(p["W"], 0.0, math.sqrt(2.0 / p["W"].shape[0]), at)
            hip.rand_normal(p["bias"], 0.0, 0.05, at + 1)
        elif layer.kind == "batchnorm":
            hip.rand_uniform(p["bn_g"], 0.4, at)
            hip.add_scalar(p["bn_g"], p["bn_g"], 0.8)
            hip.rand_normal(p["bn_b"], 0.0, 0.1, at + 1)
            hip.rand_normal(p["mean"], 0.0, 0.1, at + 2)
            hip.rand_uniform(p["variance"], 1.0, at + 3)
            hip.add_scalar(p["variance"], p["variance"], 0.5)


class _Shared:
    """Device memory of a framework tensor, as torch reads it without a copy; keeps the tensor."""

    def __init__(self, t):
        self.owner = t
        self.__cuda_array_interface__ = {"shape": tuple(t.shape), "typestr": "<f4", "data": (t.ptr, False), "strides": None, "version": 2}


def _as_torch(t):
    return torch.as_tensor(_Shared(t), device="cuda")


def prepare(case, seed):
    hip = _backend()
    net = _graph(case)
    hip.conv_autotune(bool(case["search"]))
    net.build(hip, fuse=bool(case["fuse"]))
    _fill(hip, net, seed)
    shape = net.lin[0].out_shape
    uniform = case["model"] in ("vgg16", "unet")  # pixels in 0 ... 1; the others take normalised images or feature maps
    state = {"case": case, "net": net}
    if case["mode"] == "forward":
        x = net.input_tensor()
        if uniform:
            hip.rand_uniform(x, 1.0, seed + 77)
        else:
            hip.rand_normal(x, 0.0, 1.0, seed + 77)
        state["x"] = x
        net.forward([x])  # the launch plans are searched here, the workspace grows to its size
        # the network's outputs, a classifier's logits and the features that its dense head reads
        heads = [l for l in net.layers for c in l.children if c.kind in ("reshape", "softmax")]
        state["out"] = [_as_torch(net.output_of(o)) for o in net.lout + heads]
        # the coordinates of a pool's maxima are whole numbers: their bits are compared
        aux = [net.aux[id(l)] for l in net.layers if l.kind == "maxpool2d"] if case["model"] == "block" else []
        state["out"] += [_as_torch(a[key]).view(torch.int32) for a in aux for key in ("indX", "indY")]
        return state
    rng = np.random.default_rng(seed)
    count = 4 if case["mode"] == "stream" else 1
    draw_one = (lambda: rng.random(shape, dtype=np.float32)) if uniform else (lambda: rng.standard_normal(shape, dtype=np.float32))
    state["batches"] = [draw_one() for _ in range(count)]
    net.predict(state["batches"][0])
    return state


def run(state):
    net, mode = state["net"], state["case"]["mode"]
    if mode == "forward":
        net.forward([state["x"]])
        return state["out"]
    if mode == "predict":
        return net.predict(state["batches"][0])
    return list(net.predict_batches(state["batches"]))


def _conv64(x, w, bias, cd):
    """A convolution of doubles, image by image, as one matrix product over the unfolded image."""
    top, bottom, left, right = cd.pads
    filters, _, r, s = w.shape
    out = []
    for image in torch.nn.functional.pad(x, (left, right, top, bottom)):
        columns = torch.nn.functional.unfold(image[None], (r, s), stride=(cd.sr, cd.sc))[0]
        out.append(w.reshape(filters, -1) @ columns + (bias[:, None] if cd.use_bias else 0.0))
    rows = (x.shape[2] + top + bottom - r) // cd.sr + 1
    return torch.stack(out).reshape(x.shape[0], filters, rows, -1)


def _layer64(layer, ins, p):
    x, kind = ins[0], layer.kind
    if kind == "conv2d":
        return _conv64(x, p["K"], p["bias"], layer.attrs["cd"])
    if kind == "dense":
        return x @ p["W"] + p["bias"]
    if kind == "batchnorm":
        m, v, g, b = (p[k][None, :, None, None] for k in ("mean", "variance", "bn_g", "bn_b"))
        return (x - m) / torch.sqrt(v + layer.attrs["epsilon"]) * g + b
    if kind == "relu":
        return torch.relu(x)
    if kind == "maxpool2d":
        pd = layer.attrs["pd"]
        top, bottom, left, right = pd.pad
        return torch.nn.functional.max_pool2d(torch.nn.functional.pad(x, (left, right, top, bottom), value=-3.40282e38), pd.ksize, pd.stride)
    if kind == "avgpool2d":  # (the networks pool whole planes)
        return x.mean((2, 3), keepdim=True)
    if kind == "resize":
        fy, fx = layer.out_shape[2] // x.shape[2], layer.out_shape[3] // x.shape[3]
        return x.repeat_interleave(fy, 2).repeat_interleave(fx, 3)
    if kind == "concat":
        return torch.cat(ins, layer.attrs["axis"])
    if kind == "pad":
        top, right, bottom, left = layer.attrs["pads"]
        return torch.nn.functional.pad(x, (left, right, top, bottom), value=layer.attrs["constant"])
    if kind == "reshape":
        return x.reshape(x.shape[0], *layer.out_shape[1:])
    if kind == "softmax":
        return torch.softmax(x, layer.attrs["axis"])
    if kind == "sigmoid":
        return torch.sigmoid(x)
    if kind in ("sum", "add_n"):
        return sum(ins[1:], x)
    raise ValueError("no 64-bit form of layer kind " + kind)


def exact(case, seed):
    """What ``run`` returns for the parameters and inputs of ``prepare``, computed with torch in 64 bits.  The coordinates that
    the block's pool writes are choices, not computed numbers."""
    state = prepare(case, seed)
    net = state["net"]
    heads = [l for l in net.layers for c in l.children if c.kind in ("reshape", "softmax")]
    readers = {id(l): len(l.children) for l in net.layers}

    def forward(x):
        values, kept = {}, {}
        left = dict(readers)
        for layer in net.layers:
            if layer.kind == "input":
                y = x
            else:
                params = {k: _as_torch(t).double() for k, t in net.dparams.get(id(layer), {}).items()}
                y = _layer64(layer, [values[id(q)] for q in layer.parents], params)
                for q in layer.parents:
                    left[id(q)] -= 1
                    if left[id(q)] == 0:
                        del values[id(q)]
            values[id(layer)] = y
            if layer in net.lout or layer in heads:
                kept[id(layer)] = y.reshape(layer.out_shape)
        return kept

    if case["mode"] == "forward":
        kept = forward(_as_torch(state["x"]).double())
        return [kept[id(l)] for l in net.lout + heads] + [None] * (len(state["out"]) - len(net.lout + heads))
    outs = []
    for batch in state["batches"]:
        kept = forward(torch.from_numpy(batch).cuda().double())
        outs.append([kept[id(l)].cpu().numpy() for l in net.lout])
    return outs[0] if case["mode"] == "predict" else outs


def _work(case):
    """Flops of the convolutions and dense layers in the direct form; bytes: parameters, inputs and outputs of the network.
    A layer walk also hands every layer's output over in memory: written once and read once."""
    net = _graph(case)
    flops, floats = 0, 0
    for layer in net.layers:
        n_out = math.prod(layer.out_shape)
        floats += sum(v.size for v in layer.params.values())
        if layer.kind == "conv2d":
            flops += 2 * n_out * math.prod(layer.params["K"].shape[1:])
        elif layer.kind == "dense":
            flops += 2 * n_out * layer.params["W"].shape[0]
        if layer.kind == "input" or layer in net.lout:
            floats += n_out * (3 if layer.kind == "maxpool2d" else 1)  # with the two index tensors
        elif not case["fuse"] and layer.kind != "reshape":
            floats += 2 * n_out
    batches = 4 if case["mode"] == "stream" else 1
    return {"bytes": 4.0 * floats * batches, "flops": float(flops) * batches}


def work(case):
    return _work(case)


def tolerance(case):
    """About four times what the outputs of these cases move by when the same sums are taken in another order or form
    (one accumulator per output, matrix instructions, Winograd transforms; convolutions of up to 512 x 7 x 7 taps).  A softmax
    over a thousand classes and a U-Net of 23 layers amplify what a residual network's normalised layers do not."""
    return {"conv": {"rel": 1e-5, "max": 1e-4}, "block": {"rel": 2e-6, "max": 4e-5, "differ": 2e-5}, "vgg16": {"rel": 1.5e-5, "max": 8e-4},
            "resnet50": {"rel": 2e-6, "max": 1.5e-5}, "unet": {"rel": 4e-5, "max": 8e-4}}[case["model"]]
