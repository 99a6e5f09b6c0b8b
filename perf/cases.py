"""The work that this framework does for its users, as measurable cases.

Four kinds of work, each through the public entry points:

* ``layer``: one ``DepthwiseOrientedConv1d`` of any size, forward only or forward and backward.
* ``stages``: the four oriented convolutions that a network holds at its four stage extents,
  forward and backward: the block convolutions on C channels (NCHW) or the second convolutions of
  the 1D++ blocks on 4 C channels (NHWC, residual tap), at the batch and image size asked for.
* ``stem``: the two stride-2 convolutions of the stem (NHWC), forward and backward.
* ``network``: a whole ConvNeXt-1D or ConvNeXt-1D++: inference, a training pass under bf16
  autocast with fp32 master weights, or the four stage outputs of a dense-prediction backbone
  with their backward pass.

Sizes are those of the repository's benchmark, its tests and its network definitions.
"""
import math

import torch

from oriented1d_amd import DepthwiseOrientedConv1d
from oriented1d_amd.convnext1d import channel_angles, convnext_base_1d, convnext_tiny_1d

_DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
_DIMS = {"tiny": (96, 192, 384, 768), "base": (128, 256, 512, 1024)}
_DEPTHS = {"tiny": (3, 3, 9, 3), "base": (3, 3, 27, 3)}
_CLASSES = 1000


def _layer(N, C, H, W, K, stride=1, dtype="f32", layout="nchw", angles="network", mode="train"):
    return {"kind": "layer", "N": N, "C": C, "H": H, "W": W, "K": K, "stride": stride,
            "dtype": dtype, "layout": layout, "angles": angles, "mode": mode}


def _stages(size, N, H, W, dtype, hidden=False, cropped=False, angles="network"):
    return {"kind": "stages", "size": size, "N": N, "H": H, "W": W, "dtype": dtype,
            "hidden": hidden, "cropped": cropped, "angles": angles}


def _stem(N, H, W, K, dtype):
    return {"kind": "stem", "N": N, "H": H, "W": W, "K": K, "dtype": dtype}


def _network(size, variant, form, N, H, W):
    return {"kind": "network", "size": size, "variant": variant, "form": form, "N": N, "H": H, "W": W}


def listed():
    cases = {
        # a single small layer at inference: latency, the configuration a CPU can run as well
        "layer_small_forward": _layer(2, 96, 56, 56, 31, angles="round_robin", mode="forward"),
        # the headline sweep (batch 64, K = 31, eight orientations round-robin), as training sees it
        "stages_f32": _stages("tiny", 64, 224, 224, "f32", angles="round_robin"),
        "stages_bf16": _stages("tiny", 64, 224, 224, "bf16", angles="round_robin"),
        # the second convolutions of ConvNeXt-B-1D++ at its training batch: the largest launches
        "hidden_bf16_nhwc": _stages("base", 64, 224, 224, "bf16", hidden=True),
        # the reference's own layer benchmark (512 channels, fp32), with angles of any value
        "layer_any_angle": _layer(64, 512, 28, 28, 31, angles="any"),
        # the stem of a training step
        "stem_bf16": _stem(64, 224, 224, 31, "bf16"),
        # dense prediction at 512 x 512: stage maps of 128, 64, 32 and 16 squared
        "dense_stages_bf16": _stages("tiny", 8, 512, 512, "bf16", cropped=True),
        # a detection-sized image that no power of two divides, kernels cropped per stage
        "ragged_stages_f32": _stages("tiny", 2, 600, 904, "f32", cropped=True),
        # classification of one image: launches and host time
        "infer_one": _network("tiny", "1d", "infer", 1, 224, 224),
        # batched inference, the images-per-second figure
        "infer_batch": _network("tiny", "1d", "infer", 128, 224, 224),
        # the ConvNeXt-B-1D++ training pass
        "train_base_1dpp": _network("base", "1dpp", "train", 64, 224, 224),
        # dense features, forward and backward at 512 x 512
        "features_512": _network("tiny", "1d", "features", 8, 512, 512),
    }
    return [dict(case, name=name) for name, case in cases.items()]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _image(rng, lo, hi):
    """An image extent: a multiple of 32 in most programs, any number in some."""
    v = _log(rng, lo, hi)
    return max(lo, v // 32 * 32) if rng.random() < 0.7 else v


def draw(rng):
    pick = rng.random()
    dtype = rng.choice(["f32", "f32", "f32", "bf16", "bf16", "bf16", "f16"])
    angles = rng.choice(["network", "network", "network", "round_robin", "any"])
    if pick < 0.45:
        if rng.random() < 0.5:
            H = W = max(4, _image(rng, 128, 640) // rng.choice([4, 8, 16, 32]))
        else:
            H, W = _log(rng, 5, 160), _log(rng, 5, 160)
        p = rng.random()
        if p < 0.6:
            C = rng.choice([64, 96, 128, 192, 256, 384, 512, 768, 1024, 1536, 2048])
        elif p < 0.85:
            C = 8 * _log(rng, 1, 64)
        else:
            C = rng.randint(3, 520)
        most = 48 << 20
        N = min(_log(rng, 1, 64), max(1, most // (C * H * W)))
        return _layer(N, C, H, W, rng.choice([7, 13, 15, 27, 31, 31]),
                      rng.choice([1, 1, 1, 1, 1, 1, 2, 2, 4]), dtype,
                      rng.choice(["nchw", "nchw", "nhwc"]), angles,
                      rng.choice(["train", "train", "forward"]))
    if pick < 0.7:
        H = _image(rng, 128, 768)
        W = H if rng.random() < 0.5 else _image(rng, 128, 768)
        hidden = rng.random() < 0.35
        size = rng.choice(["tiny", "base"])
        elems = _DIMS[size][0] * (4 if hidden else 1) * H * W // 16
        N = min(_log(rng, 1, 64), max(1, (96 << 20) // elems))
        return _stages(size, N, H, W, dtype, hidden, rng.random() < 0.5, angles)
    if pick < 0.8:
        H, W = _image(rng, 128, 512), _image(rng, 128, 512)
        N = min(_log(rng, 2, 64), max(1, (3 << 20) // (H * W)))
        return _stem(N, H, W, rng.choice([15, 31]), rng.choice(["f32", "bf16"]))
    form = rng.choice(["infer", "infer", "train", "features"])
    H = _image(rng, 128, 512)
    W = H if form == "train" or rng.random() < 0.5 else _image(rng, 128, 512)
    if form != "features":  # classification images: whole multiples of the network's stride
        H, W = max(128, H // 32 * 32), max(128, W // 32 * 32)
    most = max(1, (1 << 20) // (H * W)) * (4 if form == "infer" else 1)
    return _network(rng.choice(["tiny", "tiny", "base"]), rng.choice(["1d", "1dpp"]), form,
                    min(_log(rng, 1, 64), most), H, W)


# ------------------------------------------------------------------------------------ sizes
def _stage_convs(case):
    """(N, C, H, W, K, nhwc) of the four convolutions of a ``stages`` case.  The stem halves an
    extent twice, rounding up; every further stage halves it rounding down (a 2 x 2 convolution
    of stride 2)."""
    h, w = -(-case["H"] // 4), -(-case["W"] // 4)
    ks = (31, 31, 27, 13) if case["cropped"] else (31,) * 4
    out = []
    for C, K in zip(_DIMS[case["size"]], ks):
        out.append((case["N"], C * (4 if case["hidden"] else 1), h, w, K, case["hidden"]))
        h, w = h // 2, w // 2
    return out


def _element_bytes(dtype):
    return 4 if dtype == "f32" else 2


def _conv_work(N, C, H, W, K, stride, dtype, mode):
    """Forward reads x and writes y; the backward pass reads x and dy and writes dx."""
    xs, ys, b = N * C * H * W, N * C * -(-H // stride) * -(-W // stride), _element_bytes(dtype)
    if mode == "forward":
        return (xs + ys) * b, 2.0 * ys * K
    return (3 * xs + 2 * ys) * b, 6.0 * ys * K


def _network_work(case):
    """Parameters, images and outputs once; every block reads and writes the residual stream.
    Training repeats the products twice in the backward pass and writes a gradient for each
    parameter."""
    dims, depths, N = _DIMS[case["size"]], _DEPTHS[case["size"]], case["N"]
    pp, train = case["variant"] == "1dpp", case["form"] != "infer"
    H, W = case["H"], case["W"]
    h, w = -(-H // 4), -(-W // 4)
    macs = 3.0 * 64 * H * W + 64.0 * 31 * (H * W / 4 + h * w) + 64.0 * dims[0] * h * w
    params, stream = 64.0 * (4 + 2 * 32 + dims[0]), 0.0
    for i, (C, depth) in enumerate(zip(dims, depths)):
        if i:
            h, w = h // 2, w // 2
            macs += 4.0 * dims[i - 1] * C * h * w
            params += 4.0 * dims[i - 1] * C
        macs += depth * h * w * (8.0 * C * C + C * (15 + 4 * 31 if pp else 31))
        params += depth * (8.0 * C * C + 45.0 * C + (128.0 * C if pp else 0.0))
        stream += depth * 2.0 * C * h * w
    if case["form"] != "features":
        macs += dims[3] * _CLASSES
        params += dims[3] * _CLASSES
    pb = 4 if case["form"] == "train" else 2
    act = N * (3.0 * H * W + stream) * 2
    return {"bytes": params * pb * (2 if train else 1) + act * (3 if train else 1),
            "flops": 2.0 * macs * N * (3 if train else 1)}


def work(case):
    kind = case["kind"]
    if kind == "network":
        return _network_work(case)
    if kind == "layer":
        convs = [(case["N"], case["C"], case["H"], case["W"], case["K"], case["stride"], case["mode"])]
    elif kind == "stages":
        convs = [(N, C, h, w, K, 1, "train") for N, C, h, w, K, _ in _stage_convs(case)]
    else:
        H, W = case["H"], case["W"]
        convs = [(case["N"], 64, H, W, case["K"], 2, "train"),
                 (case["N"], 64, -(-H // 2), -(-W // 2), case["K"], 2, "train")]
    got = [_conv_work(N, C, H, W, K, s, case["dtype"], mode) for N, C, H, W, K, s, mode in convs]
    return {"bytes": float(sum(g[0] for g in got)), "flops": float(sum(g[1] for g in got))}


# ------------------------------------------------------------------------------------ running
def _angles(kind, C, layer_offset, gen):
    if kind == "network":
        return channel_angles(C, layer_offset=layer_offset)
    if kind == "round_robin":
        return [(c % 8) * math.pi / 8 for c in range(C)]
    return torch.rand(C, device="cuda", generator=gen).mul_(math.pi).tolist()


def _conv(gen, N, C, H, W, K, stride, dtype, nhwc, angles, layer_offset=0.0, resid=False, train=True):
    """A layer with N(0, 0.02) weights and N(0, 1) activations and upstream gradient."""
    m = DepthwiseOrientedConv1d(C, C, K, groups=C, stride=stride, padding=K // 2, bias=True,
                                angle=_angles(angles, C, layer_offset, gen), nhwc=nhwc, resid=resid,
                                arbitrary_size=True).to("cuda")
    with torch.no_grad():
        m.weight.copy_(torch.randn(m.weight.shape, device="cuda", generator=gen) * 0.02)
        m.bias.copy_(torch.randn(C, device="cuda", generator=gen))
    P, Q = -(-H // stride), -(-W // stride)
    dt = _DTYPES[dtype]

    def tensor(h, w):
        return torch.randn((N, h, w, C) if nhwc else (N, C, h, w), device="cuda", generator=gen).to(dt)

    x = tensor(H, W).requires_grad_(train)
    return {"layer": m, "x": x, "dy": tensor(P, Q) if train else None}


_BUILDERS = {"tiny": convnext_tiny_1d, "base": convnext_base_1d}


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    kind = case["kind"]
    if kind == "layer":
        return {"convs": [_conv(gen, case["N"], case["C"], case["H"], case["W"], case["K"],
                                case["stride"], case["dtype"], case["layout"] == "nhwc",
                                case["angles"], train=case["mode"] == "train")]}
    if kind == "stages":
        return {"convs": [_conv(gen, N, C, h, w, K, 1, case["dtype"], nhwc, case["angles"], 0.0, nhwc)
                          for N, C, h, w, K, nhwc in _stage_convs(case)]}
    if kind == "stem":
        H, W = case["H"], case["W"]
        return {"convs": [_conv(gen, case["N"], 64, h, w, case["K"], 2, case["dtype"], True, "network",
                                off) for h, w, off in ((H, W, 0.0), (-(-H // 2), -(-W // 2), 0.5))]}
    torch.manual_seed(seed)
    form = case["form"]
    # (layer scales of a trained network, about 0.1 to 1, instead of the initial 1e-6 under which no
    # block would show in the outputs)
    with torch.device("cuda"):
        net = _BUILDERS[case["size"]](variant=case["variant"], num_classes=_CLASSES,
                                      layer_scale_init_value=0.1, arbitrary_size=True,
                                      out_stages=form == "features")
    images = torch.randn(case["N"], 3, case["H"], case["W"], device="cuda", generator=gen)
    if form == "train":
        labels = torch.randint(0, _CLASSES, (case["N"],), device="cuda", generator=gen)
        return {"form": form, "net": net.train(), "images": images, "labels": labels}
    net, images = net.to(torch.bfloat16), images.to(torch.bfloat16)
    if form == "infer":
        return {"form": form, "net": net.eval(), "images": images}
    targets, h, w = [], -(-case["H"] // 4), -(-case["W"] // 4)
    for C in _DIMS[case["size"]]:
        targets.append(torch.randn(case["N"], C, h, w, device="cuda", generator=gen))
        h, w = h // 2, w // 2
    return {"form": form, "net": net.train(), "images": images, "targets": targets}


def _flat_gradients(net):
    """The gradients as flat buckets, one for the oriented convolutions and one for each of the
    network's parts, as a data-parallel exchange or a flat optimizer takes them."""
    buckets = {}
    for name, p in net.named_parameters():
        if p.grad is not None:
            part = "oriented" if "dwconv" in name or ".dw" in name else ".".join(name.split(".")[:2])
            buckets.setdefault(part, []).append(p.grad.reshape(-1))
    return {part: torch.cat(grads) for part, grads in buckets.items()}


def run(state):
    if "convs" in state:
        out = []
        for c in state["convs"]:
            m, x = c["layer"], c["x"]
            if c["dy"] is None:
                with torch.no_grad():
                    out.append(m(x))
                continue
            y = m(x)
            out.append((y.detach(),) + torch.autograd.grad(y, (x, m.weight, m.bias), c["dy"]))
        return out
    net, form = state["net"], state["form"]
    if form == "infer":
        with torch.no_grad():
            return net(state["images"])
    for p in net.parameters():
        p.grad = None
    if form == "train":
        with torch.autocast("cuda", dtype=torch.bfloat16):
            logits = net(state["images"]).float()
            loss = torch.nn.functional.cross_entropy(logits, state["labels"])
        loss.backward()
        return {"logits": logits.detach(), "loss": loss.detach(), "gradients": _flat_gradients(net)}
    outs = net(state["images"])
    loss = sum((o.float() * r).sum() for o, r in zip(outs, state["targets"]))
    loss.backward()
    return {"features": [o.detach() for o in outs], "gradients": _flat_gradients(net)}


def tolerance(case):
    """Relative errors, about four times what was measured against the same pass in 64 bits
    (layers, stages and stem: 2e-7 to 4e-7 with fp32 tensors, 1.6e-3 to 2.2e-3 with 16-bit ones) or,
    for the bf16 networks, against the same weights in fp32 (logits 3.5e-3 at inference, gradients
    0.5e-2 to 1.2e-2)."""
    if case["kind"] == "network":
        return {"rel": 1.5e-2} if case["form"] == "infer" else {"rel": 3e-2}
    return {"rel": 1e-5} if case["dtype"] == "f32" else {"rel": 1e-2}
