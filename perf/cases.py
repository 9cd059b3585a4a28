"""The work whose speed counts: what programs on this package have it do, from one digit to a training step of the deep
shape network, each case one pass through the public entry points.

`listed()` names the cases, `draw(rng)` gives more of the same ranges, `prepare` makes what a program holds before the
call (inputs and models on the GPU, from a seed), `run` is the pass, `work` what the pass cannot do without and
`tolerance` how far another correct float32 implementation may be off.
"""
import math

import torch

import s2cnn_amd
from s2cnn_amd import harness
from s2cnn_amd.soft.so3_fft import SO3_fft_real, SO3_ifft_real

# Bandwidths, features and input size of the networks: (first layer on the sphere, then layers on SO(3)).
NETWORKS = {
    "digits": {"bands": (30, 10, 6), "features": (1, 20, 40), "classes": 10},
    "shapes": {"bands": (64, 16, 10), "features": (6, 100, 100), "classes": 55},
    "shapes_original": {"bands": (128, 32, 22, 7), "features": (6, 50, 70, 350), "classes": 55},
    "deep": {"bands": (128, 32, 22, 7), "features": (6, 100, 100, 55), "classes": None},
}


def listed():
    return [
        # one digit classified as it arrives: the smallest call, where launches and the host's work count
        {"name": "digits_infer_1", "kind": "network", "net": "digits", "train": False, "batch": 1},
        # the digit network's evaluation pass at its usual batch
        {"name": "digits_infer_32", "kind": "network", "net": "digits", "train": False, "batch": 32},
        # forward and backward of the digit network: a training step without the optimizer's update
        {"name": "digits_train_32", "kind": "network", "net": "digits", "train": True, "batch": 32},
        # the shape network's training step, normalisations inside the transforms
        {"name": "shapes_train_32", "kind": "network", "net": "shapes", "train": True, "batch": 32},
        # evaluation of the shape network's first published form: 50, 70 and 350 features, maximum over the grid
        {"name": "shapes_original_infer_16", "kind": "network", "net": "shapes_original", "train": False, "batch": 16},
        # the deep shape network's forward and backward pass with the activations inside the layers: the largest case
        {"name": "deep_train_32", "kind": "network", "net": "deep", "train": True, "batch": 32},
        # one wide layer at full bandwidth, forward and backward: what most of a big model's time goes to
        {"name": "layer_b32_64to64", "kind": "layer", "batch": 16, "f_in": 64, "f_out": 64, "b_in": 32, "b_out": 32},
        # a layer whose sizes divide nothing: odd features and batch, a bandwidth without a power of two
        {"name": "layer_b18to13_33to45", "kind": "layer", "batch": 11, "f_in": 33, "f_out": 45, "b_in": 18, "b_out": 13},
        # a first layer on the sphere, forward and backward down to the signal (saliency maps), sizes that divide nothing
        {"name": "sphere_b50to20_3to26", "kind": "sphere", "batch": 9, "f_in": 3, "f_out": 26, "b_in": 50, "b_out": 20},
        # signals to spectra and back at full bandwidth: filtering and smoothing of signals on SO(3)
        {"name": "transform_256_b32", "kind": "transform", "volumes": 256, "b": 32, "b_spec": 32},
        # the same for few volumes of an odd bandwidth with a truncated spectrum
        {"name": "transform_50_b27to19", "kind": "transform", "volumes": 50, "b": 27, "b_spec": 19},
        # the complex product of two spectra with both gradients, for programs that keep their signals in the spectral domain
        {"name": "product_b32_64to64", "kind": "product", "nl": 32, "batch": 16, "f_in": 64, "f_out": 64},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49))))))


def draw(rng):
    while True:
        kind = rng.choice(["network", "network", "layer", "layer", "sphere", "transform", "product"])
        if kind == "network":
            net = rng.choice(["digits", "digits", "shapes", "shapes_original", "deep"])
            case = {"kind": kind, "net": net, "train": net == "deep" or (net != "shapes_original" and rng.random() < 0.6),
                    "batch": _log_int(rng, 1, {"digits": 64, "shapes": 32, "shapes_original": 16, "deep": 32}[net])}
        elif kind == "transform":
            b = rng.randint(4, 32)
            case = {"kind": kind, "volumes": _log_int(rng, 1, 1024), "b": b, "b_spec": rng.randint(max(2, b // 3), b)}
        elif kind == "product":
            case = {"kind": kind, "nl": rng.randint(4, 32), "batch": _log_int(rng, 1, 32), "f_in": _log_int(rng, 2, 100),
                    "f_out": _log_int(rng, 2, 100)}
        else:
            b = _log_int(rng, 8, 128) if kind == "sphere" else rng.randint(4, 32)
            case = {"kind": kind, "batch": _log_int(rng, 1, 32), "f_in": _log_int(rng, 1, 8) if kind == "sphere" else _log_int(rng, 2, 100),
                    "f_out": _log_int(rng, 4, 100), "b_in": b, "b_out": rng.randint(max(2, b // 4), min(b, 32))}
        if _cost(case) <= _cost(listed()[11 if kind == "product" else 6]):
            return case


def _cost(case):
    w = work(case)
    return w["flops"] / 1e14 + w["bytes"] / 3e12 if case["kind"] != "network" else 0.0


# ---------------------------------------------------------------------------------------------------------------------
def _near_identity_so3(b_in):
    """The 192-point grid around the identity, its size scaled with the resolution of the input as the shape networks do."""
    return s2cnn_amd.so3_near_identity_grid(max_beta=math.pi / 8 * min(1.0, 30 / b_in), max_gamma=2 * math.pi, n_alpha=8, n_beta=3, n_gamma=8)


def _near_identity_s2(b_in):
    return s2cnn_amd.s2_near_identity_grid(max_beta=math.pi / 8 * min(1.0, 30 / b_in), n_alpha=8, n_beta=3)


def _network(net):
    if net == "digits":
        return harness.S2ConvNet_original()
    if net == "shapes":
        return harness.Shrec17Model(55, fused_norm=True)
    if net == "shapes_original":
        return harness.Shrec17ModelOriginal(55)
    d = NETWORKS["deep"]
    b, f = d["bands"], d["features"]
    layers = [s2cnn_amd.S2Convolution(f[0], f[1], b[0], b[1], _near_identity_s2(b[0]), activation="relu"),
              s2cnn_amd.SO3Convolution(f[1], f[2], b[1], b[2], _near_identity_so3(b[1]), activation="relu"),
              s2cnn_amd.SO3Convolution(f[2], f[3], b[2], b[3], _near_identity_so3(b[2]))]
    return torch.nn.Sequential(*layers)


def prepare(case, seed):
    torch.manual_seed(seed)
    dev = torch.device("cuda", torch.cuda.current_device())
    g = torch.Generator(device=dev).manual_seed(seed)
    kind = case["kind"]
    if kind == "network":
        net = case["net"]
        d = NETWORKS[net]
        n, c, b = case["batch"], d["features"][0], d["bands"][0]
        if net == "digits":        # projected digits: most of the sphere is empty
            x = torch.rand(n, c, 2 * b, 2 * b, device=dev, generator=g) * (torch.rand(n, c, 2 * b, 2 * b, device=dev, generator=g) < 0.3)
        else:                      # ray-cast depths and normals: smooth, with fine structure on top
            x = harness.smooth_spherical_batch(n, c, b, dev, seed=seed)
        model = _network(net).to(dev)
        model.train(case["train"])
        state = {"model": model, "x": x}
        if net == "deep":
            state["grad_out"] = torch.randn(n, d["features"][-1], device=dev, generator=g)
        elif case["train"]:
            state["labels"] = torch.randint(0, d["classes"], (n,), device=dev, generator=g)
        return state
    if kind in ("layer", "sphere"):
        dims = 3 if kind == "layer" else 2
        b_in, b_out = case["b_in"], case["b_out"]
        make = s2cnn_amd.SO3Convolution if kind == "layer" else s2cnn_amd.S2Convolution
        grid = _near_identity_so3(b_in) if kind == "layer" else _near_identity_s2(b_in)
        layer = make(case["f_in"], case["f_out"], b_in, b_out, grid).to(dev)
        x = torch.randn(case["batch"], case["f_in"], *(2 * b_in,) * dims, device=dev, generator=g)
        x.requires_grad_()         # a layer inside a network: its input needs a gradient too
        return {"model": layer, "x": x, "grad_out": torch.randn(case["batch"], case["f_out"], *(2 * b_out,) * 3, device=dev, generator=g)}
    if kind == "transform":
        return {"x": torch.randn(case["volumes"], *(2 * case["b"],) * 3, device=dev, generator=g), "b": case["b"], "b_spec": case["b_spec"]}
    ns, n, fi, fo = _nspec(case["nl"]), case["batch"], case["f_in"], case["f_out"]
    x = torch.randn(ns, n, fi, 2, device=dev, generator=g)
    y = torch.randn(ns, fi, fo, 2, device=dev, generator=g) / math.sqrt(fi)
    return {"x": x.requires_grad_(), "y": y.requires_grad_(), "grad_out": torch.randn(ns, n, fo, 2, device=dev, generator=g)}


def run(state):
    if "model" in state:
        model, x = state["model"], state["x"]
        if "grad_out" in state:                      # forward, then backward from a gradient that is given
            out = model(x)
            if isinstance(model, torch.nn.Sequential):
                out = s2cnn_amd.so3_integrate(out)
            leaves = ([x] if x.requires_grad else []) + list(model.parameters())
            return [out.detach(), *torch.autograd.grad(out, leaves, state["grad_out"])]
        if "labels" in state:
            out = model(x)
            loss = torch.nn.functional.cross_entropy(out, state["labels"])
            grads = torch.autograd.grad(loss, list(model.parameters()))
            # A batch normalisation takes the mean off again, so the bias of a layer in front of one has no gradient: what
            # comes out for it is rounding and nothing to compare.
            normed = getattr(model, "fused_norm", None) is not None
            return [out.detach(), loss.detach(), *(gr for gr in grads if not (normed and gr.dim() == 5))]
        with torch.no_grad():
            return model(x)
    if "y" in state:
        z = s2cnn_amd.so3_mm(state["x"], state["y"])
        return [z.detach(), *torch.autograd.grad(z, (state["x"], state["y"]), state["grad_out"])]
    with torch.no_grad():
        spec = SO3_fft_real.apply(state["x"], state["b_spec"])
        return [spec, SO3_ifft_real.apply(spec, state["b"])]


# ---------------------------------------------------------------------------------------------------------------------
def _nspec(b):
    return b * (4 * b * b - 1) // 3


def _block_product(nl, n, fi, fo):
    """Multiply-adds of the products of (2l+1) x (2l+1) blocks over all degrees."""
    return n * fi * fo * nl * nl * (2 * nl * nl - 1)


def _so3_transform(n, b, b_spec):
    """Flops of n transforms of real signals: FFTs of the 2b planes and, per spectral entry of half the spectrum, a sum over
    the 2b planes (half of them by the mirror symmetry in beta)."""
    return n * (2.5 * (2 * b) ** 3 * math.log2((2 * b) ** 2) + 2.0 * _nspec(min(b, b_spec)) / 2 * 2 * b)


def _s2_transform(n, b, b_spec):
    return n * (2.5 * (2 * b) ** 2 * math.log2(2 * b) + 2.0 * min(b, b_spec) ** 2 / 2 * 2 * b)


def _layer_flops(first, n, fi, fo, b_in, b_out, backward):
    """Forward, and as often again for the gradients asked for (backward: 0, 1 = weights only, 2 = weights and input)."""
    product = 2.0 * (n * fi * fo * _nspec(b_out) if first else _block_product(b_out, n, fi, fo))
    into = _s2_transform(n * fi, b_in, b_out) if first else _so3_transform(n * fi, b_in, b_out)
    out = _so3_transform(n * fo, b_out, b_out)
    return product * (1 + backward) + into * (2 if backward == 2 else 1) + out * (2 if backward else 1)


def work(case):
    kind = case["kind"]
    if kind == "network":
        d, n = NETWORKS[case["net"]], case["batch"]
        b, f, back = d["bands"], d["features"], case["train"]
        flops = sum(_layer_flops(i == 0, n, f[i], f[i + 1], b[i], b[i + 1], 0 if not back else 1 if i == 0 else 2) for i in range(len(f) - 1))
        points = [24 if i == 0 else 192 for i in range(len(f) - 1)] if case["net"] in ("digits", "deep") else [2 * v for v in b[:-1]]
        weights = sum(f[i] * f[i + 1] * points[i] + f[i + 1] for i in range(len(f) - 1))
        return {"bytes": 4.0 * (n * f[0] * (2 * b[0]) ** 2 + weights * (2 if back else 1) + n * f[-1]), "flops": flops}
    if kind in ("layer", "sphere"):
        n, fi, fo, b_in, b_out = (case[k] for k in ("batch", "f_in", "f_out", "b_in", "b_out"))
        signal = n * fi * (2 * b_in) ** (3 if kind == "layer" else 2)
        kernel = fi * fo * (192 if kind == "layer" else 24)
        return {"bytes": 8.0 * (signal + kernel + n * fo * (2 * b_out) ** 3), "flops": _layer_flops(kind == "sphere", n, fi, fo, b_in, b_out, 2)}
    if kind == "transform":
        n, b, bs = case["volumes"], case["b"], case["b_spec"]
        return {"bytes": 8.0 * n * (2 * b) ** 3 + 8.0 * n * _nspec(bs), "flops": 2 * _so3_transform(n, b, bs)}
    nl, n, fi, fo = case["nl"], case["batch"], case["f_in"], case["f_out"]
    # three products; a complex multiply-add from three real ones
    return {"bytes": 16.0 * _nspec(nl) * (n * fi + fi * fo + n * fo), "flops": 3 * 6.0 * _block_product(nl, n, fi, fo)}


def tolerance(case):
    """About four times what this path differs by from itself on complex spectra (other products, sums in another order) and
    from 64-bit sums.  Forward passes and transforms 1e-7 to 3e-7; gradients, long sums of terms of both signs, up to 2.6e-6.
    Where an activation sits on a sample next to zero the sample counts or not: up to 8e-6.  Behind batch normalisations what
    is left of a gradient is small against the sums it is the difference of: 9e-5."""
    if case["kind"] == "network":
        return {"rel": {"shapes": 3e-4}.get(case["net"], 3e-5)} if case["train"] else {"rel": 1e-6}
    return {"rel": 1e-6} if case["kind"] == "transform" else {"rel": 1e-5}
