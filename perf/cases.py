"""The calls that box convolution is timed and compared on: ``BoxConv2d`` as a program uses it.

A case names one layer call through the public entry points and its sizes. ``mode`` is

* ``train``        one training step of a layer inside a network: ``module(x)`` and ``backward``, all
                   five gradients;
* ``first_layer``  the same for a network's first layer, whose input needs no gradient;
* ``infer``        ``module.eval()`` and ``module(x)`` without autograd;
* ``fused``        the eval-mode tail of a bottleneck block in one call (``forward_fused``: batch norm
                   folded to scale and shift, residual add, ReLU).

Sizes: ``B`` batch, ``C`` input planes, ``F`` filters per plane, ``h`` x ``w`` pixels. The boxes are
the module's own seeded initialisation for an image of that size.
"""
import math
import os
import random
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "box-convolutions_amd"))

from box_convolution import BoxConv2d  # noqa: E402

DTYPES = {"float32": torch.float32, "bfloat16": torch.bfloat16, "float16": torch.float16}


def _case(mode, dtype, B, C, F, h, w, normalize=True, exact=True, name=None):
    case = {"mode": mode, "dtype": dtype, "B": B, "C": C, "F": F, "h": h, "w": w,
            "normalize": normalize, "exact": exact}
    if name is not None:
        case["name"] = name
    return case


def listed():
    return [
        # the MNIST example's layer: 40 filters on one 28 x 28 plane, batch 32. The smallest call:
        # launches, autograd and chains of dependent work, hardly any bytes
        _case("train", "float32", 32, 1, 40, 28, 28, name="train_mnist_28x28"),
        # the deep blocks of a segmentation encoder at 1/8 resolution: many narrow planes
        _case("train", "float32", 8, 64, 4, 64, 128, name="train_planes_64x128"),
        # a bottleneck block at 1/4 resolution, and the same in bfloat16 with a larger batch
        _case("train", "float32", 4, 32, 4, 128, 256, name="train_block_128x256"),
        _case("train", "bfloat16", 8, 32, 4, 128, 256, name="train_block_bf16_128x256"),
        # the full-resolution layer (the benchmark's default workload)
        _case("train", "float32", 2, 16, 8, 512, 1024, name="train_fullres_512x1024"),
        # a camera image, not a power of two
        _case("train", "float32", 1, 16, 8, 720, 1280, name="train_camera_720x1280"),
        # odd and ragged: rows that neither fill a wave nor start on aligned addresses; box sums
        # instead of averages (normalize=False)
        _case("train", "float32", 2, 8, 6, 301, 767, normalize=False, name="train_ragged_sums_301x767"),
        # the first layer of a network: colour images that need no gradient
        _case("first_layer", "float32", 8, 3, 16, 480, 640, name="first_layer_480x640"),
        # large images, two filters per plane: the largest listed case
        _case("train", "float32", 1, 128, 2, 1024, 2048, name="train_large_1024x2048"),
        # inference: full resolution in half precision; rounded boxes (exact=False, the fast mode) in
        # float32 on an odd size; a whole block tail
        _case("infer", "float16", 2, 16, 8, 512, 1024, name="infer_fp16_512x1024"),
        _case("infer", "float32", 4, 16, 8, 270, 481, exact=False, name="infer_rounded_270x481"),
        _case("fused", "bfloat16", 8, 32, 4, 128, 256, name="fused_tail_bf16_128x256"),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


# most output elements (B*C*F*h*w) and input elements a drawn case has: those of the largest listed one
_MOST_OUT, _MOST_IN = 128 * 2 * 1024 * 2048, 128 * 1024 * 2048


def draw(rng):
    mode = rng.choice(["train", "train", "train", "train", "first_layer", "infer", "infer", "fused"])
    dtype = rng.choice(["float32", "float32", "float32", "bfloat16", "float16"])
    h, w = _log_uniform(rng, 16, 1100), _log_uniform(rng, 16, 2048)
    if rng.random() < 0.4:                       # feature maps are often multiples of 8
        h, w = max(8, h // 8 * 8), max(8, w // 8 * 8)
    C = rng.randint(1, 4) if mode == "first_layer" else _log_uniform(rng, 1, 128)
    F = _log_uniform(rng, 1, 40)
    B = _log_uniform(rng, 1, 32)
    # down to a size that costs no more than the largest listed case, up to one that is a layer's work
    while B * C * F * h * w > _MOST_OUT // 2 or B * C * h * w > _MOST_IN // 2:
        if B > 1:
            B = (B + 1) // 2
        elif C > 1:
            C = (C + 1) // 2
        else:
            F = (F + 1) // 2
    while B * C * F * h * w < 1 << 18:
        B *= 2
    exact = not (mode in ("infer", "fused") and rng.random() < 0.4)
    return _case(mode, dtype, B, C, F, h, w, normalize=rng.random() < 0.8, exact=exact)


def _module(case, seed):
    kept = random.getstate()
    random.seed(seed)
    module = BoxConv2d(case["C"], case["F"], case["h"], case["w"], normalize=case["normalize"])
    random.setstate(kept)
    module.exact = case["exact"]
    return module.cuda()


def prepare(case, seed):
    B, C, F, h, w = (case[k] for k in "BCFhw")
    dtype, mode = DTYPES[case["dtype"]], case["mode"]
    gen = torch.Generator(device="cuda").manual_seed(seed)

    def normal(*shape):
        return torch.randn(*shape, generator=gen, device="cuda")

    module = _module(case, seed)
    if mode == "first_layer":
        # images, brought to mean 0 and deviation 1 as data loaders do
        x = ((torch.rand(B, C, h, w, generator=gen, device="cuda") - 0.5) * math.sqrt(12)).to(dtype)
    else:
        # what a batch norm leaves
        x = normal(B, C, h, w).to(dtype)
    state = {"mode": mode, "module": module, "x": x}
    if mode in ("train", "first_layer"):
        module.train()
        x.requires_grad_(mode == "train")
        state["grad"] = normal(B, C * F, h, w).to(dtype)
    else:
        module.eval()
        for p in module.parameters():
            p.requires_grad_(False)
    if mode == "fused":
        state["scale"] = 0.5 + torch.rand(C * F, generator=gen, device="cuda")
        state["shift"] = 0.1 * normal(C * F)
        state["residual"] = normal(B, C * F, h, w).clamp_(min=0).to(dtype)
    return state


def run(state):
    module, x = state["module"], state["x"]
    if state["mode"] == "fused":
        return module.forward_fused(x, channel_scale=state["scale"], channel_shift=state["shift"],
                                    residual=state["residual"], relu=True)
    if state["mode"] == "infer":
        with torch.no_grad():
            return module(x)
    x.grad = None
    for p in module.parameters():
        p.grad = None
    out = module(x)
    out.backward(state["grad"])
    result = {"out": out.detach(), "x_min": module.x_min.grad, "x_max": module.x_max.grad,
              "y_min": module.y_min.grad, "y_max": module.y_max.grad}
    if x.grad is not None:
        result["grad_input"] = x.grad
    return result


def work(case):
    n_in = case["B"] * case["C"] * case["h"] * case["w"]
    n_out = n_in * case["F"]
    elem = 4 if case["dtype"] == "float32" else 2
    mode = case["mode"]
    # input in, output out; then grad_output in and the gradient w.r.t. the input out; or the residual in
    elems = n_in + n_out
    flops = 2 * n_in + 12 * n_out                    # integral image; separable box sums
    if mode in ("train", "first_layer"):
        elems += n_out
        flops += 22 * n_out                          # the four bounds' derivatives
    if mode == "train":
        elems += n_in
        flops += 8 * n_out                           # the adjoint
    if mode == "fused":
        elems += n_out
        flops += 4 * n_out
    return {"bytes": elem * elems, "flops": flops}


def tolerance(case):
    # Measured against the same call with float64 tensors and parameters, over the listed cases and
    # 28 drawn ones; stated is about four times the worst relative error seen in any output:
    #   float32   1.5e-5 (a bound's gradient at 192 x 1384; outputs and input gradients up to 9e-6:
    #             1/area of boxes a fraction of a pixel thin)
    #   float16   2.1e-4 and bfloat16 1.7e-3: one rounding of the output or the input's gradient
    return {"rel": {"float32": 6e-5, "float16": 8e-4, "bfloat16": 7e-3}[case["dtype"]]}


def _overlap(lo, hi, n, dev):
    # [i, k]: how much of pixel k the box [i + lo, i + hi + 1] covers
    i = torch.arange(n, dtype=torch.float64, device=dev)[:, None]
    k = torch.arange(n, dtype=torch.float64, device=dev)[None, :]
    return (torch.minimum(i + hi + 1, k + 1) - torch.maximum(i + lo, k)).clamp_(min=0)


def _edge(offset, n, dev):
    # for each i the pixel i + offset an edge lies in, and whether there is such a pixel
    e = torch.arange(n, device=dev) + offset
    return e.clamp(0, n - 1), ((e >= 0) & (e < n)).double()


def _pixel_bounds(module, clip_to):
    """The box bounds in pixels, as float32 holds them, after the projection that a training-mode
    forward and ``eval()`` apply to the stored bounds."""
    bounds = []
    min_size = 1.001 if module.exact else 2.001
    for lo, hi, factor, size in ((module.x_min, module.x_max, module.reparametrization_h, clip_to[0]),
                                 (module.y_min, module.y_max, module.reparametrization_w, clip_to[1])):
        lo, hi = (p.detach().double().clamp(-(size + 1) / factor, (size - 1) / factor) for p in (lo, hi))
        gap = (min_size - 0.9999) / factor
        mean = (0.5 * (lo + hi)).float().double()
        thin = lo + gap > hi
        lo, hi = torch.where(thin, mean - 0.5 * gap, lo), torch.where(thin, mean + 0.5 * gap, hi)
        bounds += [(p.float() * factor).double() for p in (lo, hi)]
    return bounds


def exact(case, seed):
    """``run``'s outputs in float64: every box filter as two dense matrices of pixel overlaps."""
    state = prepare(case, seed)
    module, x = state["module"], state["x"].detach().double()
    B, C, F, h, w = (case[k] for k in "BCFhw")
    dev, train = x.device, state["mode"] in ("train", "first_layer")
    bounds = _pixel_bounds(module, (h, w))
    values = [b.cpu().tolist() for b in bounds]
    out = torch.empty(B, C * F, h, w, dtype=torch.float64, device=dev)
    grad_input = torch.zeros_like(x) if state["mode"] == "train" else None
    grads = [torch.zeros(C, F, dtype=torch.float64, device=dev) for _ in range(4)]
    for c in range(C):
        plane = x[:, c].contiguous()
        for f in range(F):
            x0, x1, y0, y1 = (v[c][f] for v in values)
            if not case["exact"]:
                x0, x1, y0, y1 = math.ceil(x0), math.floor(x1), math.ceil(y0), math.floor(y1)
            rows, cols = _overlap(x0, x1, h, dev), _overlap(y0, y1, w, dev)
            scale = 1 / ((x1 - x0 + 1) * (y1 - y0 + 1)) if case["normalize"] else 1.0
            across = torch.matmul(plane, cols.t().contiguous())
            result = torch.matmul(rows, across) * scale
            out[:, c * F + f] = result
            if not train:
                continue
            g = state["grad"][:, c * F + f].double()
            if grad_input is not None:
                grad_input[:, c] += torch.matmul(rows.t().contiguous(), torch.matmul(g, cols)) * scale
            down = torch.matmul(rows, plane)
            total = (g * result).sum()
            for n, (value, offset, sign, source, dim) in enumerate((
                    (x0, math.ceil(x0) - 1, -1, across, 1), (x1, math.floor(x1) + 1, 1, across, 1),
                    (y0, math.ceil(y0) - 1, -1, down, 2), (y1, math.floor(y1) + 1, 1, down, 2))):
                at, there = _edge(offset, source.size(dim), dev)
                there = there[:, None] if dim == 1 else there
                d = sign * scale * (g * source.index_select(dim, at) * there).sum()
                if case["normalize"]:
                    d = d - sign * total / ((x1 - x0 + 1) if dim == 1 else (y1 - y0 + 1))
                grads[n][c, f] = d * (module.reparametrization_h if dim == 1 else module.reparametrization_w)
    if state["mode"] == "fused":
        out = out * state["scale"].double().view(1, -1, 1, 1) + state["shift"].double().view(1, -1, 1, 1)
        return (out + state["residual"].double()).clamp_(min=0)
    if state["mode"] == "infer":
        return out
    result = {"out": out, "x_min": grads[0], "x_max": grads[1], "y_min": grads[2], "y_max": grads[3]}
    if grad_input is not None:
        result["grad_input"] = grad_input
    return result
