"""Forward with half-precision output and the fused tail (scale, shift, residual, ReLU).

The reference has no such function; what it computes is the reference's forward followed by
element-wise steps (how its BottleneckBoxConv ends in eval mode,
examples/Cityscapes/models/ENet.py:290-304). Expected values therefore come from the CPU oracle:
oracle integral image -> oracle forward -> scale / shift / residual / ReLU in float32 on the host
-> rounded to the output type on the host. Tolerances against the oracle: the forward's 1e-4 of the
largest entry, plus one unit in the last place of the half type for half-precision output. On top
of that the entry point is held much tighter to the library's own plain forward (a few float32
roundings; half precision: the float32 result rounded once), which pins the tail arithmetic itself.
"""
import numpy as np
import pytest
import torch

from box_convolution import BoxConv2d
from helpers import make_boxes

pytestmark = pytest.mark.gpu
DEV = "cuda"

# B, C, F, h, w: partial rows, full rows at 256 and 512 threads, three columns per lane, gather
SHAPES = [(2, 3, 4, 37, 53), (1, 2, 2, 64, 256), (1, 1, 2, 40, 1024), (1, 2, 1, 18, 1536),
          (1, 1, 1, 8, 2100), (3, 1, 5, 9, 64)]
HALF_ULP = {torch.float16: 2.0 ** -10, torch.bfloat16: 2.0 ** -7}


class OracleForward:
    """The reference's forward on the host for one test case (float32, numpy)."""

    def __init__(self, oracle, x, boxes):
        self.oracle = oracle
        self.boxes = boxes
        self.integ = oracle.integral_image(x)

    def __call__(self, normalize, exact):
        return self.oracle.box_forward(self.integ, *self.boxes, normalize, exact)


def setup_case(hip, shape, seed, kind="inside", oracle=None):
    B, C, F, h, w = shape
    rng = np.random.default_rng(seed)
    boxes_np = make_boxes(rng, C, F, h, w, kind)
    boxes = [torch.from_numpy(b).to(DEV) for b in boxes_np]
    g = torch.Generator(device="cpu").manual_seed(seed)
    x_host = torch.randn(B, C, h, w, generator=g)
    x = x_host.to(DEV)
    integ = hip.integral_image(x)
    scale = (torch.rand(C * F, generator=g) * 2 - 0.7).to(DEV)
    shift = torch.randn(C * F, generator=g).to(DEV)
    residual = torch.randn(B, C * F, h, w, generator=g).to(DEV)
    if oracle is None:
        return integ, boxes, scale, shift, residual
    return integ, boxes, scale, shift, residual, OracleForward(oracle, x_host.numpy(), boxes_np)


def compose_host(plain, scale, shift, residual, relu):
    """The tail in float32 on the host: numpy in, numpy out."""
    y = plain.astype(np.float32)
    if scale is not None:
        y = y * scale.cpu().numpy()[None, :, None, None]
    if shift is not None:
        y = y + shift.cpu().numpy()[None, :, None, None]
    if residual is not None:
        y = y + residual.float().cpu().numpy()
    return np.maximum(y, 0) if relu else y


def to_half_on_host(a, dtype):
    """float32 numpy -> torch tensor of a half type, rounded to nearest even on the host."""
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).to(dtype)


def compose(plain, scale, shift, residual, relu):
    y = plain
    if scale is not None:
        y = y * scale[None, :, None, None]
    if shift is not None:
        y = y + shift[None, :, None, None]
    if residual is not None:
        y = y + residual
    return torch.relu(y) if relu else y


@pytest.mark.parametrize("exact", [True, False])
@pytest.mark.parametrize("shape", SHAPES)
def test_fused_tail_float32(hip, oracle, shape, exact):
    integ, boxes, scale, shift, residual, ref = setup_case(hip, shape, 11, oracle=oracle)
    plain = hip.box_convolution_forward(integ, *boxes, True, exact)
    plain_c = ref(True, exact)
    # nothing to fuse: the very same numbers as the plain entry point, and the oracle's to 1e-4
    assert torch.equal(hip.box_convolution_forward_fused(integ, *boxes, True, exact), plain)
    assert np.abs(plain.cpu().numpy() - plain_c).max() <= 1e-4 * np.abs(plain_c).max()
    for use_scale, use_shift, use_res, relu in [(1, 1, 1, 1), (1, 0, 0, 0), (0, 1, 0, 0), (0, 0, 1, 0),
                                                (0, 0, 0, 1), (1, 1, 0, 1), (0, 0, 1, 1)]:
        args = (scale if use_scale else None, shift if use_shift else None,
                residual if use_res else None, bool(relu))
        got = hip.box_convolution_forward_fused(integ, *boxes, True, exact, torch.float32, *args)
        want = compose(plain, *args)
        # sizes of the terms that get rounded
        mag = (plain.abs() * (scale.abs().max() if use_scale else 1)).max().item() + 4.0
        assert (got - want).abs().max().item() <= 4e-7 * mag, (use_scale, use_shift, use_res, relu)
        # against the oracle's forward with the tail applied on the host
        want_c = compose_host(plain_c, *args)
        assert np.abs(got.cpu().numpy() - want_c).max() <= 1e-4 * mag, (use_scale, use_shift, use_res, relu)
        if relu:
            assert got.min().item() >= 0


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("shape", SHAPES)
def test_half_precision_output(hip, oracle, shape, dtype):
    integ, boxes, scale, shift, residual, ref = setup_case(hip, shape, 23, kind="hanging", oracle=oracle)
    for normalize in (True, False):
        plain = hip.box_convolution_forward(integ, *boxes, normalize, True)
        got = hip.box_convolution_forward_fused(integ, *boxes, normalize, True, dtype)
        assert got.dtype == dtype and got.shape == plain.shape
        # against the oracle's forward rounded to the half type on the host: the forward's 1e-4
        # of the largest entry plus one unit in the last place of the half type
        plain_c = ref(normalize, True)
        want_c = to_half_on_host(plain_c, dtype).float().numpy()
        ok = np.isfinite(want_c)
        assert np.array_equal(np.isfinite(got.float().cpu().numpy()), ok)
        err = np.abs(got.float().cpu().numpy()[ok] - plain_c[ok])
        assert np.all(err <= HALF_ULP[dtype] * np.abs(plain_c[ok]) + 1e-4 * np.abs(plain_c[ok]).max())
        # (float16 overflows to inf where the unnormalized sums exceed 65504, as .to() does)
        want = plain.to(dtype)
        # The kernel may round the product sum * (1/area) to the half type in one step
        # (mixed-precision multiply); where the float32 product is a tie between two half
        # values that differs from rounding twice, and is then the closer one.
        assert (got != want).float().mean().item() < 1e-3
        finite = want.float().isfinite()
        assert torch.equal(got.float().isfinite(), finite)
        assert torch.all(((got.float() - plain).abs() <= (want.float() - plain).abs() * (1 + 1e-6))[finite])
    plain = hip.box_convolution_forward(integ, *boxes, True, True)
    res16 = residual.to(dtype)
    got = hip.box_convolution_forward_fused(integ, *boxes, True, True, dtype, scale, shift, res16, True)
    want = compose(plain, scale, shift, res16.float(), True)
    err = (got.float() - want).abs()
    bound = HALF_ULP[dtype] * want.abs().clamp_min(2.0 ** -14) + 1e-6
    assert torch.all(err <= bound)
    # and nearly all entries are the correctly rounded value of the float32 composition
    assert (got != want.to(dtype)).float().mean().item() < 0.02
    # the same against the oracle: forward on the host, tail on the host, rounded on the host
    want_c = compose_host(ref(True, True), scale, shift, res16, True)
    mag = (np.abs(ref(True, True)).max() * scale.abs().max().item()) + 4.0
    err_c = np.abs(got.float().cpu().numpy() - want_c)
    assert np.all(err_c <= HALF_ULP[dtype] * np.abs(want_c) + 1e-4 * mag)
    assert (got.cpu() != to_half_on_host(want_c, dtype)).float().mean().item() < 0.05


# planes, h, w: single pass (full rows), two passes (partial rows, vector and element loads),
# one band, 64 bands, wider than the direct path reads
HALF_INTEGRAL_SHAPES = [(3, 96, 256), (2, 130, 1024), (2, 70, 2048), (3, 200, 36), (1, 300, 1023),
                        (2, 100, 1000), (5, 9, 17), (40, 33, 257), (1, 2048, 64), (1, 12, 2500)]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("planes,h,w", HALF_INTEGRAL_SHAPES)
def test_integral_image_of_half_precision_input(hip, switches, planes, h, w, dtype):
    """float32 integral image straight from float16 / bfloat16: the same bits as converting the
    input to float32 first (which is pinned against the oracle in test_gpu_parity.py)."""
    x = (torch.randn(planes, h, w, device=DEV) * 3 + 0.5).to(dtype)
    want = hip.integral_image(x.float())
    got = hip.integral_image(x)
    assert got.dtype == torch.float32 and torch.equal(got, want)
    # an odd start address (no 8-byte alignment): element-wise loads
    flat = torch.empty(x.numel() + 1, device=DEV, dtype=dtype)
    shifted = flat[1:].view_as(x).copy_(x)
    assert shifted.data_ptr() % 8 != 0 and torch.equal(hip.integral_image(shifted), want)
    switches("BOXCONV_INTEGRAL_LOOKBACK", "2")     # single pass wherever it applies
    assert torch.equal(hip.integral_image(x), hip.integral_image(x.float()))


def test_argument_checks(hip):
    integ, boxes, scale, shift, residual = setup_case(hip, (1, 2, 2, 8, 8), 3)
    with pytest.raises(RuntimeError, match="float32 integral image"):
        hip.box_convolution_forward_fused(integ.double(), *boxes, True, True)
    with pytest.raises(RuntimeError, match="float32, float16 or bfloat16"):
        hip.box_convolution_forward_fused(integ, *boxes, True, True, torch.float64)
    with pytest.raises(RuntimeError, match="must hold 4 values"):
        hip.box_convolution_forward_fused(integ, *boxes, True, True, torch.float32, scale[:3])
    with pytest.raises(RuntimeError, match="shape of the output"):
        hip.box_convolution_forward_fused(integ, *boxes, True, True, torch.float32, None, None,
                                          residual[:, :3])


def make_module(C, F, h, w, seed):
    import random
    random.seed(seed)
    return BoxConv2d(C, F, h, w).to(DEV)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def oracle_module_forward(oracle, m, x_host):
    """The reference's BoxConv2d.forward on the host for module `m` (its stored parameters)."""
    stored = [p.detach().cpu().numpy() for p in (m.x_min, m.x_max, m.y_min, m.y_max)]
    out, _ = oracle.module_forward(np.ascontiguousarray(x_host, dtype=np.float32), *stored,
                                   m.reparametrization_h, m.reparametrization_w, m.normalize, m.exact)
    return out


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_module_takes_half_precision_input(oracle, dtype):
    m = make_module(3, 4, 40, 72, 5).eval()
    x = torch.randn(2, 3, 40, 72, device=DEV).to(dtype)
    with torch.no_grad():
        got = m(x)
        want = m(x.float())
    assert got.dtype == dtype and (got != want.to(dtype)).float().mean().item() < 1e-3
    assert torch.allclose(got.float(), want, rtol=HALF_ULP[dtype], atol=1e-7)
    # the oracle on the same (half-precision) input values, rounded to the half type on the host
    want_c = oracle_module_forward(oracle, m, x.float().cpu().numpy())
    err = np.abs(got.float().cpu().numpy() - want_c)
    assert np.all(err <= HALF_ULP[dtype] * np.abs(want_c) + 1e-4 * np.abs(want_c).max())
    # with autograd: float32 in between, gradients come back in the input's type
    m.train()
    xg = x.clone().requires_grad_(True)
    out = m(xg)
    assert out.dtype == dtype and out.requires_grad
    go = torch.randn_like(out)
    out.backward(go)
    x32 = x.float().requires_grad_(True)
    ref_grads = torch.autograd.grad(m(x32), [x32, m.x_min, m.y_max], go.float())
    assert xg.grad.dtype == dtype
    assert torch.allclose(xg.grad.float(), ref_grads[0], rtol=2 * HALF_ULP[dtype], atol=1e-3)
    assert torch.allclose(m.x_min.grad, ref_grads[1], rtol=1e-4, atol=1e-4 * ref_grads[1].abs().max().item())
    assert torch.allclose(m.y_max.grad, ref_grads[2], rtol=1e-4, atol=1e-4 * ref_grads[2].abs().max().item())


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_bottleneck_tail_in_one_launch(oracle, dtype):
    """BoxConv2d -> BatchNorm2d -> Dropout2d -> + x -> ReLU in eval mode, as the reference's
    BottleneckBoxConv ends (ENet.py:290-304), against the same chain of torch modules."""
    C, F, h, w = 4, 4, 32, 64
    m = make_module(C, F, h, w, 9).eval()
    bn = torch.nn.BatchNorm2d(C * F).to(DEV)
    with torch.no_grad():
        bn.running_mean.normal_()
        bn.running_var.uniform_(0.5, 2.0)
        bn.weight.normal_()
        bn.bias.normal_()
    bn.eval()
    drop = torch.nn.Dropout2d(0.25).eval()
    x = torch.randn(2, C, h, w, device=DEV)
    skip = torch.randn(2, C * F, h, w, device=DEV).to(dtype)
    with torch.no_grad():
        want = torch.relu(skip.float() + drop(bn(m(x))))
        scale, shift = BoxConv2d.fold_batch_norm(bn)
        got = m.forward_fused(x.to(dtype), scale, shift, skip, relu=True)
        want_in = torch.relu(skip.float() + drop(bn(m(x.to(dtype).float()))))
    assert got.dtype == dtype
    if dtype == torch.float32:
        assert torch.allclose(got, want, rtol=1e-5, atol=1e-5)
    else:
        assert torch.all((got.float() - want_in).abs() <= HALF_ULP[dtype] * want_in.abs() + 1e-5)
    # the oracle's box convolution, then BatchNorm (eval) + residual + ReLU written out on the host
    conv_c = oracle_module_forward(oracle, m, x.to(dtype).float().cpu().numpy())
    g, b = bn.weight.detach().cpu().numpy(), bn.bias.detach().cpu().numpy()
    mu, var = bn.running_mean.cpu().numpy(), bn.running_var.cpu().numpy()
    y = (conv_c - mu[None, :, None, None]) / np.sqrt(var + bn.eps)[None, :, None, None]
    want_c = np.maximum(y * g[None, :, None, None] + b[None, :, None, None] + skip.float().cpu().numpy(), 0)
    err = np.abs(got.float().cpu().numpy() - want_c)
    ulp = HALF_ULP[dtype] if dtype != torch.float32 else 0.0
    assert np.all(err <= ulp * np.abs(want_c) + 1e-4 * (np.abs(want_c).max() + 4.0))


def test_forward_fused_modes_and_double_input():
    """forward_fused follows the module's normalize / exact switches and takes float64 input
    (integrated in float32, as the entry point works on a float32 integral image)."""
    m = make_module(2, 3, 24, 40, 21).eval()
    x = torch.randn(2, 2, 24, 40, device=DEV)
    for normalize, exact in ((True, True), (False, True), (True, False), (False, False)):
        m.normalize, m.exact = normalize, exact
        with torch.no_grad():
            want = m(x)
        assert torch.equal(m.forward_fused(x), want)
        got = m.forward_fused(x.double(), output_dtype=torch.float32)
        assert torch.allclose(got, want, rtol=1e-5, atol=1e-5)
    assert not m.forward_fused(x).requires_grad


@pytest.mark.parametrize("exact", [True, False])
@pytest.mark.parametrize("tail", [False, True])
@pytest.mark.parametrize("dtype,h,w", [
    # one wave: three eighths of the lanes, an odd number of rows, all lanes
    (torch.float32, 9, 96), (torch.float32, 35, 100), (torch.float32, 40, 252), (torch.float32, 12, 256),
    (torch.bfloat16, 17, 132), (torch.float16, 8, 256),
    # 16-bit rows of several waves
    (torch.float16, 21, 512), (torch.bfloat16, 11, 1000), (torch.float16, 10, 1280), (torch.bfloat16, 7, 1284),
    (torch.float16, 9, 2048)])
def test_forward_with_consecutive_columns(switches, dtype, h, w, tail, exact):
    """The forward kernel with four consecutive columns per lane against the one with wave-strided
    columns (BOXCONV_FWD_QUADS=2, whatever the size, and =0): the same expressions per pixel, so at most the contraction of a
    product and a sum differs, a unit in the last place of float32 or one rounding to 16 bits.
    Boxes hang over every edge; without a residual the output's memory holds NaN beforehand."""
    from box_convolution import _native as hip
    gen = torch.Generator().manual_seed(h * w)
    B, C, F = 2, 2, 3
    x = torch.randn(B, C, h, w, generator=gen).cuda().to(dtype)
    lo_x, lo_y = ((torch.rand(C, F, generator=gen) * 2 - 1.2) * n for n in (h, w))
    boxes = [t.cuda() for t in (lo_x, lo_x + 2.2 + torch.rand(C, F, generator=gen) * h,
                                lo_y, lo_y + 2.2 + torch.rand(C, F, generator=gen) * w)]
    integ = hip.integral_image(x)
    variants = [(None, None, None, False)]
    if tail:
        scale, shift = torch.rand(C * F, generator=gen).cuda(), torch.randn(C * F, generator=gen).cuda()
        residual = torch.randn(B, C * F, h, w, generator=gen).cuda().to(dtype)
        variants = [(scale, shift, residual, True), (scale, None, None, True)]
    for args in variants:
        results = []
        for variant in ("2", "0"):
            switches("BOXCONV_FWD_QUADS", variant)
            filler = torch.full((B, C * F, h, w), float("nan"), device="cuda", dtype=dtype)
            del filler                                   # (the allocator hands this block out next)
            hip.profile_arm("forward_quads")
            results.append(hip.box_convolution_forward_fused(integ, *boxes, True, exact, dtype, *args).float())
            assert hip.profile_collect()[1] == (variant == "2" and (tail or w != 1284 and w != 2048))
        a, b = results
        assert torch.isfinite(a).all()
        unit = {torch.float32: 2.0 ** -20, torch.float16: 2.0 ** -10, torch.bfloat16: 2.0 ** -7}[dtype]
        assert ((a - b).abs() <= unit * b.abs() + 1e-6 * b.abs().max()).all()


@pytest.mark.parametrize("exact", [True, False])
@pytest.mark.parametrize("tail", [False, True])
@pytest.mark.parametrize("name,dtype,h,w", [
    # several rows side by side in a wave: 8, 16 and 32 lanes per row, whole and with a last lane that shares columns
    ("forward_narrow", torch.float32, 28, 28), ("forward_narrow", torch.float16, 9, 16), ("forward_narrow", torch.bfloat16, 130, 17),
    ("forward_narrow", torch.float32, 3, 23), ("forward_narrow", torch.float32, 40, 33), ("forward_narrow", torch.float16, 64, 64),
    ("forward_narrow", torch.bfloat16, 37, 63), ("forward_narrow", torch.float32, 65, 65), ("forward_narrow", torch.bfloat16, 70, 96),
    ("forward_narrow", torch.float16, 21, 127), ("forward_narrow", torch.float32, 200, 128),
    # rows of a wave and more that are no multiple of four columns
    ("forward_quads", torch.float32, 17, 129), ("forward_quads", torch.bfloat16, 12, 255), ("forward_quads", torch.float16, 11, 257),
    ("forward_quads", torch.float32, 9, 514), ("forward_quads", torch.bfloat16, 13, 767), ("forward_quads", torch.float32, 7, 1021),
    ("forward_quads", torch.float16, 8, 2047)])
def test_forward_of_narrow_and_odd_rows(switches, name, dtype, h, w, tail, exact):
    """The forward kernels for rows of at most 128 columns (BOXCONV_NARROW=2) and for rows that are no multiple
    of four columns (BOXCONV_FWD_QUADS=2) against the one with wave-strided columns (BOXCONV_FWD_QUADS=0): the
    same expressions per pixel, so at most the contraction of a product and a sum differs, or one rounding to
    16 bits. Boxes hang over every edge; the output's memory holds NaN beforehand."""
    from box_convolution import _native as hip
    gen = torch.Generator().manual_seed(h * w)
    B, C, F = 2, 3, 2
    x = torch.randn(B, C, h, w, generator=gen).cuda().to(dtype)
    lo_x, lo_y = ((torch.rand(C, F, generator=gen) * 2 - 1.2) * n for n in (h, w))
    boxes = [t.cuda() for t in (lo_x, lo_x + 2.2 + torch.rand(C, F, generator=gen) * h,
                                lo_y, lo_y + 2.2 + torch.rand(C, F, generator=gen) * w)]
    integ = hip.integral_image(x)
    variants = [(None, None, None, False)]
    if tail:
        scale, shift = torch.rand(C * F, generator=gen).cuda(), torch.randn(C * F, generator=gen).cuda()
        residual = torch.randn(B, C * F, h, w, generator=gen).cuda().to(dtype)
        variants = [(scale, shift, residual, True), (scale, None, None, True)]
    for args in variants:
        results = []
        for variant in ("2", "0"):
            switches("BOXCONV_NARROW" if name == "forward_narrow" else "BOXCONV_FWD_QUADS", "2" if variant == "2" else None)
            if variant == "0":
                switches("BOXCONV_FWD_QUADS", "0")
            filler = torch.full((B, C * F, h, w), float("nan"), device="cuda", dtype=dtype)
            del filler                                   # (the allocator hands this block out next)
            hip.profile_arm(name)
            results.append(hip.box_convolution_forward_fused(integ, *boxes, True, exact, dtype, *args).float())
            assert hip.profile_collect()[1] == (variant == "2")
            switches("BOXCONV_FWD_QUADS", None)
        a, b = results
        assert torch.isfinite(a).all()
        unit = {torch.float32: 2.0 ** -20, torch.float16: 2.0 ** -10, torch.bfloat16: 2.0 ** -7}[dtype]
        assert ((a - b).abs() <= unit * b.abs() + 1e-6 * b.abs().max()).all()


def test_tail_without_residual_loads_none():
    """Scale, shift and ReLU alone move half the bytes of the same tail with a residual (a load of
    something else in its place, thrown away, would take as long). Kernel times at a size that no
    cache holds: 91 against 153 us."""
    from box_convolution import _native as hip
    B, C, F, h, w = 2, 16, 8, 512, 1024
    integ = hip.integral_image(torch.randn(B, C, h, w, device="cuda").half())
    lo = torch.full((C, F), -20.25, device="cuda")
    scale, shift = torch.rand(C * F, device="cuda"), torch.randn(C * F, device="cuda")
    residual = torch.randn(B, C * F, h, w, device="cuda").half()
    times = {}
    for name, res in (("with", residual), ("without", None), ("with", residual), ("without", None)):
        hip.profile_arm("forward_quads")
        for _ in range(5):
            hip.box_convolution_forward_fused(integ, lo, -lo, lo, -lo, True, True, torch.float16, scale, shift, res, True)
        ms, launches = hip.profile_collect()
        assert launches == 5
        times[name] = min(times.get(name, ms), ms)
    assert times["without"] < 0.85 * times["with"]


@pytest.mark.parametrize("dtype,planes,F,h,w", [
    # a residual of 128 MB and more is read with the streaming policy: one, two, four, five waves per row
    (torch.float32, 140, 1, 1001, 244), (torch.bfloat16, 37, 4, 900, 508), (torch.float16, 9, 8, 923, 1020),
    (torch.bfloat16, 7, 8, 955, 1276)])
def test_large_residual(switches, dtype, planes, F, h, w):
    from box_convolution import _native as hip
    gen = torch.Generator(device="cuda").manual_seed(w)
    integ = hip.integral_image(torch.randn(1, planes, h, w, generator=gen, device="cuda"))
    lo_x, lo_y = (-torch.rand(planes, F, generator=gen, device="cuda") * n for n in (h, w))
    boxes = (lo_x, lo_x + 3 + h // 3, lo_y, lo_y + 3 + w // 3)
    scale, shift = (torch.randn(planes * F, generator=gen, device="cuda") for _ in range(2))
    residual = torch.randn(1, planes * F, h, w, generator=gen, device="cuda").to(dtype)
    assert residual.numel() * residual.element_size() > 128 << 20
    results = []
    for variant in (None, "0"):
        switches("BOXCONV_FWD_QUADS", variant)
        results.append(hip.box_convolution_forward_fused(integ, *boxes, True, True, dtype, scale, shift, residual, True))
    a, b = (r.float() for r in results)
    # the same expressions per pixel: one contraction of a product and a sum, or one rounding to 16 bits
    unit = {torch.float32: 2.0 ** -20, torch.float16: 2.0 ** -10, torch.bfloat16: 2.0 ** -7}[dtype]
    assert ((a - b).abs() <= unit * b.abs() + 1e-6 * b.abs().max()).all()


@pytest.mark.parametrize("quads,dtype,planes,h,w,tail", [
    # 96 to 127 columns from 2^21 pixels on where narrow_forward_kernel does not take them, never 128; 129 to 192 below
    # 2^22; above with a residual
    (False, torch.float32, 19, 59, 96, None), (False, torch.float32, 219, 100, 96, None),
    (True, torch.float32, 160, 1000, 112, "relu"), (True, torch.float32, 310, 1000, 112, "residual"),
    (False, torch.float32, 219, 100, 128, None), (True, torch.float32, 100, 200, 192, None),
    (False, torch.float32, 150, 200, 160, None), (True, torch.float32, 150, 200, 160, "residual"),
    (False, torch.bfloat16, 150, 200, 160, None),
    # float32 rows that start on 64-byte boundaries, and others
    (True, torch.float32, 90, 200, 224, None), (False, torch.float32, 110, 200, 224, None),
    (True, torch.float32, 110, 200, 224, "relu"), (True, torch.float32, 110, 200, 220, None),
    (True, torch.bfloat16, 110, 200, 224, None), (True, torch.float32, 512, 128, 256, None),
    # 256 MB and more of output and integral images
    (False, torch.float32, 140, 1000, 256, None), (False, torch.float32, 262, 1000, 256, None), (False, torch.float32, 600, 1000, 112, None),
    (True, torch.float32, 320, 1000, 212, None)])
def test_consecutive_columns_only_where_they_pay(quads, dtype, planes, h, w, tail):
    """Rows of one wave: which forward kernel takes them, by columns and output pixels."""
    from box_convolution import _native as hip
    integ = hip.integral_image(torch.randn(1, planes, h, w, device="cuda"))
    lo = torch.full((planes, 1), -3.25, device="cuda")
    residual = torch.randn(1, planes, h, w, device="cuda").to(dtype) if tail == "residual" else None
    hip.profile_arm("forward_quads")
    hip.box_convolution_forward_fused(integ, lo, -lo, lo, -lo, True, True, dtype, None, None, residual, tail == "relu")
    assert hip.profile_collect()[1] == quads


@pytest.mark.parametrize("narrow,dtype,planes,h,w,tail", [
    # up to 32 columns and 16-bit outputs always; float32 while output and integral images fit the memory-side cache,
    # with a tail always; 96 to 124 columns in a multiple of four with a tail while they take less than half of it
    (False, torch.float32, 64, 100, 15, None), (True, torch.float32, 2100, 600, 28, None), (True, torch.float32, 300, 100, 60, None),
    (False, torch.float32, 1400, 400, 60, None), (True, torch.float32, 1400, 400, 60, "relu"), (True, torch.bfloat16, 1400, 400, 64, None),
    (True, torch.float32, 219, 100, 96, None), (False, torch.float32, 310, 1000, 112, None), (True, torch.float32, 120, 1000, 112, "relu"),
    (False, torch.float32, 160, 1000, 112, "relu"), (False, torch.float32, 160, 1000, 112, "residual"),
    (True, torch.float32, 160, 1000, 111, "relu"), (True, torch.bfloat16, 500, 1000, 112, "residual"), (False, torch.bfloat16, 8, 100, 129, None)])
def test_narrow_forward_only_where_it_pays(narrow, dtype, planes, h, w, tail):
    """Rows of at most 128 columns: which launches take the kernel with several of them in a wave."""
    from box_convolution import _native as hip
    integ = hip.integral_image(torch.randn(1, planes, h, w, device="cuda"))
    lo = torch.full((planes, 1), -3.25, device="cuda")
    residual = torch.randn(1, planes, h, w, device="cuda").to(dtype) if tail == "residual" else None
    hip.profile_arm("forward_narrow")
    hip.box_convolution_forward_fused(integ, lo, -lo, lo, -lo, True, True, dtype, None, None, residual, tail == "relu")
    assert hip.profile_collect()[1] == narrow


@pytest.mark.parametrize("quads,C,F,h,w", [
    (True, 64, 16, 270, 481), (False, 64, 15, 270, 481), (True, 190, 16, 100, 301), (False, 200, 16, 99, 301),
    (True, 300, 4, 350, 255), (True, 16, 4, 270, 481)])
def test_large_odd_forward_by_filters(quads, C, F, h, w):
    """float32 rows of more than 256 columns that the memory-side cache does not hold: four consecutive columns per
    lane where many filters read the same integral rows."""
    from box_convolution import _native as hip
    integ = hip.integral_image(torch.randn(1, C, h, w, device="cuda"))
    lo = torch.full((C, F), -3.25, device="cuda")
    hip.profile_arm("forward_quads")
    hip.box_convolution_forward_fused(integ, lo, -lo, lo, -lo, True, True, torch.float32, None, None, None, False)
    assert hip.profile_collect()[1] == quads


@pytest.mark.parametrize("dtype,h,w", [(torch.float32, 130, 252), (torch.bfloat16, 40, 512)])
def test_residual_at_any_offset(switches, dtype, h, w):
    """A residual that does not start on four elements takes the kernel with wave-strided columns and
    returns what that kernel returns for an aligned copy, bit for bit."""
    from box_convolution import _native as hip
    planes = 8
    integ = hip.integral_image(torch.randn(1, planes, h, w, device="cuda"))
    lo = torch.full((planes, 1), -3.25, device="cuda")
    aligned = torch.randn(1, planes, h, w, device="cuda").to(dtype)
    shifted = torch.empty(aligned.numel() + 1, device="cuda", dtype=dtype)[1:].view_as(aligned).copy_(aligned)
    assert shifted.data_ptr() % (4 * shifted.element_size()) != 0

    def forward(residual):
        return hip.box_convolution_forward_fused(integ, lo, -lo, lo, -lo, True, True, dtype, None, None, residual, True)
    hip.profile_arm("forward_quads")
    got = forward(shifted)
    assert hip.profile_collect()[1] == 0
    hip.profile_arm("forward_quads")
    forward(aligned)
    assert hip.profile_collect()[1] == 1
    switches("BOXCONV_FWD_QUADS", "0")
    assert torch.equal(got, forward(aligned))


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("h,w", [(40, 28), (64, 64), (33, 128)])
def test_narrow_rows_with_a_residual_at_any_offset(dtype, h, w):
    """Rows of at most 128 columns in a multiple of four whose residual or (through the C entry point) output does not
    start on four elements: accesses that need aligned elements only, the same result bit for bit."""
    from box_convolution import _native as hip
    B, C, F = 4, 16, 3
    integ = hip.integral_image(torch.randn(B, C, h, w, device="cuda"))
    lo = torch.full((C, F), -3.25, device="cuda")
    residual = torch.randn(B, C * F, h, w, device="cuda").to(dtype)
    lib = hip.load()

    def at_odd_element(t):
        return torch.empty(t.numel() + 1, device="cuda", dtype=dtype)[1:].view_as(t).copy_(t)

    def forward(res, out, name):
        hip.profile_arm(name)
        assert lib.boxconv_forward_fused_f32(
            integ.data_ptr(), lo.data_ptr(), (-lo).data_ptr(), lo.data_ptr(), (-lo).data_ptr(), out.data_ptr(),
            hip._FUSED_OUTPUT[dtype], None if res is None else res.data_ptr(), None, None, 1, B, C, F, h, w, 1, 1,
            torch.cuda.current_stream().cuda_stream) == 0
        assert hip.profile_collect()[1] == 1
        return out

    for res in (residual, None):
        want = forward(res, torch.empty_like(residual), "forward_narrow")
        shifted = at_odd_element(residual)
        if res is not None:
            assert torch.equal(forward(shifted, torch.empty_like(residual), "forward_narrow_unaligned"), want)
        assert torch.equal(forward(res, at_odd_element(residual), "forward_narrow_unaligned"), want)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("h,w", [
    # rows that are no multiple of four columns: a last wave with a single lane in use, whose neighbour is in another
    # wave (257 to 259, 513, 770, 1025 columns), and with more; several rows in a wave; whole quads; one element per lane
    (37, 257), (38, 258), (41, 259), (33, 513), (30, 770), (29, 1025), (36, 301), (70, 129), (33, 31), (24, 127), (40, 64),
    (30, 256), (21, 512), (20, 2100)])
def test_residual_in_the_memory_of_the_output(dtype, h, w):
    """The C entry point adds a residual in place: every pixel is read and written by one lane. The result is that of
    a residual elsewhere, bit for bit."""
    from box_convolution import _native as hip
    B, C, F = 2, 6, 3
    gen = torch.Generator().manual_seed(h * w)
    integ = hip.integral_image(torch.randn(B, C, h, w, generator=gen).cuda())
    lo_x, lo_y = ((torch.rand(C, F, generator=gen) * 2 - 1.2) * n for n in (h, w))
    boxes = [t.cuda() for t in (lo_x, lo_x + 2.2 + torch.rand(C, F, generator=gen) * h,
                                lo_y, lo_y + 2.2 + torch.rand(C, F, generator=gen) * w)]
    scale, shift = torch.rand(C * F, generator=gen).cuda(), torch.randn(C * F, generator=gen).cuda()
    residual = torch.randn(B, C * F, h, w, generator=gen).cuda().to(dtype)
    want = hip.box_convolution_forward_fused(integ, *boxes, True, True, dtype, scale, shift, residual, True)
    lib = hip.load()
    stream = torch.cuda.current_stream().cuda_stream
    for _ in range(5):
        both = residual.clone()
        assert lib.boxconv_forward_fused_f32(
            integ.data_ptr(), *[b.data_ptr() for b in boxes], both.data_ptr(), hip._FUSED_OUTPUT[dtype], both.data_ptr(),
            scale.data_ptr(), shift.data_ptr(), 1, B, C, F, h, w, 1, 1, stream) == 0
        assert torch.equal(both, want)
