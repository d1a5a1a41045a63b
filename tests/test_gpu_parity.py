"""HIP kernels vs the CPU oracle on identical seeded inputs, through the C ABI (ctypes).

Tolerances: forward and grad_input max|gpu-cpu|/max|cpu| <= 1e-4, box-parameter gradients <= 1e-3
for float32 (the targets the build is held to); 1e-9 for float64.
"""
import os

import numpy as np
import pytest
import torch

from helpers import make_boxes, param_grad_floor, rel_err

pytestmark = pytest.mark.gpu

TOL = {np.float32: (1e-4, 1e-3), np.float64: (1e-9, 1e-9)}


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def host(t):
    return t.detach().cpu().numpy()


# planes, h, w: chosen to hit one band / several bands, one wave / four waves, vector / scalar
# loads, several column tiles.
INTEGRAL_SHAPES = [
    (1, 2, 2), (3, 5, 7), (2, 10, 10), (6, 28, 28), (1, 33, 257), (2, 64, 128), (1, 200, 36),
    (1, 300, 1023), (2, 130, 1024), (1, 70, 2048), (1, 40, 2500), (1, 36, 4100), (1, 9, 9000),
    (2, 100, 4096), (1, 170, 3000),                     # sixteen waves per row, several bands
    (5, 1, 1), (2, 1, 300), (2, 300, 1),
    # single-pass kernel: many bands, partial last band, 64 bands, one band too many for it
    (3, 512, 1000), (1, 2048, 64), (1, 2100, 40), (40, 100, 520), (9, 97, 1536),
]


# (the single-pass kernel is float32 only)
@pytest.mark.parametrize("dtype,single_pass", [(np.float32, "where_faster"), (np.float64, "where_faster"),
                                               (np.float32, "wherever_possible")])
@pytest.mark.parametrize("planes,h,w", INTEGRAL_SHAPES)
def test_integral_image(hip, oracle, switches, planes, h, w, dtype, single_pass):
    if single_pass == "wherever_possible":
        # by default that kernel serves only the shapes it is faster on; reach the others too
        switches("BOXCONV_INTEGRAL_LOOKBACK", "2")
    rng = np.random.default_rng(planes * 1000003 + h * 1009 + w)
    x = (rng.random((planes, h, w)) * 2 - 0.5).astype(dtype)
    got = host(hip.integral_image(dev(x)))
    want = oracle.integral_image(x)
    assert got.shape == want.shape
    # closed form: float64 cumulative sums (the reference's own test oracle, test.py:12-35)
    exact = np.zeros((planes, h + 1, w + 1))
    exact[:, 1:, 1:] = x.astype(np.float64).cumsum(1).cumsum(2)
    assert np.all(got[:, 0, :] == 0) and np.all(got[:, :, 0] == 0)
    tol = 1e-6 if dtype == np.float32 else 1e-13
    assert rel_err(got, exact) <= tol
    assert rel_err(got, want) <= 10 * tol
    if dtype == np.float32:
        # sums are carried in double and rounded once: (almost) every entry is the correctly
        # rounded exact sum, and none is off by more than one unit in the last place
        ideal = exact.astype(np.float32)
        assert np.mean(got != ideal) < 1e-4
        assert np.all(np.abs(got - ideal) <= np.spacing(np.abs(ideal)))


@pytest.mark.parametrize("planes,h,w", [(1, 33, 257), (3, 200, 36), (2, 130, 1024), (2, 512, 1000),
                                        (1, 2048, 64), (17, 96, 2048)])
def test_integral_image_single_pass_waits_are_bounded(hip, switches, planes, h, w):
    """The single-pass kernel waits a bounded number of polls for the bands above; a band whose
    flag is still down is summed from the input instead. With a limit of zero polls every band
    goes that way, and the result is the same bit for bit. So is the three-launch path's."""
    x = torch.from_numpy(np.random.default_rng(h * w).random((planes, h, w), dtype=np.float32) - 0.3).cuda()
    switches("BOXCONV_INTEGRAL_LOOKBACK", "2")       # single pass for every shape it covers
    usual = hip.integral_image(x)
    for limit in ("0", "1", "2"):     # never wait / give up at once: a mix of both ways per launch
        switches("BOXCONV_INTEGRAL_SPIN", limit)
        assert torch.equal(hip.integral_image(x), usual)
    switches("BOXCONV_INTEGRAL_SPIN", None)
    switches("BOXCONV_INTEGRAL_LOOKBACK", "0")       # same bands, three launches
    three = hip.integral_image(x)
    switches("BOXCONV_INTEGRAL_LOOKBACK", None)
    # (the default may cut the planes into different bands: same sums, associated differently)
    assert torch.allclose(three, usual, rtol=2e-7, atol=0) and torch.allclose(hip.integral_image(x), usual, rtol=2e-7, atol=0)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("planes,h,w", [(5, 1, 1), (3, 5, 7), (6, 28, 28), (2, 64, 128), (40, 64, 128), (3, 8, 256),
                                        (2, 9, 255), (4, 57, 100), (3, 128, 256), (2, 129, 33), (7, 135, 240),
                                        (2, 192, 256), (3, 191, 254), (2, 170, 3), (1, 100, 253)])
def test_integral_image_plane_per_workgroup(hip, switches, planes, h, w, dtype):
    """Planes of at most 192 rows and 256 columns are scanned by one workgroup each (a wave per
    band of 8 to 24 rows, the bands' column sums handed over through LDS);
    BOXCONV_INTEGRAL_PLANE=0 sends them through the launches that larger planes take (other bands:
    the same sums, associated differently). Both against float64 cumulative sums."""
    x = torch.from_numpy(np.random.default_rng(planes + 7 * h + 1000 * w).random((planes, h, w), dtype=np.float32)
                         * 4 - 1).cuda().to(dtype)
    exact = torch.zeros(planes, h + 1, w + 1, dtype=torch.float64, device="cuda")
    exact[:, 1:, 1:] = x.double().cumsum(1).cumsum(2)
    got = hip.integral_image(x)
    assert got.dtype == torch.float32 and got.shape == exact.shape
    ideal = exact.float()
    assert torch.all((got - ideal).abs() <= torch.from_numpy(np.spacing(np.abs(ideal.cpu().numpy()))).cuda())
    assert (got != ideal).float().mean().item() < 1e-4
    switches("BOXCONV_INTEGRAL_PLANE", "0")
    two_launches = hip.integral_image(x)
    switches("BOXCONV_INTEGRAL_PLANE", None)
    assert torch.allclose(got, two_launches, rtol=2e-7, atol=0)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("planes,h,w", [(3, 28, 28), (5, 64, 128), (2, 100, 64), (4, 33, 256), (3, 64, 1024), (2, 40, 2048)])
def test_integral_image_of_a_misaligned_tensor(hip, planes, h, w, dtype):
    """A contiguous tensor whose first element is not 16-byte aligned (a view into a larger
    buffer) takes the kernels' element-wise loads instead of the 16-byte ones, and small planes
    other bands; the sums are the same."""
    for shift in (1, 3):
        flat = torch.randn(planes * h * w + shift, device="cuda").to(dtype)
        x = flat[shift:].view(planes, h, w)
        assert x.is_contiguous() and x.data_ptr() % 16 != 0
        assert torch.allclose(hip.integral_image(x), hip.integral_image(x.clone()), rtol=2e-7, atol=0)


INT_TYPES = [(np.uint8, torch.uint8), (np.int8, torch.int8), (np.int16, torch.int16),
             (np.int32, torch.int32), (np.int64, torch.int64)]


@pytest.mark.parametrize("np_dtype,torch_dtype", INT_TYPES)
@pytest.mark.parametrize("shape", [(1, 1, 1), (3, 5, 7), (2, 33, 257), (1, 70, 2500), (2, 2, 130, 1024), (1, 300, 3)])
def test_integral_image_of_integer_tensors(hip, oracle, shape, np_dtype, torch_dtype):
    """Integer tensors (src/integral_image.cpp:14): bit-exact against the oracle and against
    numpy's wrapping cumulative sums, with values over the type's full range."""
    rng = np.random.default_rng(sum(shape) + np.dtype(np_dtype).itemsize)
    info = np.iinfo(np_dtype)
    x = rng.integers(info.min, info.max, size=shape, dtype=np_dtype, endpoint=True)
    got = hip.integral_image(torch.from_numpy(x).cuda())
    assert got.dtype == torch_dtype and tuple(got.shape) == shape[:-2] + (shape[-2] + 1, shape[-1] + 1)
    got = got.cpu().numpy()
    want = np.zeros(got.shape, dtype=np_dtype)
    want[..., 1:, 1:] = x.cumsum(-2, dtype=np_dtype).cumsum(-1, dtype=np_dtype)
    assert np.array_equal(got, oracle.integral_image(x))
    assert np.array_equal(got, want)


def test_integral_image_leading_dims(hip, oracle):
    x = np.random.default_rng(5).random((2, 3, 2, 17, 19)).astype(np.float32)
    got = host(hip.integral_image(dev(x)))
    assert got.shape == (2, 3, 2, 18, 20)
    assert rel_err(got, oracle.integral_image(x)) <= 1e-6
    x2 = np.random.default_rng(6).random((17, 19)).astype(np.float32)
    assert rel_err(host(hip.integral_image(dev(x2))), oracle.integral_image(x2)) <= 1e-6


def run_both(hip, oracle, x, boxes, reparam_h, reparam_w, normalize, exact, grad_out,
             needs=(True,) * 5):
    """Forward + backward of the native functions on both sides, parameters in real units."""
    integ_cpu = oracle.integral_image(x)
    out_cpu = oracle.box_forward(integ_cpu, *boxes, normalize, exact)
    back_cpu = oracle.box_backward(integ_cpu, *boxes, grad_out, out_cpu, reparam_h, reparam_w,
                                   normalize, exact, needs)
    integ = hip.integral_image(dev(x))
    b = [dev(p) for p in boxes]
    out = hip.box_convolution_forward(integ, *b, normalize, exact)
    back = hip.box_convolution_backward(integ, *b, dev(grad_out), out, reparam_h, reparam_w,
                                        normalize, exact, *needs)
    torch.cuda.synchronize()
    scales = dict(i_max=float(np.abs(integ_cpu).max()),
                  gi_max=float(np.abs(oracle.integral_image(grad_out)).max()),
                  pg_scale=float(np.abs(integ_cpu).max() * np.abs(grad_out).max()
                                 * max(abs(reparam_h), abs(reparam_w))
                                 * np.sqrt(grad_out.shape[-1] * grad_out.shape[-2])) if grad_out.size else 0.0)
    return (out_cpu, back_cpu), (host(out), [None if g is None else host(g) for g in back]), scales


# comparisons made by assert_parity in this process, and how many of them passed only thanks to
# the additive noise term or the sibling-tensor scale (see its docstring)
NOISE_STATS = {"comparisons": 0, "needed_noise_term": 0, "of_those_reference_all_zero": 0,
               "worst_ratio": 0.0, "worst_case": ""}


def assert_parity(cpu, gpu, dtype, what="", i_max=0.0, gi_max=0.0, pg_scale=0.0):
    """max|gpu-cpu| <= tol * scale + rounding noise, per tensor.

    forward / grad_input: scale = max|cpu|, noise = 8 eps * (largest integral-image entry): every
    output is a difference of integral-image entries, each known to half a unit in its last place;
    it only matters for tensors that are (nearly) zero, e.g. a box that misses the image.
    i_max / gi_max: largest |entry| of the integral image of the input / of grad_output.

    Parameter gradients: scale = max(max|cpu|, 1e-2 * largest of the four tensors), noise =
    eps * pg_scale with pg_scale = i_max * max|grad_output| * reparametrization * sqrt(h*w). They
    are sums over all pixels of grad_output times differences of integral-image entries, scaled
    by the reparametrization factor, so the float32 reference itself carries a random-walk error
    of that order (checked against the float64 oracle: e.g. input mean 3, 65x1535, whole-pixel
    boxes: the float32 CPU result is off by 0.55 %, the GPU result by 0.09 %); for boxes that miss
    the image the true gradients are exactly zero and the reference returns pure noise."""
    tol_f, tol_p = TOL[dtype]
    eps = float(np.finfo(dtype).eps)
    (out_c, back_c), (out_g, back_g) = cpu, gpu

    def close(got, want, tol, atol, name, scale_floor=0.0, magnitude=0.0):
        want = np.asarray(want, dtype=np.float64)
        diff = np.abs(np.asarray(got, dtype=np.float64) - want).max() if want.size else 0.0
        own_scale = np.abs(want).max() if want.size else 0.0
        ok = diff <= tol * max(own_scale, scale_floor) + atol
        # bookkeeping: how often the plain bound (tol * max|cpu| of the tensor itself) would not
        # have been enough; printed at the end of the run
        NOISE_STATS["comparisons"] += 1
        if ok and diff > tol * own_scale:
            NOISE_STATS["needed_noise_term"] += 1
            # a reference tensor a million times smaller than what it is made of (the integral
            # image for forward / grad_input; for a parameter gradient the largest sibling, or the
            # size of the sums it is a difference of) counts as zero: it lies below the float32
            # resolution of those sums, its entries are the reference's own rounding noise
            negligible = own_scale <= 1e-6 * magnitude
            NOISE_STATS["of_those_reference_all_zero"] += int(negligible)
            # how far beyond the plain bound the others sit: diff / (tol * max|cpu|)
            if not negligible and diff / (tol * own_scale) > NOISE_STATS["worst_ratio"]:
                NOISE_STATS["worst_ratio"] = diff / (tol * own_scale)
                NOISE_STATS["worst_case"] = "%s %s %s, max|cpu| %.3g, diff %.3g" % (
                    what, name, np.dtype(dtype).name, own_scale, diff)
        return ok

    assert close(out_g, out_c, tol_f, 8 * eps * i_max, "forward", magnitude=i_max), what + " forward"
    if back_c[0] is not None:
        assert close(back_g[0], back_c[0], tol_f, 8 * eps * gi_max, "grad_input", magnitude=gi_max), what + " grad_input"
    floor = param_grad_floor(back_c[1:])
    for k, name in enumerate(("x_min", "x_max", "y_min", "y_max")):
        if back_c[1 + k] is not None:
            assert close(back_g[1 + k], back_c[1 + k], tol_p, eps * pg_scale, "grad_" + name, floor, max(100 * floor, pg_scale)), what + " grad_" + name


SMALL_CASES = [
    # B, C, F, h, w
    (1, 1, 1, 2, 2), (1, 1, 1, 5, 9), (2, 3, 2, 7, 6), (1, 2, 3, 10, 10), (2, 1, 5, 28, 28),
    (1, 2, 2, 17, 65), (1, 1, 3, 40, 130), (1, 2, 2, 33, 300), (1, 1, 2, 20, 600),
    (1, 1, 2, 12, 1100), (1, 1, 1, 9, 2100), (1, 1, 2, 1, 1), (1, 1, 2, 1, 70), (1, 1, 2, 70, 1),
    (1, 1, 2, 12, 700), (1, 2, 1, 10, 768), (1, 1, 2, 11, 1300), (1, 1, 1, 9, 1536),   # three columns per lane
    (1, 1, 2, 40, 2048), (1, 2, 2, 21, 1800), (1, 1, 1, 10, 2047),      # 512 threads, four columns per lane
    # the same shape with an even number of row pairs per band (a band then ends in the second LDS
    # buffer; float64 in rounded mode once returned wrong parameter gradients exactly there)
    (1, 1, 2, 4, 1538), (2, 1, 3, 32, 1537), (1, 1, 4, 8, 1800), (1, 1, 2, 16, 2047), (1, 1, 2, 12, 1300),
    # narrow images with four filters or more: the waves of a grad-input workgroup share the
    # filters (one turn with idle waves, two turns with the second partial, full-width rows)
    (1, 2, 4, 9, 20), (1, 2, 11, 19, 33), (2, 1, 16, 12, 64),
    (1, 2, 2, 12, 128), (1, 1, 3, 35, 100),          # two waves per row, full and partial
    # the same sharing of filters for rows of two and four waves
    (1, 2, 5, 20, 100), (1, 1, 6, 12, 128), (1, 1, 4, 20, 200), (1, 2, 7, 9, 256),
    # one and two waves with three or four columns per lane (rows of 129 to 512 columns), rows that
    # fill the workgroup's column slots exactly and rows that do not
    (1, 2, 2, 14, 192), (1, 1, 2, 13, 150), (2, 1, 2, 10, 384), (1, 1, 3, 9, 512), (1, 1, 2, 11, 500),
    (1, 2, 1, 16, 257),
    # rows of 2049 to 4096 columns: 1024 threads, three or four columns per lane (float32; float64
    # rows this wide and anything wider take the gather kernels)
    (1, 1, 1, 8, 3072), (1, 2, 1, 7, 4096), (1, 1, 2, 6, 3500), (1, 1, 1, 5, 2049), (1, 1, 1, 5, 4100),
]


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("kind", ["inside", "hanging", "integer"])
@pytest.mark.parametrize("B,C,F,h,w", SMALL_CASES)
def test_forward_backward_small(hip, oracle, B, C, F, h, w, kind, dtype):
    seed = (B * 7 + C * 11 + F * 13 + h * 17 + w * 19) * 3 + len(kind)
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((B, C, h, w)).astype(dtype)
    g = rng.standard_normal((B, C * F, h, w)).astype(dtype)
    boxes = make_boxes(rng, C, F, max(h, 4), max(w, 4), kind, dtype)
    for normalize in (True, False):
        for exact in (True, False):
            if not exact:
                # rounded mode needs boxes at least one whole pixel thick to have a finite area
                bx = list(boxes)
                bx[1] = (np.maximum(bx[1], np.ceil(bx[0]) + 1)).astype(dtype)
                bx[3] = (np.maximum(bx[3], np.ceil(bx[2]) + 1)).astype(dtype)
                use = tuple(bx)
            else:
                use = boxes
            cpu, gpu, sc = run_both(hip, oracle, x, use, 3.5 * h, 2.25 * w, normalize, exact, g)
            assert_parity(cpu, gpu, dtype, "%s normalize=%s exact=%s" % (kind, normalize, exact), **sc)


@pytest.mark.parametrize("kind", ["inside", "hanging", "inverted"])
@pytest.mark.parametrize("h,w", [(150, 90), (257, 256), (97, 520), (140, 400), (131, 170), (100, 2600), (3000, 40)])
def test_backward_across_row_bands(hip, oracle, h, w, kind):
    """Images tall enough that the backward pass cuts grad_output into several row bands, with
    boxes whose top and bottom rows fall into different bands; 'inverted' boxes have min > max
    along the rows (their bottom rows lie above their top rows)."""
    rng = np.random.default_rng(h * 1000 + w + len(kind))
    B, C, F = 1, 2, 3
    x = rng.standard_normal((B, C, h, w)).astype(np.float32)
    g = (rng.standard_normal((B, C * F, h, w)) + 0.5).astype(np.float32)
    boxes = list(make_boxes(rng, C, F, h, w, "hanging" if kind == "inverted" else kind,
                            away_from_integers=0.05))
    if kind == "inverted":
        lo = rng.uniform(-0.6 * h, 0.6 * h, (C, F))
        boxes[0] = lo.astype(np.float32)                                  # x_min
        boxes[1] = (lo - rng.uniform(3.3, 0.5 * h, (C, F))).astype(np.float32)   # x_max < x_min
    cpu, gpu, sc = run_both(hip, oracle, x, tuple(boxes), 3.5 * h, 2.25 * w, False, True, g)
    assert_parity(cpu, gpu, np.float32, "%s %dx%d" % (kind, h, w), **sc)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("exact", [True, False])
@pytest.mark.parametrize("h,w", [(12, 40), (70, 300), (40, 1024), (16, 512), (9, 700), (33, 1500), (36, 1800),
                                 (40, 2048), (18, 3000)])
def test_backward_lower_bound_one_ulp_above_an_integer(hip, oracle, h, w, exact, dtype):
    """A lower bound so close above an integer that `bound - 1` rounds to the integer below: the
    split the reference uses for the parameter gradients (src/box_convolution.cpp:80-96) and the
    mirrored split it uses for the input gradient (:51-67) then cut the box at different whole
    pixels. The grad_output pass computes separate column weights for the two in that case; in
    rounded mode a shared set would put a whole column of grad_input off. The widths reach every
    workgroup shape of that pass; the heights give bands with odd and with even numbers of row
    pairs."""
    rng = np.random.default_rng(h * 31 + w + int(exact))
    B, C, F = 1, 2, 2
    x = rng.standard_normal((B, C, h, w)).astype(dtype)
    g = rng.standard_normal((B, C * F, h, w)).astype(dtype)
    one = dtype(1.0)

    def above(v):
        return np.nextafter(dtype(v), dtype(0.0))

    just_above = above(-1.0)                                         # float32: -0.99999994
    assert dtype(just_above - one) == dtype(-2.0)
    x_min = np.array([[just_above, -3.3], [above(-3.0), -0.4]], dtype)
    x_max = np.array([[4.6, 2.2], [5.0, 3.5]], dtype)
    y_min = np.array([[just_above, just_above], [-7.25, above(-2.0)]], dtype)
    y_max = np.array([[6.4, 9.0], [3.75, 11.5]], dtype)
    for normalize in (False, True):
        # Rounded mode with normalisation: the reference's second summand multiplies grad_output with
        # the saved forward output (forward split), while the sums of the grad_output pass follow the
        # split of the parameter-gradient pass; at these bounds the two differ by a whole row or
        # column, and the GPU takes that one sum again with the forward split (finalize_box).
        cpu, gpu, sc = run_both(hip, oracle, x, (x_min, x_max, y_min, y_max), 3.5 * h, 2.25 * w,
                                normalize, exact, g)
        assert_parity(cpu, gpu, dtype, "normalize=%s exact=%s" % (normalize, exact), **sc)


@pytest.mark.parametrize("w", [48, 100, 200])
@pytest.mark.parametrize("kind", ["inside", "hanging"])
def test_backward_across_row_bands_narrow_image(hip, oracle, kind, w):
    """As above for images one, two and four waves wide with many filters, where the waves of a
    grad-input workgroup take the filters in turns."""
    rng = np.random.default_rng(77 + len(kind) + w)
    B, C, F, h = 2, 2, 9, 150
    x = rng.standard_normal((B, C, h, w)).astype(np.float32)
    g = (rng.standard_normal((B, C * F, h, w)) + 0.5).astype(np.float32)
    boxes = make_boxes(rng, C, F, h, w, kind, away_from_integers=0.05)
    for normalize in (False, True):
        cpu, gpu, sc = run_both(hip, oracle, x, tuple(boxes), 3.5 * h, 2.25 * w, normalize, True, g)
        assert_parity(cpu, gpu, np.float32, "%s normalize=%s" % (kind, normalize), **sc)


@pytest.mark.parametrize("B,C,F,h,w", [(2, 1, 9, 40, 48), (1, 2, 13, 70, 100), (1, 1, 6, 33, 256)])
def test_grad_input_filter_sharing_matches_one_set_per_workgroup(hip, switches, B, C, F, h, w):
    """Small problems on narrow images: the grad-input workgroups whose thread sets take the
    filters in turns give the same result, up to the order of the float32 additions over the
    filters, as workgroups that walk through all filters themselves."""
    rng = np.random.default_rng(B + C + F + h + w)
    x = dev(rng.standard_normal((B, C, h, w)).astype(np.float32))
    g = dev(rng.standard_normal((B, C * F, h, w)).astype(np.float32))
    boxes = [dev(b) for b in make_boxes(rng, C, F, h, w, "hanging")]
    integ = hip.integral_image(x)

    def grad_input():
        return hip.box_convolution_backward(integ, *boxes, g, None, 5.0, 3.0, True, True,
                                            True, False, False, False, False)[0].clone()
    preset = os.environ.get("BOXCONV_GI_SPLIT_FILTERS")     # (a run of the suite with the switch set)
    shared = grad_input()
    switches("BOXCONV_GI_SPLIT_FILTERS", "0")
    single = grad_input()
    if os.environ.get("BOXCONV_FORCE_GATHER") != "1" and preset is None:
        assert not torch.equal(shared, single) or F < 3   # really two different code paths
    scale = single.abs().max().item()
    assert (shared - single).abs().max().item() <= 4e-6 * scale


@pytest.mark.parametrize("exact", [True, False])
@pytest.mark.parametrize("h,w", [(67, 256), (130, 512), (70, 1024), (66, 2048),
                                 # rows that leave lanes of that workgroup idle (whole waves, half a wave, one lane)
                                 (36, 240), (30, 640), (40, 960), (64, 1000), (18, 1280), (22, 1800), (34, 1920),
                                 (20, 2044), (50, 160), (33, 44), (36, 100), (40, 96), (34, 92), (30, 272), (31, 132)])
def test_grad_output_pass_variants_agree(hip, oracle, switches, h, w, exact):
    """Rows of a multiple of four columns that fill at least three eighths of a workgroup at four
    columns per lane run the grad_output pass with consecutive columns per lane (the lanes past
    the row's end idle along); BOXCONV_STREAM_CONSEC=0 sends them to the kernel with wave-strided
    columns, as every other width. Both against the oracle, and against each other to the last
    few bits (the sums differ only in which columns share a lane)."""
    rng = np.random.default_rng(h + w + int(exact))
    B, C, F = 1, 2, 3
    x = rng.standard_normal((B, C, h, w)).astype(np.float32)
    g = (rng.standard_normal((B, C * F, h, w)) + 0.25).astype(np.float32)
    boxes = list(make_boxes(rng, C, F, h, w, "hanging", away_from_integers=0.05))
    if not exact:
        boxes[1] = np.maximum(boxes[1], np.ceil(boxes[0]) + 1).astype(np.float32)
        boxes[3] = np.maximum(boxes[3], np.ceil(boxes[2]) + 1).astype(np.float32)
    results = []
    for variant in (None, "0"):
        switches("BOXCONV_STREAM_CONSEC", variant)
        cpu, gpu, sc = run_both(hip, oracle, x, tuple(boxes), 3.5 * h, 2.25 * w, True, exact, g)
        assert_parity(cpu, gpu, np.float32, "consecutive=%s %dx%d exact=%s" % (variant, h, w, exact), **sc)
        results.append(gpu)
    (_, back_a), (_, back_b) = results
    assert np.abs(back_a[0] - back_b[0]).max() <= 2e-6 * np.abs(back_b[0]).max()
    for a, b in zip(back_a[1:], back_b[1:]):
        # (float32 sums of a few hundred thousand products in two different orders)
        assert np.abs(a - b).max() <= 1e-4 * max(np.abs(b).max(), 1e-30) + 1e-5 * max(np.abs(t).max() for t in back_b[1:])


@pytest.mark.parametrize("exact", [True, False])
@pytest.mark.parametrize("h,w", [(67, 256), (30, 640), (70, 1024), (22, 1800), (20, 2044), (36, 100), (33, 44), (25, 2048)])
def test_parameter_gradients_alone(hip, oracle, h, w, exact):
    """When the input needs no gradient (a network's first layer) the grad_output pass forms the
    parameter sums only: on rows that take the kernel with consecutive columns per lane, that
    kernel without its column workspace. The sums are formed the same way with or without it, so
    the four gradients equal those of the full backward bit for bit; and they meet the oracle."""
    rng = np.random.default_rng(11 * h + w + int(exact))
    B, C, F = 2, 2, 3
    x = rng.standard_normal((B, C, h, w)).astype(np.float32)
    g = (rng.standard_normal((B, C * F, h, w)) + 0.25).astype(np.float32)
    boxes = list(make_boxes(rng, C, F, h, w, "hanging", away_from_integers=0.05))
    if not exact:
        boxes[1] = np.maximum(boxes[1], np.ceil(boxes[0]) + 1).astype(np.float32)
        boxes[3] = np.maximum(boxes[3], np.ceil(boxes[2]) + 1).astype(np.float32)
    needs = (False, True, True, True, True)
    cpu, gpu, sc = run_both(hip, oracle, x, tuple(boxes), 3.5 * h, 2.25 * w, True, exact, g, needs)
    assert gpu[1][0] is None
    assert_parity(cpu, gpu, np.float32, "parameters only %dx%d exact=%s" % (h, w, exact), **sc)
    _, full, _ = run_both(hip, oracle, x, tuple(boxes), 3.5 * h, 2.25 * w, True, exact, g)
    for a, b in zip(gpu[1][1:], full[1][1:]):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("exact", [True, False])
@pytest.mark.parametrize("h,w", [(37, 130), (40, 256), (34, 300), (70, 512), (21, 700), (36, 1024), (18, 1025),
                                 (12, 1100), (16, 1536), (10, 1538), (14, 2047), (12, 2048)])
def test_float64_grad_output_pass_shapes_agree(hip, oracle, switches, h, w, exact):
    """float64 rows of up to 1024 columns run the grad_output pass with at most two columns per
    lane, and on four or eight waves as two launches (parameter sums, column workspace); rows of
    1025 to 2048 columns as two launches as well, the parameter sums by two workgroups per band
    with two columns per lane. BOXCONV_STREAM_F64_NARROW=0 gives all of them float32's three or
    four columns per lane and the one launch. Both against the oracle and against each other."""
    rng = np.random.default_rng(3 * h + w + int(exact))
    B, C, F = 2, 2, 3
    x = rng.standard_normal((B, C, h, w))
    g = rng.standard_normal((B, C * F, h, w)) + 0.25
    boxes = list(make_boxes(rng, C, F, h, w, "hanging", away_from_integers=0.05))
    if not exact:
        boxes[1] = np.maximum(boxes[1], np.ceil(boxes[0]) + 1)
        boxes[3] = np.maximum(boxes[3], np.ceil(boxes[2]) + 1)
    boxes = tuple(np.asarray(b, dtype=np.float64) for b in boxes)
    results = []
    for variant in (None, "0"):
        switches("BOXCONV_STREAM_F64_NARROW", variant)
        cpu, gpu, sc = run_both(hip, oracle, x, boxes, 3.5 * h, 2.25 * w, True, exact, g)
        assert_parity(cpu, gpu, np.float64, "narrow=%s %dx%d exact=%s" % (variant, h, w, exact), **sc)
        results.append(gpu)
    (_, back_a), (_, back_b) = results
    for a, b in zip(back_a, back_b):
        assert np.abs(a - b).max() <= 1e-11 * max(np.abs(b).max(), 1e-30) + 1e-12 * max(np.abs(t).max() for t in back_b[1:])


@pytest.mark.parametrize("h,w,F", [(64, 20, 3), (64, 40, 5), (96, 200, 3), (128, 256, 2), (256, 512, 3),
                                   (64, 1024, 3), (128, 2500, 2)])
def test_workspace_layouts_agree(hip, oracle, switches, h, w, F):
    """Planes that are cut into whole bands of a power-of-two number of rows keep the rows of the
    column workspace interleaved over the bands (row k of every band side by side);
    BOXCONV_M_INTERLEAVE=0 keeps them in their natural order. Only the place of a row changes,
    so the two give the same bits, and both meet the oracle."""
    rng = np.random.default_rng(h * 7 + w)
    B, C = 2, 2
    x = rng.standard_normal((B, C, h, w)).astype(np.float32)
    g = (rng.standard_normal((B, C * F, h, w)) + 0.25).astype(np.float32)
    boxes = tuple(make_boxes(rng, C, F, h, w, "hanging", away_from_integers=0.05))
    results = []
    for layout in ("1", "0"):
        switches("BOXCONV_M_INTERLEAVE", layout)
        cpu, gpu, sc = run_both(hip, oracle, x, boxes, 2.5 * h, 1.5 * w, True, True, g)
        assert_parity(cpu, gpu, np.float32, "interleave=%s %dx%d" % (layout, h, w), **sc)
        results.append(gpu)
    (_, back_a), (_, back_b) = results
    for a, b in zip(back_a, back_b):
        assert np.array_equal(a, b)


def test_parameter_gradients_are_reproducible(hip):
    """The streaming backward adds the per-workgroup partial sums in a fixed order (no atomics),
    so repeated calls agree bit for bit."""
    rng = np.random.default_rng(5)
    B, C, F, h, w = 3, 2, 3, 130, 200
    x = dev(rng.standard_normal((B, C, h, w)).astype(np.float32))
    g = dev(rng.standard_normal((B, C * F, h, w)).astype(np.float32))
    boxes = [dev(b) for b in make_boxes(rng, C, F, h, w, "hanging")]
    integ = hip.integral_image(x)
    out = hip.box_convolution_forward(integ, *boxes, True, True)
    runs = [hip.box_convolution_backward(integ, *boxes, g, out, 11.0, 7.0, True, True,
                                         True, True, True, True, True) for _ in range(3)]
    torch.cuda.synchronize()
    for other in runs[1:]:
        for a, b in zip(runs[0], other):
            assert torch.equal(a, b)


def test_unit_box_is_identity(hip):
    x = torch.randn(2, 3, 13, 31, device="cuda")
    z = torch.zeros(3, 2, device="cuda")
    out = hip.box_convolution_forward(hip.integral_image(x), z, z, z, z, True, True)
    want = x.repeat_interleave(2, dim=1)
    assert torch.allclose(out, want, rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("needs", [(True, False, False, False, False), (False, True, True, True, True),
                                   (False, False, True, False, False), (True, True, False, False, True)])
def test_selective_gradients(hip, oracle, needs):
    rng = np.random.default_rng(77)
    B, C, F, h, w = 2, 2, 3, 19, 23
    x = rng.standard_normal((B, C, h, w)).astype(np.float32)
    g = rng.standard_normal((B, C * F, h, w)).astype(np.float32)
    boxes = make_boxes(rng, C, F, h, w, "hanging")
    cpu, gpu, sc = run_both(hip, oracle, x, boxes, 40.0, 50.0, True, True, g, needs)
    for k in range(5):
        assert (gpu[1][k] is None) == (not needs[k])
    assert_parity(cpu, gpu, np.float32, **sc)


def test_gather_kernels_match_row_streaming(hip, oracle, switches):
    """The per-pixel gather kernels (used for very wide images) against the oracle."""
    rng = np.random.default_rng(123)
    B, C, F, h, w = 2, 2, 3, 31, 77
    x = rng.standard_normal((B, C, h, w)).astype(np.float32)
    g = rng.standard_normal((B, C * F, h, w)).astype(np.float32)
    boxes = make_boxes(rng, C, F, h, w, "hanging")
    switches("BOXCONV_FORCE_GATHER", "1")
    for normalize in (True, False):
        for exact in (True, False):
            if not exact:
                boxes = make_boxes(rng, C, F, h, w, "inside")
            cpu, gpu, sc = run_both(hip, oracle, x, boxes, 40.0, 50.0, normalize, exact, g)
            assert_parity(cpu, gpu, np.float32, "gather normalize=%s exact=%s" % (normalize, exact), **sc)


def test_clip_parameters_matches_oracle(hip, oracle):
    rng = np.random.default_rng(9)
    for dtype in (np.float32, np.float64):
        for exact in (True, False):
            n = 257
            rh, rw, mh, mw = 8.0 * 28, 3.3 * 40, 28.0, 40.0
            p = [(rng.uniform(-1.5, 1.5, n) * s).astype(dtype) for s in (mh / rh, mh / rh, mw / rw, mw / rw)]
            p[1][:40] = p[0][:40] + rng.uniform(-0.5, 0.5, 40).astype(dtype) / rh   # thin / inverted boxes
            want = [a.copy() for a in p]
            oracle.clip_parameters(*want, rh, rw, mh, mw, exact)
            t = [dev(a) for a in p]
            hip.clip_parameters(*t, rh, rw, mh, mw, exact)
            for a, b in zip(t, want):
                assert np.array_equal(host(a), b)


def launches(hip, kernel, call):
    """How often `kernel` is launched by `call`."""
    hip.profile_arm(kernel)
    call()
    return hip.profile_collect()[1]


SNAPSHOT_SHAPES = [
    # groups of 8 output rows: one group, a ragged last one, several bands of the grad_output pass
    (1, 2, 8, 256), (2, 1, 33, 100), (2, 3, 130, 300), (1, 4, 97, 640), (1, 2, 40, 1920), (1, 1, 50, 2048),
    # groups of 16 rows: the smallest launch that takes them, ragged rows and columns
    (256, 1, 113, 160), (128, 2, 129, 260), (64, 1, 250, 516), (40, 3, 210, 1024), (33, 2, 257, 1400)]


@pytest.mark.parametrize("exact,normalize", [(True, True), (False, True), (True, False)])
@pytest.mark.parametrize("planes,F,h,w", SNAPSHOT_SHAPES)
def test_grad_input_from_snapshots(hip, oracle, switches, planes, F, h, w, exact, normalize):
    """grad_input formed from grad_output itself and the snapshots of its column sums (rows of a
    multiple of four columns; BOXCONV_GI_SNAPSHOTS=2: launches of any size) against the oracle (the
    groups of 8 rows up to two planes, those of 16 at their smallest launch), and against the column
    workspace (BOXCONV_GI_SNAPSHOTS=0): the two differ in the order of float32 additions, i.e. by a few
    units in the last place of the largest partial sum. The boxes hang over every edge, so the rows
    where the groups start clamp to both ends of the image. Parameter gradients keep their bits."""
    rng = np.random.default_rng(planes + F + h + w)
    x = rng.standard_normal((1, planes, h, w)).astype(np.float32)
    g = (rng.standard_normal((1, planes * F, h, w)) + 0.25).astype(np.float32)
    boxes = list(make_boxes(rng, planes, F, h, w, "hanging", away_from_integers=0.05))
    if not exact:
        boxes[1] = np.maximum(boxes[1], np.ceil(boxes[0]) + 1).astype(np.float32)
        boxes[3] = np.maximum(boxes[3], np.ceil(boxes[2]) + 1).astype(np.float32)
    integ, dg, db = hip.integral_image(dev(x)), dev(g), [dev(b) for b in boxes]
    results = []
    for variant in ("2", "0"):
        switches("BOXCONV_GI_SNAPSHOTS", variant)

        def backward():
            return hip.box_convolution_backward(integ, *db, dg, None, 3.5 * h, 2.25 * w, normalize, exact,
                                                True, True, True, True, True)
        if planes <= 2 or planes == 256:
            cpu, gpu, sc = run_both(hip, oracle, x, tuple(boxes), 3.5 * h, 2.25 * w, normalize, exact, g)
            assert_parity(cpu, gpu, np.float32, "snapshots=%s %dx%d" % (variant, h, w), **sc)
        assert launches(hip, "grad_input_taps", backward) == (variant == "2")
        results.append([t.cpu().numpy() for t in backward()])
    a, b = results
    assert np.abs(a[0] - b[0]).max() <= 4e-6 * np.abs(b[0]).max()
    for p, q in zip(a[1:], b[1:]):
        assert np.array_equal(p, q)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("planes,F,h,w", SNAPSHOT_SHAPES)
def test_grad_input_from_snapshots_half(hip, switches, planes, F, h, w, dtype):
    """The same with a 16-bit grad_output against its float32 copy through the column workspace:
    grad_input is rounded once more, parameter gradients see the same float32 values."""
    rng = np.random.default_rng(planes + F + h + w)
    integ = hip.integral_image(dev(rng.standard_normal((1, planes, h, w)).astype(np.float32)))
    g = dev((rng.standard_normal((1, planes * F, h, w)) + 0.25).astype(np.float32)).to(dtype)
    boxes = [dev(b) for b in make_boxes(rng, planes, F, h, w, "hanging", away_from_integers=0.05)]

    def backward(grad):
        return hip.box_convolution_backward(integ, *boxes, grad, None, 3.5 * h, 2.25 * w, True, True,
                                            True, True, True, True, True)
    switches("BOXCONV_GI_SNAPSHOTS", "2")
    assert launches(hip, "grad_input_taps", lambda: backward(g)) == 1
    a = backward(g)
    switches("BOXCONV_GI_SNAPSHOTS", "0")
    b = backward(g.float())
    assert a[0].dtype == dtype
    # half a unit in the last place of the 16-bit type, and of denormals of float16, beside the float32
    # difference of the test above
    unit, least = {torch.float16: (2.0 ** -11, 2.0 ** -25), torch.bfloat16: (2.0 ** -8, 0.0)}[dtype]
    assert ((a[0].float() - b[0]).abs() <= unit * b[0].abs() + 4.1e-6 * b[0].abs().max() + least).all()
    for p, q in zip(a[1:], b[1:]):
        assert torch.equal(p, q)


@pytest.mark.parametrize("exact", [True, False])
@pytest.mark.parametrize("h,w", [
    # remainders of one, two and three columns: the smallest rows, rows of just under, on and over a
    # whole number of waves, lanes behind the row's end in the same wave or a wave of their own
    (33, 129), (26, 130), (31, 191), (40, 255), (24, 257), (37, 258), (24, 301), (29, 510), (25, 513),
    (70, 767), (24, 1021), (27, 1023), (24, 1281), (26, 2045), (25, 2047)])
def test_grad_output_pass_of_odd_rows(hip, oracle, switches, h, w, exact):
    """Rows that are not a multiple of four columns in the grad_output pass with consecutive columns
    per lane, whose last lane takes the row's last four columns and shares some with its neighbour:
    with snapshots, with the column workspace and with the parameter sums alone, against the oracle
    (BOXCONV_STREAM_CONSEC=3: in launches of any size), and against the kernel with wave-strided
    columns (=2). The boxes hang over both ends of the rows."""
    rng = np.random.default_rng(h * w + int(exact))
    B, C, F = 1, 2, 3
    x = rng.standard_normal((B, C, h, w)).astype(np.float32)
    g = (rng.standard_normal((B, C * F, h, w)) + 0.25).astype(np.float32)
    boxes = list(make_boxes(rng, C, F, h, w, "hanging", away_from_integers=0.05))
    if not exact:
        boxes[1] = np.maximum(boxes[1], np.ceil(boxes[0]) + 1).astype(np.float32)
        boxes[3] = np.maximum(boxes[3], np.ceil(boxes[2]) + 1).astype(np.float32)
    results = []
    for snapshots, consecutive in (("2", "3"), ("0", "3"), ("0", "2")):
        switches("BOXCONV_GI_SNAPSHOTS", snapshots)
        switches("BOXCONV_STREAM_CONSEC", consecutive)
        cpu, gpu, sc = run_both(hip, oracle, x, tuple(boxes), 3.5 * h, 2.25 * w, True, exact, g)
        assert_parity(cpu, gpu, np.float32, "snapshots=%s consecutive=%s %dx%d" % (snapshots, consecutive, h, w), **sc)
        results.append(gpu[1])
        alone = run_both(hip, oracle, x, tuple(boxes), 3.5 * h, 2.25 * w, True, exact, g, (False, True, True, True, True))
        if consecutive == "3":
            for a, b in zip(alone[1][1][1:], results[0][1:]):
                assert np.array_equal(a, b)
    for r in results[:2]:
        assert np.abs(r[0] - results[2][0]).max() <= 4e-6 * np.abs(results[2][0]).max()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("h,w", [(24, 133), (33, 255), (25, 259), (40, 767), (24, 2046)])
def test_grad_output_pass_of_odd_rows_half(hip, switches, h, w, dtype):
    """The same with a 16-bit grad_output that starts on an odd element, and so on any 2-byte address in
    every row, against its float32 copy: parameter gradients see the same float32 values in the same
    order, grad_input is rounded once more."""
    rng = np.random.default_rng(h + w)
    planes, F = 3, 4
    integ = hip.integral_image(dev(rng.standard_normal((1, planes, h, w)).astype(np.float32)))
    flat = dev((rng.standard_normal(planes * F * h * w + 1) + 0.25).astype(np.float32)).to(dtype)
    g = flat[1:].view(1, planes * F, h, w)
    boxes = [dev(b) for b in make_boxes(rng, planes, F, h, w, "hanging", away_from_integers=0.05)]

    def backward(grad):
        return hip.box_convolution_backward(integ, *boxes, grad, None, 3.5 * h, 2.25 * w, True, True,
                                            True, True, True, True, True)
    switches("BOXCONV_GI_SNAPSHOTS", "2")
    assert launches(hip, "grad_input_taps", lambda: backward(g)) == 1
    a, b = backward(g), backward(g.float())
    # half a unit in the last place of the 16-bit type, and of denormals of float16: the float32 sums
    # are the same ones
    unit, least = {torch.float16: (2.0 ** -11, 2.0 ** -25), torch.bfloat16: (2.0 ** -8, 0.0)}[dtype]
    assert ((a[0].float() - b[0]).abs() <= unit * b[0].abs() + least).all()
    for p, q in zip(a[1:], b[1:]):
        assert torch.equal(p, q)


@pytest.mark.parametrize("h,w", [(272, 1029), (285, 1281), (271, 1534), (272, 1536), (287, 1792)])
def test_bands_that_make_one_round(hip, switches, h, w):
    """Rows of five to seven waves of 256 planes and filters: two long bands each, 512 workgroups, with
    snapshots and for the parameter sums alone, against the kernel with wave-strided columns (0). 1029 and 1281
    columns end with a wave, 1281 with a single lane in use, 1536 and 1792 with a full one."""
    rng = np.random.default_rng(h * w)
    C, F = 32, 8
    integ = hip.integral_image(dev(rng.standard_normal((1, C, h, w)).astype(np.float32)))
    g = torch.randn(1, C * F, h, w, device="cuda", generator=torch.Generator("cuda").manual_seed(h * w)).add_(0.25)
    boxes = [dev(b) for b in make_boxes(rng, C, F, h, w, "hanging", away_from_integers=0.05)]

    def backward(need_input):
        return hip.box_convolution_backward(integ, *boxes, g, None, 3.5 * h, 2.25 * w, True, True,
                                            need_input, True, True, True, True)
    assert launches(hip, "grad_input_taps", lambda: backward(True)) == 1
    full, alone = backward(True), backward(False)

    def bands():                       # sums that a call leaves per plane and filter: all that its scratch memory holds
        hip.release_workspaces()
        backward(False)
        (scratch,) = hip._workspaces.values()
        scratch.fill_(255)             # (a NaN in float64)
        backward(False)
        n = int(scratch.view(torch.float64).isfinite().sum())
        assert n % (5 * C * F) == 0
        return n // (5 * C * F)
    assert bands() == 2
    switches("BOXCONV_STREAM_CONSEC", "0")
    ref = backward(True)
    assert (full[0] - ref[0]).abs().max() <= 4e-6 * ref[0].abs().max()
    # as in assert_parity: the order of the float32 sums inside a row differs, each term a difference of
    # integral-image entries that are known to half a unit in the last place, over h * w pixels
    noise = 2.0 ** -23 * integ.abs().max() * g.abs().max() * 3.5 * (h * w) ** 0.5
    for p, q, r, side in zip(full[1:], alone[1:], ref[1:], (h, h, w, w)):
        assert torch.equal(p, q)
        assert (p - r).abs().max() <= 1e-5 * r.abs().max() + noise * side


@pytest.mark.parametrize("h,w", [(272, 1029), (285, 1281), (272, 1536), (287, 1792)])
def test_long_bands_lose_no_bits(hip, h, w):
    """The column sums that the first backward kernel leaves for the second, over bands of up to 144 rows. Rows of
    grad_output are multiples of 2**-18 from 1 to 1.5, so that float32 holds the sums of 32 of them exactly, but not
    of all: a band's sum, added up in double from there on, is rounded once."""
    rng = np.random.default_rng(h + w)
    C, F = 32, 8
    g = 1 + torch.randint(0, 1 << 17, (1, C * F, h, w), device="cuda").float() * 2.0 ** -18
    boxes = [dev(b) for b in make_boxes(rng, C, F, h, w, "inside")]
    integ = hip.integral_image(torch.randn(1, C, h, w, device="cuda"))
    hip.release_workspaces()
    assert launches(hip, "grad_input_taps", lambda: hip.box_convolution_backward(
        integ, *boxes, g, None, 1.0, 1.0, True, True, True, True, True, True, True)) == 1
    # rows of the scratch memory: zeros; per plane and filter two snapshots per group of 16 output rows, a sum per band
    (scratch,) = hip._workspaces.values()
    pitch, groups = (w + 3) // 4 * 4, (h + 15) // 16
    bands = scratch.view(torch.float32)[pitch:][:C * F * (2 * groups + 2) * pitch].view(C * F, 2 * groups + 2, pitch)[:, -2:, :w]
    first = (h + 1) // 2 + (h + 1) // 2 % 2
    exact = torch.stack([g[0, :, :first].double().sum(1), g[0, :, first:].double().sum(1)], 1)
    assert torch.equal(bands, exact.float())


NARROW_SHAPES = [
    # 8, 16 and 32 lanes per row, full, with idle lanes, and with a last lane that shares columns; one band,
    # bands past the plane, several waves per plane; filters shared by 1, 2, 4 and 8 waves, evenly or not
    (8, 16, 1), (28, 28, 9), (17, 17, 3), (33, 32, 2), (9, 31, 16), (130, 23, 5), (64, 33, 4), (40, 48, 3),
    (200, 63, 1), (31, 64, 8), (64, 65, 2), (70, 95, 3), (129, 100, 2), (64, 128, 4), (300, 127, 1)]


@pytest.mark.parametrize("exact,normalize", [(True, True), (False, True), (True, False)])
@pytest.mark.parametrize("h,w,F", NARROW_SHAPES)
def test_narrow_rows_side_by_side(hip, oracle, switches, h, w, F, exact, normalize):
    """Rows of at most 128 columns with several bands (or groups of output rows) side by side in a wave
    (BOXCONV_NARROW=2: launches of any size), against the oracle and against the kernels for wider
    rows; the parameter sums alone are those of the full pass, bit for bit. The boxes hang over every edge."""
    rng = np.random.default_rng(h * w + F)
    B, C = 2, 3
    x = rng.standard_normal((B, C, h, w)).astype(np.float32)
    g = (rng.standard_normal((B, C * F, h, w)) + 0.25).astype(np.float32)
    boxes = list(make_boxes(rng, C, F, h, w, "hanging", away_from_integers=0.05))
    if not exact:
        boxes[1] = np.maximum(boxes[1], np.ceil(boxes[0]) + 1).astype(np.float32)
        boxes[3] = np.maximum(boxes[3], np.ceil(boxes[2]) + 1).astype(np.float32)
    results = []
    for variant in ("2", "0"):
        switches("BOXCONV_NARROW", variant)
        switches("BOXCONV_GI_SNAPSHOTS", None if variant == "2" else "0")
        cpu, gpu, sc = run_both(hip, oracle, x, tuple(boxes), 3.5 * h, 2.25 * w, normalize, exact, g)
        assert_parity(cpu, gpu, np.float32, "narrow=%s %dx%d" % (variant, h, w), **sc)
        results.append(gpu[1])
    assert np.abs(results[0][0] - results[1][0]).max() <= 4e-6 * np.abs(results[1][0]).max()
    switches("BOXCONV_NARROW", "2")
    switches("BOXCONV_GI_SNAPSHOTS", None)
    _, alone, _ = run_both(hip, oracle, x, tuple(boxes), 3.5 * h, 2.25 * w, normalize, exact, g, (False, True, True, True, True))
    for a, b in zip(alone[1][1:], results[0][1:]):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("h,w,F", [(28, 28, 9), (41, 45, 3), (64, 128, 4), (33, 127, 2), (20, 18, 1)])
def test_narrow_rows_half(hip, switches, h, w, F, dtype):
    """The same with a 16-bit grad_output, for odd rows one that starts on any 2-byte address, against its
    float32 copy: the same float32 sums, grad_input rounded once more."""
    rng = np.random.default_rng(h + w)
    planes = 5
    switches("BOXCONV_NARROW", "2")
    integ = hip.integral_image(dev(rng.standard_normal((1, planes, h, w)).astype(np.float32)))
    flat = dev((rng.standard_normal(planes * F * h * w + 1) + 0.25).astype(np.float32)).to(dtype)
    g = flat[1:].view(1, planes * F, h, w) if w % 4 else flat[:-1].view(1, planes * F, h, w)
    boxes = [dev(b) for b in make_boxes(rng, planes, F, h, w, "hanging", away_from_integers=0.05)]

    def backward(grad):
        return hip.box_convolution_backward(integ, *boxes, grad, None, 3.5 * h, 2.25 * w, True, True,
                                            True, True, True, True, True)
    a, b = backward(g), backward(g.float())
    unit, least = {torch.float16: (2.0 ** -11, 2.0 ** -25), torch.bfloat16: (2.0 ** -8, 0.0)}[dtype]
    assert ((a[0].float() - b[0]).abs() <= unit * b[0].abs() + least).all()
    for p, q in zip(a[1:], b[1:]):
        assert torch.equal(p, q)


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
@pytest.mark.parametrize("h,w,F", [
    # several rows side by side in a wave, bands past the plane among them; rows that are no multiple of four columns;
    # rows of five waves
    (33, 32, 2), (28, 28, 9), (17, 17, 3), (70, 60, 3), (45, 100, 2), (50, 127, 4), (41, 128, 2), (40, 129, 3), (36, 301, 2),
    (34, 767, 2), (40, 1281, 2)])
def test_infinities_and_nan_stay_where_they_act(hip, switches, h, w, F, bad):
    """An input pixel that no box reaches has no effect on the parameter gradients, whatever its value; a value of
    grad_output makes what depends on it infinite or NaN, and changes no bit of other planes' and other boxes' gradients."""
    switches("BOXCONV_NARROW", "2")
    switches("BOXCONV_GI_SNAPSHOTS", "2" if w > 128 else None)
    switches("BOXCONV_STREAM_CONSEC", "3")
    C = 3
    gen = torch.Generator().manual_seed(h * w)
    x = torch.randn(1, C, h, w, generator=gen)
    g = torch.randn(1, C * F, h, w, generator=gen).cuda()
    y_lo = -2.3 - 3 * torch.rand(C, F, generator=gen).cuda()

    def backward(x, boxes, g):
        return hip.box_convolution_backward(hip.integral_image(x.cuda()), *boxes, g, None, 1.0, 1.0, True, True,
                                            True, True, True, True, True)
    # boxes that end 2.6 rows and more above the image's last row for every output pixel
    x_hi = -3.6 - torch.rand(C, F, generator=gen).cuda()
    above = (x_hi - 2.2 - 3 * torch.rand(C, F, generator=gen).cuda(), x_hi, y_lo, -y_lo)
    spoiled, clean = x.clone(), x.clone()
    spoiled[..., -1, w // 3], clean[..., -1, :] = bad, 0.0
    spoiled[..., -1, 1] = -bad
    for a, b in zip(backward(spoiled, above, g)[1:], backward(clean, above, g)[1:]):
        assert torch.equal(a, b)
    # boxes around the pixel, far enough inside the image to be whole
    boxes = (y_lo - 0.1, -y_lo, y_lo, 0.2 - y_lo)
    i, j = h // 2, w // 2
    spoiled = g.clone()
    spoiled[0, 0, i, j] = bad
    got, want = backward(x, boxes, spoiled), backward(x, boxes, g)
    assert torch.equal(got[0][:, 1:], want[0][:, 1:])
    assert not torch.isfinite(got[0][0, 0, i - 2:i + 3, j - 2:j + 3]).any()
    for a, b in zip(got[1:], want[1:]):
        assert not torch.isfinite(a[0, 0])
        assert torch.equal(a.flatten()[1:], b.flatten()[1:])


@pytest.mark.parametrize("consecutive,planes,F,h,w", [
    # 129 to 192 columns from 2^23 output pixels on, 257 to 384 from 2^22, 513 to 640 from 2^21, between them always; more
    # than 1024 columns with more than 256 workgroups
    (False, 9, 10, 116, 161), (False, 64, 10, 70, 187), (True, 64, 10, 71, 187), (True, 9, 10, 116, 193), (True, 2, 4, 100, 255),
    (False, 8, 5, 300, 331), (True, 32, 5, 100, 331), (True, 2, 4, 100, 385), (False, 2, 2, 900, 534), (True, 8, 4, 125, 525),
    (True, 2, 4, 100, 641), (False, 12, 1, 700, 1279), (True, 32, 1, 300, 1279)])
def test_parameter_sums_of_odd_rows_only_where_they_pay(hip, switches, consecutive, planes, F, h, w):
    """The launches for which consecutive columns per lane are the slower way return what BOXCONV_STREAM_CONSEC=2 returns, bit
    for bit; the others what =3 does, and that differs."""
    integ = hip.integral_image(torch.randn(1, planes, h, w, device="cuda"))
    g = torch.randn(1, planes * F, h, w, device="cuda")
    boxes = [dev(b) for b in make_boxes(np.random.default_rng(h + w), planes, F, h, w, "inside")]

    def same(variant):
        got = sums()
        switches("BOXCONV_STREAM_CONSEC", variant)
        result = all(torch.equal(a, b) for a, b in zip(got, sums()))
        switches("BOXCONV_STREAM_CONSEC", None)
        return result

    def sums():
        return hip.box_convolution_backward(integ, *boxes, g, None, 1.0, 1.0, True, True, False, True, True, True, True)[1:]
    assert same("3" if consecutive else "2") and not same("2" if consecutive else "3")


@pytest.mark.parametrize("narrow,planes,F,h,w", [
    # from 28 rows on; bands that leave up to a quarter (96 to 124 columns in a multiple of four) or 0.45 of the
    # lanes without rows; enough pixels for the filters, from 400 rows on more of them
    (True, 64, 4, 28, 60), (False, 64, 4, 27, 60), (False, 51, 23, 20, 36), (False, 185, 12, 33, 110), (True, 185, 12, 64, 110),
    (False, 554, 3, 135, 96), (True, 554, 3, 128, 96), (True, 512, 4, 64, 128), (False, 479, 2, 69, 100), (False, 32, 40, 28, 28),
    (True, 64, 4, 500, 40), (False, 4, 8, 754, 90)])
def test_narrow_rows_only_where_they_pay(hip, switches, narrow, planes, F, h, w):
    """The launches for which several rows side by side in a wave are the slower way return what BOXCONV_NARROW=0
    returns, bit for bit; the others what BOXCONV_NARROW=2 does, and that differs."""
    integ = hip.integral_image(torch.randn(1, planes, h, w, device="cuda"))
    g = torch.randn(1, planes * F, h, w, device="cuda")
    boxes = [dev(b) for b in make_boxes(np.random.default_rng(h + w), planes, F, h, w, "inside")]

    def backward(need_input):
        return hip.box_convolution_backward(integ, *boxes, g, None, 1.0, 1.0, True, True, need_input, True, True, True, True)
    for need_input in (True, False):
        got = backward(need_input)
        results = {}
        for variant in ("0", "2"):
            switches("BOXCONV_NARROW", variant)
            results[variant] = [torch.equal(a, b) for a, b in zip(got, backward(need_input)) if a is not None]
            switches("BOXCONV_NARROW", None)
        assert all(results["2" if narrow else "0"])
        assert not all(results["0" if narrow else "2"])


@pytest.mark.parametrize("need_input", [True, False])
@pytest.mark.parametrize("h,w", [(40, 31), (33, 64), (50, 100), (64, 128)])
def test_narrow_rows_add_few_products_in_float(hip, switches, h, w, need_input):
    """Neighbouring columns whose contributions to a parameter gradient cancel, 2^26, 1, -2^26, 1, and again: no more than a
    row pair's products of one column may meet in a float sum, where the ones would be lost."""
    switches("BOXCONV_NARROW", "2")
    x = torch.zeros(1, 2, h, w, device="cuda")
    x[..., 0] = 1.0                                     # (the same V in every column)
    g = torch.tensor([2.0 ** 26, 1.0, -2.0 ** 26, 1.0], device="cuda").repeat(w)[:w].expand(1, 2, h, w).contiguous()
    if w % 4:
        g[..., w // 4 * 4:] = 1.0
    whole = torch.ones(2, 1, device="cuda")
    boxes = (-2.5 * whole, 2.5 * whole, -3.0 * w * whole, 0.0 * whole)
    got = hip.box_convolution_backward(hip.integral_image(x), *boxes, g, None, 1.0, 1.0, False, True, need_input,
                                       True, True, True, True)
    # the border row of output row i is i - 3 and i + 3: a sum of grad_output over the rows that have one
    want = g[0, 0, 3:].double().sum().item()
    assert torch.equal(got[1].double().cpu(), torch.full((2, 1), -want, dtype=torch.float64))
    assert torch.equal(got[2].double().cpu(), torch.full((2, 1), want, dtype=torch.float64))


@pytest.mark.parametrize("snapshots,planes,F,h,w", [
    (True, 128, 4, 128, 256), (True, 32, 8, 128, 512), (True, 16, 1, 256, 512), (True, 2, 2, 512, 1024),
    # few input pixels for the filters, fewer than 24 rows, a second round with hardly anything in it
    (False, 8, 40, 17, 100), (False, 1, 8, 96, 256), (False, 16, 8, 200, 252), (False, 2, 1, 64, 1024),
    (False, 86, 8, 17, 1212), (False, 15, 1, 552, 1124), (False, 479, 2, 69, 100),
    # a third wave with a single lane in use, from 2^22 to 2^25 output pixels
    (False, 53, 10, 55, 514), (True, 16, 8, 512, 514), (True, 6, 2, 500, 513)])
def test_snapshots_only_where_they_pay(hip, switches, snapshots, planes, F, h, w):
    """The launches for which snapshots are the slower way keep the column workspace, and then
    return what BOXCONV_GI_SNAPSHOTS=0 returns, bit for bit."""
    rng = np.random.default_rng(h + w)
    integ = hip.integral_image(torch.randn(1, planes, h, w, device="cuda"))
    g = torch.randn(1, planes * F, h, w, device="cuda")
    boxes = [dev(b) for b in make_boxes(rng, planes, F, h, w, "inside")]

    def backward():
        return hip.box_convolution_backward(integ, *boxes, g, None, 1.0, 1.0, True, True, True, True, True, True, True)
    assert launches(hip, "grad_input_taps", backward) == snapshots
    assert launches(hip, "grad_input_cols", backward) == (not snapshots)
    if not snapshots:
        got = backward()
        switches("BOXCONV_GI_SNAPSHOTS", "0")
        for a, b in zip(got, backward()):
            assert torch.equal(a, b)


@pytest.mark.parametrize("spin", [None, "0"])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("planes,h,w,single", [
    (3, 40, 257, True), (2, 33, 258, True), (16, 301, 767, True), (64, 65, 481, True), (1, 97, 1021, True),
    (2, 100, 1537, True), (1, 64, 2047, True),
    # few pixels of 64 to 256 rows and up to 512 columns: two passes; the first size that takes the single pass
    (5, 70, 259, False), (9, 256, 511, False), (47, 65, 511, False), (48, 65, 511, True), (1, 64, 513, True)])
def test_integral_image_single_pass_of_odd_rows(hip, switches, dtype, planes, h, w, single, spin):
    """Rows of 256 columns and more that are not a multiple of four columns: the single pass reads
    them with loads of four elements that start anywhere, the lane at the row's end from the row's
    last four columns. Against the two passes on the same bands (BOXCONV_INTEGRAL_LOOKBACK=0), which
    associate the double sums differently; spin = 0 sums every band above again."""
    x = torch.randn(1, planes, h, w, generator=torch.Generator().manual_seed(h * w)).cuda().to(dtype)
    switches("BOXCONV_INTEGRAL_LOOKBACK", "0")
    two = hip.integral_image(x).clone()
    switches("BOXCONV_INTEGRAL_LOOKBACK", None)
    switches("BOXCONV_INTEGRAL_SPIN", spin)
    one = hip.integral_image(x)
    assert launches(hip, "band_colsum", lambda: hip.integral_image(x)) == (not single)
    assert launches(hip, "fill_marker", lambda: hip.integral_image(x)) == single
    assert torch.allclose(one, two, rtol=2e-7, atol=0)
    want = np.cumsum(np.cumsum(x.double().cpu().numpy(), axis=2), axis=3)
    got = one.cpu().numpy()
    assert not got[:, :, 0].any() and not got[..., 0].any()
    # a float32 rounding of a double sum: half a unit in the last place of the largest entry
    assert np.abs(got[:, :, 1:, 1:] - want).max() <= 2.0 ** -24 * 1.01 * np.abs(want).max()


def test_integral_image_switch_one_is_the_default(hip, switches):
    """BOXCONV_INTEGRAL_LOOKBACK=1 takes the single pass where the default does, odd widths included."""
    x = torch.randn(1, 16, 301, 767, device="cuda")
    switches("BOXCONV_INTEGRAL_LOOKBACK", "1")
    assert launches(hip, "fill_marker", lambda: hip.integral_image(x)) == 1


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("planes,h,w", [
    # a workgroup per plane, rows of one, two and four lanes' groups of 16: last lanes that share one, two and three
    # columns, whole rows, a single lane
    (2, 50, 4), (2, 33, 7), (3, 29, 17), (2, 191, 62), (3, 130, 66), (2, 100, 127), (1, 192, 129), (2, 135, 241), (2, 40, 255),
    # taller than the workgroup holds at a time: one more row, several chunks, rows of the last chunk missing
    (2, 769, 33), (3, 1000, 64), (2, 850, 19), (2, 385, 127), (3, 512, 128), (130, 530, 100), (33, 193, 129), (40, 300, 256),
    (128, 470, 203),
    # 8 to 24 rows per band and wave; low float planes with a wave per row, and with several rows in a wave: more rows, more planes
    (2, 65, 140), (2, 100, 131), (3, 160, 202), (2, 190, 40), (3, 40, 61), (200, 48, 60), (3, 49, 99), (257, 48, 99)])
def test_integral_image_of_a_plane_per_workgroup(hip, switches, dtype, planes, h, w):
    """Planes of at most 256 columns in one launch, against the two passes on the same planes, which add the
    double sums in another order, and against a float64 cumulative sum."""
    x = torch.randn(1, planes, h, w, generator=torch.Generator().manual_seed(h * w)).cuda().to(dtype)
    switches("BOXCONV_INTEGRAL_PLANE", "0")
    two = hip.integral_image(x).clone()
    switches("BOXCONV_INTEGRAL_PLANE", None)
    assert launches(hip, "band_colsum", lambda: hip.integral_image(x)) == 0
    assert launches(hip, "band_scan", lambda: hip.integral_image(x)) == 1
    one = hip.integral_image(x)
    assert torch.allclose(one, two, rtol=2e-7, atol=0)
    want = np.cumsum(np.cumsum(x.double().cpu().numpy(), axis=2), axis=3)
    got = one.cpu().numpy()
    assert not got[:, :, 0].any() and not got[..., 0].any()
    # one rounding to float32, and that of double sums in another order
    assert (np.abs(got[:, :, 1:, 1:] - want) <= 2.0 ** -24 * np.abs(want) * 1.001 + 1e-12 * np.abs(want).max()).all()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("planes,h,w", [(3, 28, 28), (2, 61, 51), (2, 100, 96), (3, 33, 130), (2, 190, 241), (2, 100, 256), (128, 470, 203)])
def test_integral_image_of_infinities_and_nan(hip, dtype, planes, h, w):
    """Lanes behind a row and bands behind the plane load pixels of the plane: an infinite one in the first column of its last
    row, or a NaN in the middle of that column, reaches the entries that it is part of and no others."""
    x = torch.randn(planes, h, w, device="cuda").to(dtype)
    clean = hip.integral_image(x)
    for i, j, bad in ((h - 1, 0, float("inf")), (h // 2, 0, float("nan"))):
        y = x.clone()
        y[1, i, j] = bad
        got = hip.integral_image(y)
        assert not got[1, i + 1:, j + 1:].isfinite().any()
        got[1, i + 1:, j + 1:] = clean[1, i + 1:, j + 1:]
        assert torch.equal(got, clean)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16, torch.float64])
@pytest.mark.parametrize("planes,h,w", [
    # bands: every number of waves, rows that end on, just behind and just before a wave's end, last lanes that
    # share one, two and three columns, last bands of a single row
    (2, 97, 257), (3, 66, 511), (2, 70, 513), (2, 65, 767), (1, 129, 769), (2, 64, 1022), (2, 67, 1027), (1, 100, 1281),
    (2, 66, 1535), (1, 75, 1538), (2, 64, 1793), (1, 97, 2047), (1, 64, 2049), (1, 70, 4095), (2, 300, 1036), (1, 520, 604),
    # a workgroup per plane, one band of at most 256 rows
    (280, 11, 1025), (320, 9, 1000), (430, 10, 514), (640, 7, 301), (280, 257, 1284), (641, 5, 512)])
def test_integral_image_in_bands(hip, switches, dtype, planes, h, w):
    """The launches with and without a column-sum pass (BOXCONV_INTEGRAL_LOOKBACK=0), from aligned addresses and from
    an odd element on, against a float64 cumulative sum."""
    flat = torch.randn(planes * h * w + 1, generator=torch.Generator().manual_seed(h * w)).cuda().to(dtype)
    switches("BOXCONV_INTEGRAL_LOOKBACK", "0")
    for x in (flat[:-1].view(1, planes, h, w), flat[1:].view(1, planes, h, w)):
        got = hip.integral_image(x)
        want = x.double().cumsum(2).cumsum(3)
        assert not got[:, :, 0].any() and not got[..., 0].any()
        # one rounding to the output type, and that of double sums in another order
        unit = 2.0 ** -24 if got.dtype == torch.float32 else 0.0
        assert ((got[:, :, 1:, 1:].double() - want).abs() <= unit * 1.001 * want.abs() + 1e-12 * want.abs().max()).all()
