"""float32 convolutions against float64: the three-way bf16 split of both operands keeps float32's precision.

Bound on the relative 2-norm of the error.  A product leaves out at most 2^-24 of itself (ml + lm, 2 x 2^-8 x 2^-17; 5e-9, 0.08
of that, root mean square); the running sum of n K-steps
(sixteen products each, the first accumulator) is rounded n times, half a unit in the last place (2^-24 relative, uniform:
2^-24 / sqrt(3) root mean square) of a sum that grows like sqrt(i / n): 2^-24 sqrt(n / 6) = 0.41 sqrt(n) 2^-24 in all.  Twice
that, plus 2 units for the final roundings (small sums, bias), is allowed.  Leaving out the hi * low products alone would be
2^-18 of each product: 20 times over the bound at one K-step.
"""
import numpy as np
import pytest

from smallframework_amd import capi, layout, synth
from hip_util import dev, dev_empty, host, ptr, stream

pytestmark = pytest.mark.gpu


def run(shape, x, f, bias, act, pool=False):
    n, k, s, co, ci, h, w = shape
    lib = capi.load()
    t, b = capi.calc_padding(h, k, s)
    l, r = capi.calc_padding(w, k, s)
    ho, wo = capi.out_dim(h, t, b, k, s), capi.out_dim(w, l, r, k, s)
    dx, df = dev(layout.pack_activations(x)), dev(layout.pack_conv_filter(f))
    db = dev(bias) if bias is not None else None
    if pool:
        y = dev_empty(n * co * (ho // 2) * (wo // 2), np.float32)
        capi.check(lib.small_hip_conv2d_bias_act_maxpool2d_f32(n, k, k, s, t, b, l, r, 2, 2, 2, 0, 0, 0, 0, co, ci, h, w, ptr(dx), ptr(df),
                                                               ptr(db), act, 0.0, ptr(y), stream()))
        return layout.unpack_activations(host(y), n, co, ho // 2, wo // 2), (t, b, l, r)
    y = dev_empty(n * co * ho * wo, np.float32)
    capi.check(lib.small_hip_conv2d_bias_act_f32(n, k, k, s, t, b, l, r, co, ci, h, w, ptr(dx), ptr(df), ptr(db), act, 0.0, ptr(y), stream()))
    return layout.unpack_activations(host(y), n, co, ho, wo), (t, b, l, r)


def reference(x, f, bias, s, pads):
    import torch
    t, b, l, r = pads
    y = torch.nn.functional.conv2d(torch.nn.functional.pad(torch.from_numpy(x).double(), (l, r, t, b)), torch.from_numpy(f).double(), stride=s)
    return y.numpy() if bias is None else y.numpy() + bias.astype(np.float64)[None, :, None, None]


SHAPES = [  # batch, window, stride, Co, Ci, H, W
    (1, 1, 1, 16, 16, 1, 1),          # one K-step, one pixel
    (2, 1, 1, 48, 16, 7, 5),
    (1, 3, 1, 32, 16, 9, 11),         # 9 steps: odd
    (1, 3, 2, 80, 48, 17, 13),        # split K over four waves, ragged channels
    (1, 3, 1, 96, 128, 13, 13),       # 72 steps: split K over eight waves
    (1, 3, 1, 48, 464, 6, 7),         # 261 steps: sixteen waves, uneven shares
    (1, 5, 1, 16, 48, 12, 12),        # 75 steps: an uneven share per wave
    (6, 1, 1, 128, 112, 29, 31),      # whole tiles
    (24, 3, 1, 64, 32, 28, 28),
    (40, 1, 1, 256, 64, 28, 28),      # two channel tiles per wave
    (20, 3, 2, 128, 64, 57, 57),
    (16, 3, 1, 128, 64, 52, 52),      # whole tiles, 164 of them in the last round
    (15, 3, 1, 64, 64, 56, 56),       # cut tail: 112 left over
    (8, 3, 1, 512, 160, 13, 13),      # 90 steps: split K over eight waves
    (16, 3, 1, 512, 240, 13, 13),     # equal shares of the reduction (equal_shares below)
    (56, 3, 1, 128, 64, 56, 56),      # 2 x 2 tiles
    (40, 1, 1, 48, 64, 31, 31),       # pairs of channel tiles with a last tile that is half there
    (20, 3, 1, 208, 48, 23, 25),      # ... that is not there, ragged channels
    (50, 3, 1, 96, 32, 30, 30),       # one channel tile, two pixel tiles a wave
    (13, 3, 1, 32, 32, 105, 103),     # the same with one channel tile in all, odd map
]


def equal_shares(shape):
    """Does the launcher cut this shape into equal shares?  Those launches alone need scratch."""
    n, k, s, co, ci, h, w = shape
    return capi.load().small_hip_conv2d_f32_workspace_bytes(n, k, k, s, *capi.calc_padding(h, k, s), *capi.calc_padding(w, k, s), co, ci, h, w) > 0


def test_equal_share_shapes():
    assert [s for s in SHAPES if equal_shares(s)] == [(16, 3, 1, 512, 240, 13, 13)]
    assert [s for s in FORMS if equal_shares(s)] == [(16, 3, 1, 512, 240, 13, 13)]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("pool", [False, True])
def test_error_against_float64(shape, pool):
    n, k, s, co, ci, h, w = shape
    if pool and min(capi.out_dim(d, *capi.calc_padding(d, k, s), k, s) for d in (h, w)) < 2:
        pytest.skip("no pooling window fits")
    x = synth.normal(11, n * ci * h * w).reshape(n, ci, h, w)
    f = synth.he_normal(12, co * ci * k * k, ci * k * k).reshape(co, ci, k, k)
    bias = synth.normal(13, co, 0.1)
    got, pads = run(shape, x, f, bias, capi.ACT_NONE, pool)
    ref = reference(x, f, bias, s, pads)
    if pool:
        ref = ref[:, :, :ref.shape[2] // 2 * 2, :ref.shape[3] // 2 * 2]
        ref = ref.reshape(n, co, ref.shape[2] // 2, 2, ref.shape[3] // 2, 2).max((3, 5))
    rel = np.linalg.norm(got - ref) / np.linalg.norm(ref)
    steps = k * k * ci // 16
    assert rel <= 2.0 ** -24 * (2 + 2 * 0.41 * steps ** 0.5), (rel, steps)


@pytest.mark.parametrize("shape", [(1, 3, 1, 32, 32, 9, 9), (1, 3, 1, 32, 128, 9, 9), (24, 3, 1, 64, 32, 28, 28)])
def test_infinities_and_nan_as_float32(shape):
    """One infinite and one NaN input: infinite or NaN outputs exactly where float arithmetic has them."""
    n, k, s, co, ci, h, w = shape
    x = synth.normal(21, n * ci * h * w).reshape(n, ci, h, w)
    f = synth.he_normal(22, co * ci * k * k, ci * k * k).reshape(co, ci, k, k)
    f[3] = 0.0
    x[0, 5, 2, 2], x[0, 7, 6, 6] = np.inf, np.nan
    got, pads = run(shape, x, f, None, capi.ACT_NONE)
    ref = reference(x, f, None, s, pads)
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    assert np.array_equal(np.isinf(got), np.isinf(ref)) and np.array_equal(got[np.isinf(ref)], ref[np.isinf(ref)])
    ok = np.isfinite(ref)
    assert np.linalg.norm(got[ok] - ref[ok]) <= 1e-6 * np.linalg.norm(ref[ok])


def test_range():
    """Magnitudes from 2^-100 to 2^100: float32 precision; below 2^-110 an absolute error of 2^-133 of the other factor."""
    shape = (1, 1, 1, 16, 16, 4, 8)
    f = np.eye(16, dtype=np.float32).reshape(16, 16, 1, 1)
    x = synth.normal(31, 16 * 32).reshape(1, 16, 4, 8)
    x *= np.exp2(np.linspace(-100, 100, 32)).astype(np.float32).reshape(1, 1, 4, 8)
    got, _ = run(shape, x, f, None, capi.ACT_NONE)
    assert np.array_equal(got, x)                        # times one and zero: exact
    tiny = x * np.float32(2.0 ** -24) * np.exp2(-np.linspace(0, 200, 32)).astype(np.float32).reshape(1, 1, 4, 8)
    got, _ = run(shape, tiny, f, None, capi.ACT_NONE)
    assert np.abs(got.astype(np.float64) - tiny).max() <= 2.0 ** -133


def test_largest_finite_numbers():
    """The largest float32 numbers (lowest values used as masks among them) stay finite: they have no bf16 neighbour above."""
    shape = (1, 1, 1, 16, 16, 4, 8)
    big = np.finfo(np.float32).max
    x = synth.normal(41, 16 * 32).reshape(1, 16, 4, 8)
    x[0, 3], x[0, 5, 1], x[0, 6, 2] = big, -big, np.nextafter(big, 0)
    f = np.zeros((16, 16, 1, 1), np.float32)
    f[np.arange(16), np.arange(16)] = 0.25
    got, _ = run(shape, x, f, None, capi.ACT_NONE)
    assert np.array_equal(got, x * np.float32(0.25))


# One shape for each form of the kernels: batch, window, stride, Co, Ci, H, W
FORMS = [
    (2, 1, 1, 48, 16, 7, 5),          # one K-step
    (6, 1, 1, 128, 64, 29, 31),       # whole tiles
    (1, 3, 2, 80, 48, 17, 13),        # split K: four, eight and sixteen waves
    (1, 3, 1, 96, 128, 13, 13),
    (1, 3, 1, 48, 464, 6, 7),
    (40, 1, 1, 256, 64, 28, 28),      # two channel tiles a wave
    (13, 3, 1, 32, 32, 105, 103),     # two pixel tiles a wave
    (56, 3, 1, 128, 64, 56, 56),      # 2 x 2
    (16, 3, 1, 128, 64, 52, 52),      # whole tiles, 164 of them in the last round
    (15, 3, 1, 64, 64, 56, 56),       # cut tail: 112 left over
    (16, 3, 1, 512, 240, 13, 13),     # equal shares of the reduction
]
PAIR_CHANNELS = [16, 32, 48, 64, 96, 128]    # input channels of the pointwise + depthwise kernel


def run_pair(ci, co, n, h, w, x, f):
    """Pointwise + depthwise in one launch, the depthwise window passing its centre through: the pointwise sums themselves."""
    lib = capi.load()
    centre = np.zeros((co, 3, 3), np.float32)
    centre[:, 1, 1] = 1.0
    dx, df, dd = dev(layout.pack_activations(x)), dev(layout.pack_conv_filter(f)), dev(layout.pack_dw_filter(centre))
    y = dev_empty(n * co * h * w, np.float32)
    capi.check(lib.small_hip_conv2d_bias_act_dwconv2d_bias_act_f32(n, 1, 1, 1, 0, 0, 0, 0, 3, 3, 1, 1, 1, 1, 1, co, ci, h, w, ptr(dx), ptr(df),
                                                                   None, ptr(dd), None, capi.ACT_NONE, 0.0, ptr(y), stream()))
    return layout.unpack_activations(host(y), n, co, h, w)


def sparse_filter(shape, products):
    """`products` weights of full precision in each output channel, the rest zero."""
    n, k, s, co, ci, h, w = shape
    rng = np.random.default_rng(5)
    f = np.zeros((co, ci * k * k), np.float32)
    for c in range(co):
        f[c, rng.choice(ci * k * k, products, replace=False)] = rng.standard_normal(products)
    return f.reshape(co, ci, k, k)


def check_few(got, x, f, s, pads, products):
    ref, size = reference(x, f, None, s, pads), reference(np.abs(x), np.abs(f), None, s, pads)
    err = got - ref
    assert (np.abs(err) <= 2.05 * 2.0 ** -24 * products * size).all()
    # sqrt of 1 (the products) plus (2 + ... + products) / products (the sums of the first i of them)
    limit = 2.75e-8 * (1 + (products * (products + 1) / 2 - 1) / products) ** 0.5
    assert np.linalg.norm(err) <= limit * np.linalg.norm(ref), np.linalg.norm(err) / np.linalg.norm(ref)


@pytest.mark.parametrize("products", [1, 2, 3, 6])
@pytest.mark.parametrize("shape", FORMS, ids=str)
def test_few_products(shape, products):
    """Sums of a few products (permuting, scaling, sparse filters).  Each product leaves out ml + lm, below 2 x 2^-8 x 2^-17 =
    2^-24 of it; another 2^-24 is the rounding of the sum.  Root mean square: float32 products of normal numbers are rounded by
    2.5e-8 of themselves, and so is each sum of two; 2.75e-8 leaves a tenth for the three products left out (2.6e-8 measured), and
    every product may be rounded by itself and added to the others in turn, as where workgroups or waves share a reduction."""
    n, k, s, co, ci, h, w = shape
    x = synth.normal(51, n * ci * h * w).reshape(n, ci, h, w)
    f = sparse_filter(shape, products)
    got, pads = run(shape, x, f, None, capi.ACT_NONE)
    check_few(got, x, f, s, pads, products)


@pytest.mark.parametrize("products", [1, 2, 3, 6])
@pytest.mark.parametrize("ci", PAIR_CHANNELS)
def test_few_products_pair(ci, products):
    x = synth.normal(52, 3 * ci * 29 * 31).reshape(3, ci, 29, 31)
    f = sparse_filter((3, 1, 1, 64, ci, 29, 31), products)
    check_few(run_pair(ci, 64, 3, 29, 31, x, f), x, f, 1, (0, 0, 0, 0), products)


def special_input(n, ci, h, w, value):
    x = synth.normal(61, n * ci * h * w).reshape(n, ci, h, w)
    x.view(np.uint32)[n // 2, ci - 3, h // 2, w // 3] = value
    return x


def check_special(got, ref):
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    assert np.array_equal(np.isinf(got), np.isinf(ref)) and np.array_equal(got[np.isinf(ref)], ref[np.isinf(ref)])
    ok = np.isfinite(ref)
    assert np.linalg.norm(got[ok] - ref[ok]) <= 2e-6 * np.linalg.norm(ref[ok])


# infinity; NaN: quiet, with a payload in the low half alone (signalling), and negative
SPECIALS = [0x7f800000, 0x7fc00000, 0x7f800001, 0xff80ffff, 0x7fa00000]


@pytest.mark.parametrize("value", SPECIALS, ids=hex)
@pytest.mark.parametrize("where", ["input", "filter"])
@pytest.mark.parametrize("shape", FORMS, ids=str)
def test_specials(shape, where, value):
    """One infinity or NaN among the inputs or the filter's values: infinite or NaN outputs exactly where float arithmetic has them."""
    n, k, s, co, ci, h, w = shape
    x = special_input(n, ci, h, w, value) if where == "input" else synth.normal(61, n * ci * h * w).reshape(n, ci, h, w)
    f = synth.he_normal(62, co * ci * k * k, ci * k * k).reshape(co, ci, k, k)
    if where == "filter":
        f.view(np.uint32)[co - 2, ci // 2, k // 2, k // 2] = value        # (the middle tap: padding would multiply it by zero)
    got, pads = run(shape, x, f, None, capi.ACT_NONE)
    check_special(got, reference(x, f, None, s, pads))


@pytest.mark.parametrize("value", SPECIALS, ids=hex)
@pytest.mark.parametrize("ci", PAIR_CHANNELS)
def test_specials_pair(ci, value):
    x = special_input(3, ci, 29, 31, value)
    f = synth.he_normal(62, 64 * ci, ci).reshape(64, ci, 1, 1)
    got = run_pair(ci, 64, 3, 29, 31, x, f)
    # the centre tap passes a value, the others multiply it by zero: a neighbour of an infinity or NaN is NaN
    ref = reference(x, f, None, 1, (0, 0, 0, 0))
    odd = np.zeros_like(ref, bool)
    bad = np.pad(~np.isfinite(ref), ((0, 0), (0, 0), (1, 1), (1, 1)))
    for i in range(3):
        for j in range(3):
            if (i, j) != (1, 1):
                odd |= bad[:, :, i:i + 29, j:j + 31]
    ref[odd] = np.nan
    check_special(got, ref)


@pytest.mark.parametrize("scale_x, scale_f", [(-60, -60), (-100, 20), (20, -110), (-115, 30), (-70, 0), (127, -20), (0, 100)])
@pytest.mark.parametrize("shape", FORMS, ids=str)
def test_scaled(shape, scale_x, scale_f):
    """Operands scaled by powers of two far from 1: the precision that the unscaled sums have, down to where float32 itself
    ends (a product below 2^-126 is rounded to a multiple of 2^-149)."""
    n, k, s, co, ci, h, w = shape
    # between 1 and 2 in magnitude: no product far below the others
    rng = np.random.default_rng(7)
    x = (rng.uniform(1, 1.99, (n, ci, h, w)) * rng.choice((-1, 1), (n, ci, h, w))).astype(np.float32) * np.float32(2.0 ** scale_x)
    f = (rng.uniform(1, 2, (co, ci, k, k)) * rng.choice((-1, 1), (co, ci, k, k))).astype(np.float32) * np.float32(2.0 ** scale_f)
    f[:, 1:] *= np.float32(2.0 ** -6)                                     # (sums of the largest operands stay finite)
    got, pads = run(shape, x, f, None, capi.ACT_NONE)
    ref = reference(x, f, None, s, pads)
    steps = k * k * ci // 16
    tol = 2.0 ** -24 * (2 + 2 * 0.9 * steps ** 0.5) * np.linalg.norm(ref) + 2.0 ** -149 * 16 * steps * ref.size ** 0.5
    assert np.linalg.norm(got - ref) <= tol, (np.linalg.norm(got - ref) / np.linalg.norm(ref), steps)


@pytest.mark.parametrize("shape", FORMS, ids=str)
def test_overflow(shape):
    """Finite operands whose products overflow: the infinities of float arithmetic."""
    n, k, s, co, ci, h, w = shape
    x = synth.normal(71, n * ci * h * w).reshape(n, ci, h, w)
    f = np.zeros((co, ci, k, k), np.float32)
    f[:, 0, k // 2, k // 2] = np.float32(3.0e38)
    x[:, 0] = np.where(np.abs(x[:, 0]) < 0.5, 0.25, np.sign(x[:, 0]) * 2.0)
    got, pads = run(shape, x, f, None, capi.ACT_NONE)
    with np.errstate(over="ignore"):
        ref = reference(x, f, None, s, pads).astype(np.float32)
    assert np.array_equal(got, ref)
