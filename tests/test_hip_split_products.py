"""float32 convolutions against float64: the three-way bf16 split of both operands keeps float32's precision.

Bound on the relative 2-norm of the error.  A product leaves out less than 2^-24 of itself; the running sum of n K-steps
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
    (16, 3, 1, 128, 64, 52, 52),      # cut tail
    (8, 3, 1, 512, 160, 13, 13),      # equal shares of the reduction
    (56, 3, 1, 128, 64, 56, 56),      # 2 x 2 tiles
    (40, 1, 1, 48, 64, 31, 31),       # pairs of channel tiles with a last tile that is half there
    (20, 3, 1, 208, 48, 23, 25),      # ... that is not there, ragged channels
    (50, 3, 1, 96, 32, 30, 30),       # one channel tile, two pixel tiles a wave
    (13, 3, 1, 32, 32, 105, 103),     # the same with one channel tile in all, odd map
]


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
    """Magnitudes from 2^-100 to 2^100: float32 precision; below 2^-110 an absolute error of 2^-134 of the other factor."""
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
