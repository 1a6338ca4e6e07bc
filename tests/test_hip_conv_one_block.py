"""3x3 stride-1 convolutions of sixteen input channels on large maps (persistent workgroups, 16 x 16 tiles, the patch split once into
LDS), with and without the 2x2 pooling behind them: against float64 with the bound of a chain of 144 float32 roundings."""
import numpy as np
import pytest

from smallframework_amd import capi, synth
import hip_util as hu

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def lib():
    import torch
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    return capi.load()


def _float64(x, f, bias, n, co, h, w, pads, old, act, slope):
    import torch
    t, b, l, r = pads
    xs = torch.from_numpy(x).double().view(n, h, w, 16).permute(0, 3, 1, 2)
    ws = torch.from_numpy(f).double().view(co // 16, 3, 3, 16, 16).permute(0, 4, 3, 1, 2).reshape(co, 16, 3, 3)
    y = torch.nn.functional.conv2d(torch.nn.functional.pad(xs, (l, r, t, b)), ws)
    ho, wo = y.shape[2:]
    if old is not None:
        y = y + torch.from_numpy(old).double().view(n, co // 16, ho, wo, 16).permute(0, 1, 4, 2, 3).reshape(n, co, ho, wo)
    if bias is not None:
        y = y + torch.from_numpy(bias).double().view(1, -1, 1, 1)
    return torch.relu(y) if act == capi.ACT_RELU else torch.where(y > 0, y, y * slope) if act == capi.ACT_LEAKY else y


def _packed(y):
    n, co, h, w = y.shape
    return y.view(n, co // 16, 16, h, w).permute(0, 1, 3, 4, 2).reshape(-1).numpy()


# images x tiles: one run a workgroup, runs of unequal length, channel groups that are half empty, ragged right and lower edges, pads on
# some sides only (rows and columns that no window covers in the pooled form)
CASES = [(6, 16, 128, 128, (1, 1, 1, 1), True, capi.ACT_RELU), (12, 32, 77, 95, (1, 1, 1, 1), True, capi.ACT_LEAKY),
         (30, 48, 47, 61, (1, 1, 1, 1), False, capi.ACT_NONE), (4, 96, 130, 131, (0, 0, 0, 0), True, capi.ACT_RELU),
         (43, 64, 31, 33, (1, 0, 0, 1), True, capi.ACT_LEAKY), (2, 32, 209, 207, (2, 1, 0, 2), True, capi.ACT_RELU),
         (350, 16, 16, 16, (1, 1, 1, 1), True, capi.ACT_RELU), (25, 32, 111, 110, (1, 1, 1, 1), True, capi.ACT_LEAKY),
         (24, 80, 61, 47, (1, 1, 1, 1), True, capi.ACT_RELU), (24, 192, 61, 47, (1, 1, 1, 1), False, capi.ACT_NONE)]


def runs(n, co, ho, wo):
    """The launcher's rule: (workgroups of a channel group, channel groups), or None where the shape is another kernel's."""
    tiles, groups = n * -(-ho // 16) * -(-wo // 16), -(-co // 32)
    most = 512 // groups // 8 * 8
    if most == 0 or 20 * tiles * groups < 13 * -(-tiles // most) * 512 or 5 * n * ho * wo < 4 * tiles * 256:
        return None
    return min(most, -(-tiles // 8) * 8), groups


@pytest.mark.parametrize("case", CASES, ids=str)
def test_conv3x3_of_one_block(lib, case):
    import torch
    n, co, h, w, pads, has_bias, act = case
    t, b, l, r = pads
    ho, wo = capi.out_dim(h, t, b, 3, 1), capi.out_dim(w, l, r, 3, 1)
    grid = runs(n, co, ho, wo)
    assert grid and grid[0] * grid[1] <= 512, "the case would run in another kernel, or in more workgroups than are resident at once"
    x, f, bias = synth.normal(1, n * 16 * h * w), synth.he_normal(2, co * 144, 144), synth.normal(3, co) if has_bias else None
    old = synth.normal(4, n * co * ho * wo)
    dx, df, db = hu.dev(x), hu.dev(f), hu.dev(bias) if has_bias else None
    pb = hu.ptr(db) if has_bias else None
    bound = 144 ** 0.5 * 2.0 ** -24
    y = hu.dev_empty(n * co * ho * wo, np.float32)
    capi.check(lib.small_hip_conv2d_bias_act_f32(n, 3, 3, 1, t, b, l, r, co, 16, h, w, hu.ptr(dx), hu.ptr(df), pb, act, 0.1, hu.ptr(y), hu.stream()))
    plain, want = hu.host(y), _float64(x, f, bias, n, co, h, w, pads, None, act, 0.1)
    assert np.linalg.norm(plain - _packed(want)) <= bound * np.linalg.norm(_packed(want))
    acc = hu.dev(old)
    capi.check(lib.small_hip_partial_conv2d_bias_act_f32(n, 3, 3, 1, t, b, l, r, co, 16, h, w, hu.ptr(dx), hu.ptr(df), pb, act, 0.1, hu.ptr(acc),
                                                         hu.stream()))
    wacc = _packed(_float64(x, f, bias, n, co, h, w, pads, old, act, 0.1))
    assert np.linalg.norm(hu.host(acc) - wacc) <= bound * np.linalg.norm(wacc)
    # the pooled form multiplies in the same order: the maxima of the plain form's values
    z = hu.dev_empty(n * co * (ho // 2) * (wo // 2), np.float32)
    capi.check(lib.small_hip_conv2d_bias_act_maxpool2d_f32(n, 3, 3, 1, t, b, l, r, 2, 2, 2, 0, 0, 0, 0, co, 16, h, w, hu.ptr(dx), hu.ptr(df), pb,
                                                           act, 0.1, hu.ptr(z), hu.stream()))
    p = torch.from_numpy(plain).view(n, co // 16, ho, wo, 16).permute(0, 1, 4, 2, 3).reshape(n, co, ho, wo)
    assert np.array_equal(hu.host(z), _packed(torch.nn.functional.max_pool2d(p, 2)))


def test_conv3x3_of_one_block_special_values(lib):
    """Sums that are not finite or very small are made again with float32 products: infinities, NaN and the smallest numbers end where
    float64 puts them."""
    n, co, h, w = 5, 32, 130, 126
    assert runs(n, co, h, w)
    x, f = synth.normal(5, n * 16 * h * w), synth.he_normal(6, co * 144, 144)
    rng = np.random.RandomState(7)
    at = rng.choice(x.size, 24, replace=False)
    x[at[:8]], x[at[8:16]], x[at[16:]] = np.inf, -np.inf, np.nan
    x[-16 * w * 40:] *= np.float32(2.0 ** -90)            # the last rows of the last image
    y = hu.dev_empty(n * co * h * w, np.float32)
    dx, df = hu.dev(x), hu.dev(f)
    capi.check(lib.small_hip_conv2d_bias_act_f32(n, 3, 3, 1, 1, 1, 1, 1, co, 16, h, w, hu.ptr(dx), hu.ptr(df), None, capi.ACT_NONE, 0.0, hu.ptr(y),
                                                 hu.stream()))
    got, want = hu.host(y), _packed(_float64(x, f, None, n, co, h, w, (1, 1, 1, 1), None, capi.ACT_NONE, 0.0))
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isposinf(got), np.isposinf(want))
    assert np.array_equal(np.isneginf(got), np.isneginf(want))
    fin = np.isfinite(want)
    small = fin & (np.abs(want) < 2.0 ** -60)
    bound = 144 ** 0.5 * 2.0 ** -24
    assert small.sum() > 1000
    assert np.linalg.norm(got[small] - want[small]) <= bound * np.linalg.norm(want[small])
    rest = fin & ~small
    assert np.linalg.norm(got[rest] - want[rest]) <= bound * np.linalg.norm(want[rest])
