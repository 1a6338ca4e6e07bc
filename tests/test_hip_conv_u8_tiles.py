"""The uint8 convolution's LDS-staged kernel: every tile width and K-step remainder, odd channel block counts on either side, the
limits of its zero points, grouped and 1-D launches, against the CPU oracle; large launches against the same images one at a
time (bytes equal).  kernel_of restates the launcher's rule, so that a case that would take another kernel fails."""
import numpy as np
import pytest

from oracle.binding import quant as oq_
from smallframework_amd import capi, synth
from util import assert_equal_exact
import hip_util as hu

pytestmark = pytest.mark.gpu
CB = 16


def kernel_of(n, kh, kw, co, ci, ho, wo, slabs=1, zi=-128, short=True):
    """("lds", 32-channel tiles and 32-pixel tiles a wave, odd channel blocks, rounds left over from pairs of them) or
    ("16x16", channel blocks, 16-pixel groups a wave)."""
    cob, cib, px, taps = co // CB, ci // CB, n * ho * wo, kh * kw
    cop, kpt = (cob + 1) // 2, (cib + 1) // 2

    def groups(ct, pxt):
        return -(-cop // ct) * -(-px // (128 * pxt)) * slabs
    used = cob / (2 * cop) * cib / (2 * kpt)
    if short and -255 <= zi <= 0 and (used >= 0.7 or (used >= 0.45 and groups(1, 1) >= 384)) and (groups(1, 1) >= 64 or taps * kpt >= 24):
        ct, best = 1, 0.0
        for c in (1, 2, 3, 4):
            cost = -(-cop // c) * (c + 0.5)
            if c == 1 or (cost < best and groups(c, 1) >= 384):
                ct, best = c, cost
        pxt = 2 if ct == 4 and groups(4, 2) >= 384 and taps * kpt >= 32 else 1
        return "lds", ct, pxt, cib % 2, -(-taps * kpt // (4 if pxt == 1 else 2)) % 2
    for c, pxt in ((4, 2), (2, 2), (1, 2)):
        if cob % c == 0 and -(-cob // c) * -(-px // (64 * pxt)) * slabs >= 512:
            return "16x16", c, pxt
    return "16x16", 1, 1


def kernel_for(shape, zi=-128, short=True):
    n, k, s, p, co, ci, h, w = shape
    return kernel_of(n, k, k, co, ci, capi.out_dim(h, p, p, k, s), capi.out_dim(w, p, p, k, s), zi=zi, short=short)


def run(shape, x, f, zi, zf, oq, accum=None, aq=None, relu=0):
    n, k, s, p, co, ci, h, w = shape
    lib = capi.load()
    ho, wo = capi.out_dim(h, p, p, k, s), capi.out_dim(w, p, p, k, s)
    do = hu.dev_empty(n * co * ho * wo, np.uint8)
    iq, fq = hu.q(zi), hu.q(zf)
    dx, df = hu.dev(x), hu.dev(f)
    da = hu.dev(accum) if accum is not None else None
    args = (n, k, k, s, p, p, p, p, co, ci, h, w, hu.ptr(dx), hu.qref(iq), hu.ptr(df), hu.qref(fq))
    if accum is None and not relu:
        capi.check(lib.small_hip_conv2d_u8(*args, hu.ptr(do), hu.qref(oq), hu.stream()))
    else:
        capi.check(lib.small_hip_conv2d_accum_relu_u8(*args, hu.ptr(da), hu.qref(aq) if aq else None, relu, hu.ptr(do), hu.qref(oq), hu.stream()))
    return hu.host(do)


def data(shape):
    n, k, s, p, co, ci, h, w = shape
    return synth.uniform_u8(31, n * ci * h * w), synth.uniform_u8(32, co * ci * k * k)


def out_quant(shape, z=3):
    n, k, s, p, co, ci, h, w = shape
    spread = 74.0 * 74.0 * (ci * k * k) ** 0.5
    return hu.q(z, 1518500250, 0, min(15, max(0, int(np.log2(0.7 * spread / 100.0)))))


SMALL_SHAPES = [   # batch, window, stride, padding, Co, Ci, H, W -> kernel_of
    ((1, 1, 1, 0, 32, 768, 1, 1), ("lds", 1, 1, 0, 0)),          # one pixel
    ((1, 3, 1, 1, 32, 96, 5, 4), ("lds", 1, 1, 0, 1)),           # 27 pairs: three left over in the last round
    ((1, 3, 1, 1, 32, 112, 11, 13), ("lds", 1, 1, 1, 1)),        # an odd number of channel blocks
    ((3, 3, 2, 1, 64, 96, 17, 9), ("lds", 1, 1, 0, 1)),
    ((2, 3, 1, 2, 80, 112, 12, 10), ("lds", 1, 1, 1, 1)),        # ... on either side, padding wider than the window's half
    ((1, 5, 1, 2, 96, 32, 9, 20), ("lds", 1, 1, 0, 1)),          # 25 pairs: one left over
    ((1, 1, 1, 0, 32, 32, 1, 1), ("16x16", 1, 1)),               # too short a reduction for the LDS kernel
    ((1, 3, 1, 1, 32, 64, 11, 13), ("16x16", 1, 1)),
    ((1, 1, 1, 0, 1008, 160, 3, 3), ("16x16", 1, 1)),
]
LARGE_SHAPES = [
    ((60, 3, 1, 1, 16, 64, 30, 30), ("lds", 1, 1, 0, 1)),        # a half-empty channel tile on a full chip
    ((25, 3, 1, 1, 64, 32, 45, 45), ("lds", 2, 1, 0, 1)),        # 64 channels a workgroup
    ((20, 1, 1, 0, 192, 48, 31, 31), ("lds", 2, 1, 1, 1)),       # ... half-empty pairs
    ((50, 1, 1, 0, 96, 48, 31, 33), ("lds", 3, 1, 1, 1)),        # 96
    ((50, 1, 1, 0, 128, 32, 32, 31), ("lds", 4, 1, 0, 1)),       # 128
    ((30, 1, 1, 0, 256, 48, 31, 31), ("lds", 4, 1, 1, 1)),
]
# what the LDS kernel is left without on large launches: zero points that are not minus a byte
OTHER_ZERO_POINTS = [((50, 1, 1, 0, 128, 48, 31, 33), ("16x16", 4, 2)), ((50, 1, 1, 0, 96, 48, 31, 33), ("16x16", 2, 2)),
                     ((50, 1, 1, 0, 48, 48, 31, 33), ("16x16", 1, 2))]


def check_oracle(oracle, shape, zi):
    n, k, s, p, co, ci, h, w = shape
    x, f = data(shape)
    oq = out_quant(shape)
    got = run(shape, x, f, zi, -119, oq)
    rc, want = oracle.conv2d_u8(n, CB, k, k, s, p, p, p, p, co, ci, h, w, x, oq_(zi), f, oq_(-119), oq_(oq.zero, oq.multiplier, oq.lshift, oq.rshift))
    assert rc == 0
    assert zi not in (-128,) or len(np.unique(want)) > 3
    assert_equal_exact(got, want, str((shape, zi)))


@pytest.mark.parametrize("zi", [-128, 0, -255, -256, 5])
@pytest.mark.parametrize("shape, kernel", SMALL_SHAPES, ids=str)
def test_against_oracle(oracle, shape, kernel, zi):
    assert kernel_for(shape) == kernel and (-255 <= zi <= 0 or kernel_for(shape, zi)[0] == "16x16")
    check_oracle(oracle, shape, zi)


@pytest.mark.parametrize("zi", [-128, 0, -255])
@pytest.mark.parametrize("shape, kernel", LARGE_SHAPES, ids=str)
def test_large_against_oracle(oracle, shape, kernel, zi):
    assert kernel_for(shape, zi) == kernel
    check_oracle(oracle, shape, zi)


@pytest.mark.parametrize("zi", [-256, 5])
@pytest.mark.parametrize("shape, kernel", OTHER_ZERO_POINTS, ids=str)
def test_other_zero_points_on_large_launches(oracle, shape, kernel, zi):
    assert kernel_for(shape, zi) == kernel
    check_oracle(oracle, shape, zi)


@pytest.mark.parametrize("oq", [(0, 1 << 30, 0, 0), (7, (1 << 31) - 1, 0, 7), (0, 1 << 30, 3, 14), (0, -(1 << 30), 0, 9)], ids=str)
@pytest.mark.parametrize("shape", [(1, 3, 1, 1, 32, 96, 11, 13), (1, 3, 1, 1, 32, 64, 11, 13)], ids=str)
def test_requantisation_forms(oracle, shape, oq):
    """The LDS kernel's short requantisation and the 16x16 kernel's; a negative multiplier takes the general form there."""
    assert kernel_for(shape, short=oq[1] > 0)[0] == ("lds" if shape[5] == 96 and oq[1] > 0 else "16x16")
    x, f = data(shape)
    n, k, s, p, co, ci, h, w = shape
    rc, want = oracle.conv2d_u8(n, CB, k, k, s, p, p, p, p, co, ci, h, w, x, oq_(-128), f, oq_(-128), oq_(*oq))
    assert rc == 0
    assert_equal_exact(run(shape, x, f, -128, -128, hu.q(*oq)), want, str(oq))


@pytest.mark.parametrize("relu", [0, 1])
@pytest.mark.parametrize("with_accum", [False, True])
@pytest.mark.parametrize("shape, kernel", [((1, 3, 1, 1, 48, 64, 11, 13), ("16x16", 1, 1)), ((1, 3, 1, 1, 48, 96, 11, 13), ("lds", 1, 1, 0, 1)),
                                           SMALL_SHAPES[3]] + LARGE_SHAPES[2:], ids=str)
def test_accum_and_relu(oracle, shape, kernel, with_accum, relu):
    assert kernel_for(shape) == kernel
    n, k, s, p, co, ci, h, w = shape
    x, f = data(shape)
    oq = out_quant(shape, -100)
    q = oq_(oq.zero, oq.multiplier, oq.lshift, oq.rshift)
    ho, wo = capi.out_dim(h, p, p, k, s), capi.out_dim(w, p, p, k, s)
    short = synth.uniform_u8(33, n * co * ho * wo) if with_accum else None
    got = run(shape, x, f, -128, -119, oq, short, hu.q(-90) if with_accum else None, relu)
    rc, want = oracle.conv2d_u8(n, CB, k, k, s, p, p, p, p, co, ci, h, w, x, oq_(-128), f, oq_(-119), q)
    if with_accum:
        rc, want = oracle.accum_u8(n, CB, co, ho, wo, short, oq_(-90), want, q)
    if relu:
        rc, want = oracle.relu_u8(n, CB, co, ho, wo, want, q, q)
    assert_equal_exact(got, want, str((shape, with_accum, relu)))


@pytest.mark.parametrize("post", [False, True])
@pytest.mark.parametrize("shape, kernel", [((33, 3, 1, 1, 128, 128, 55, 57), ("lds", 4, 2, 0, 0)), ((33, 3, 1, 1, 128, 112, 55, 57), ("lds", 4, 2, 1, 0)),
                                           ((34, 1, 1, 0, 128, 1040, 55, 55), ("lds", 4, 2, 1, 1)), ((40, 3, 1, 1, 144, 112, 31, 29), ("lds", 3, 1, 1, 1))],
                         ids=str)
def test_images_of_a_large_batch_alone(shape, kernel, post):
    """Two pixel tiles a wave, too large for the oracle: one image takes 32 channels a workgroup and one pixel tile.  The last
    shape: 96 channels a workgroup, a half-empty pair and a half-empty tile."""
    assert kernel_for(shape) == kernel and kernel_for((1,) + shape[1:])[:3] == ("lds", 1, 1)
    n, k, s, p, co, ci, h, w = shape
    x, f = data(shape)
    oq = out_quant(shape)
    ho, wo = capi.out_dim(h, p, p, k, s), capi.out_dim(w, p, p, k, s)
    short = synth.uniform_u8(33, n * co * ho * wo).reshape(n, -1) if post else [None] * n
    aq = hu.q(-90) if post else None
    got = run(shape, x, f, -128, -119, oq, short if post else None, aq, int(post)).reshape(n, -1)
    for i in (0, n // 2, n - 1):
        one = run((1,) + shape[1:], x.reshape(n, -1)[i].copy(), f, -128, -119, oq, short[i], aq, int(post))
        assert_equal_exact(got[i], one, str((shape, i)))


@pytest.mark.parametrize("case", [  # batch, kh, kw, stride, (t, b, l, r), Co, Ci, H, W
    (2, 3, 5, 1, (1, 1, 2, 2), 32, 96, 21, 23), (2, 1, 7, 2, (0, 0, 3, 3), 64, 128, 20, 41), (3, 5, 1, 1, (2, 2, 0, 0), 96, 80, 33, 30),
    (30, 1, 3, 1, (0, 0, 1, 0), 128, 64, 31, 33), (1, 7, 2, 1, (0, 3, 1, 0), 48, 64, 15, 9)], ids=str)
def test_windows_of_unequal_sides(oracle, case):
    n, kh, kw, s, (t, b, l, r), co, ci, h, w = case
    ho, wo = capi.out_dim(h, t, b, kh, s), capi.out_dim(w, l, r, kw, s)
    assert kernel_of(n, kh, kw, co, ci, ho, wo)[0] == "lds"
    lib = capi.load()
    x, f = synth.uniform_u8(31, n * ci * h * w), synth.uniform_u8(32, co * ci * kh * kw)
    oq = (3, 1518500250, 0, min(15, int(np.log2(0.7 * 74.0 * 74.0 * (ci * kh * kw) ** 0.5 / 100.0))))
    do = hu.dev_empty(n * co * ho * wo, np.uint8)
    iq, fq, q3 = hu.q(-120), hu.q(-119), hu.q(*oq)
    dx, df = hu.dev(x), hu.dev(f)
    capi.check(lib.small_hip_conv2d_u8(n, kh, kw, s, t, b, l, r, co, ci, h, w, hu.ptr(dx), hu.qref(iq), hu.ptr(df), hu.qref(fq), hu.ptr(do),
                                       hu.qref(q3), hu.stream()))
    rc, want = oracle.conv2d_u8(n, CB, kh, kw, s, t, b, l, r, co, ci, h, w, x, oq_(-120), f, oq_(-119), oq_(*oq))
    assert rc == 0 and len(np.unique(want)) > 50
    assert_equal_exact(hu.host(do), want, str(case))


@pytest.mark.parametrize("case", [  # batch, window, padding, groups, channels of a group, H, W -> 32-channel tiles a wave, odd blocks
    (3, 3, 1, 4, 32, 40, 40, 1, 0), (4, 1, 0, 8, 64, 40, 40, 2, 0), (3, 1, 0, 10, 48, 40, 40, 2, 1), (2, 3, 1, 3, 96, 12, 13, 1, 0)], ids=str)
def test_grouped(oracle, case):
    n, k, p, g, cg, h, w, ct, odd = case
    assert kernel_of(1, k, k, cg, cg, h, w, slabs=n * g)[:4] == ("lds", ct, 1, odd)
    lib = capi.load()
    nf = cg * cg * k * k
    x, f = synth.uniform_u8(41, n * g * cg * h * w), synth.uniform_u8(42, g * nf)      # (every filter is a random one, packed or not)
    oq = (0, 1518500250, 0, min(15, int(np.log2(0.7 * 74.0 * 74.0 * (cg * k * k) ** 0.5 / 100.0))))
    do = hu.dev_empty(n * g * cg * h * w, np.uint8)
    iq, fq, q3 = hu.q(-128), hu.q(-128), hu.q(*oq)
    dx, df = hu.dev(x), hu.dev(f)
    capi.check(lib.small_hip_group_conv2d_u8(n, k, k, 1, g, p, p, p, p, cg, h, w, hu.ptr(dx), hu.qref(iq), hu.ptr(df), hu.qref(fq), hu.ptr(do),
                                             hu.qref(q3), hu.stream()))
    rc, want = oracle.group_conv2d_u8(n, CB, k, k, 1, p, p, p, p, g, cg, h, w, x, oq_(-128), f, oq_(-128), oq_(*oq))
    assert rc == 0 and len(np.unique(want)) > 50
    assert_equal_exact(hu.host(do), want, str(case))


@pytest.mark.parametrize("case", [  # batch, window, l, r, groups, Co, Ci, rows, W: stride 2 along the width, rows of their own
    (2, 5, 2, 1, 0, 32, 96, 66, 127), (1, 3, 1, 1, 0, 96, 272, 7, 30), (2, 5, 2, 2, 4, 32, 32, 21, 101), (1, 2, 0, 0, 3, 48, 48, 90, 300)], ids=str)
def test_rows_of_one_dimension(oracle, case):
    n, k, l, r, g, co, ci, rows, w = case
    groups, wo = max(g, 1), 1 + (w + l + r - k) // 2
    assert kernel_of(n if not g else 1, 1, k, co, ci, rows, wo, slabs=n * g if g else 1)[0] == "lds"
    lib = capi.load()
    x, f = synth.uniform_u8(51, n * groups * ci * rows * w), synth.uniform_u8(52, groups * co * ci * k)
    oq = (0, 1518500250, 0, min(15, int(np.log2(0.7 * 74.0 * 74.0 * (ci * k) ** 0.5 / 100.0))))
    do = hu.dev_empty(n * groups * co * rows * wo, np.uint8)
    iq, fq, q3 = hu.q(-125), hu.q(-131), hu.q(*oq)
    dx, df = hu.dev(x), hu.dev(f)
    capi.check(lib.small_hip_conv1d_u8(n, k, 2, l, r, g, co, ci, rows, w, hu.ptr(dx), hu.qref(iq), hu.ptr(df), hu.qref(fq), hu.ptr(do),
                                       hu.qref(q3), hu.stream()))
    got = hu.host(do).reshape(n, groups * co // CB, rows, wo, CB)
    xr = x.reshape(n, groups * ci // CB, rows, w, CB)
    for row in range(rows):
        one = np.ascontiguousarray(xr[:, :, row]).ravel()
        if g:
            rc, want = oracle.group_conv2d_u8(n, CB, 1, k, 2, 0, 0, l, r, g, ci, 1, w, one, oq_(-125), f, oq_(-131), oq_(*oq))
        else:
            rc, want = oracle.conv2d_u8(n, CB, 1, k, 2, 0, 0, l, r, co, ci, 1, w, one, oq_(-125), f, oq_(-131), oq_(*oq))
        assert rc == 0
        assert_equal_exact(np.ascontiguousarray(got[:, :, row]).ravel(), want, str((case, row)))
