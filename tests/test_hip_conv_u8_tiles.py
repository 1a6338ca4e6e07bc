"""The uint8 convolution's LDS-staged kernel: every tile width and K-step remainder, odd channel block counts on either side, the
limits of its zero points, against the CPU oracle; large launches against the same images one at a time (bytes equal)."""
import numpy as np
import pytest

from oracle.binding import quant as oq_
from smallframework_amd import capi, synth
from util import assert_equal_exact
import hip_util as hu

pytestmark = pytest.mark.gpu
CB = 16


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


ORACLE_SHAPES = [  # batch, window, stride, padding, Co, Ci, H, W
    (1, 1, 1, 0, 32, 32, 1, 1),        # one pixel, one pair
    (1, 3, 1, 1, 32, 64, 11, 13),      # 18 pairs: two left over in the last round
    (3, 3, 2, 1, 64, 96, 17, 9),
    (2, 3, 1, 2, 80, 112, 12, 10),     # odd numbers of channel blocks, padding wider than the window's half
    (1, 5, 1, 2, 96, 32, 9, 20),
    (1, 1, 1, 0, 1008, 160, 3, 3),
    (50, 1, 1, 0, 96, 48, 31, 33),     # 96 channels a workgroup, half-empty pairs
    (25, 3, 1, 1, 64, 32, 45, 45),     # 64 channels a workgroup
    (50, 1, 1, 0, 128, 32, 32, 31),    # 128 channels a workgroup
    (60, 3, 1, 1, 16, 64, 30, 30),     # a half-empty channel tile on a full chip
]


@pytest.mark.parametrize("zi", [-128, 0, -255, -256, 5])
@pytest.mark.parametrize("shape", ORACLE_SHAPES, ids=str)
def test_against_oracle(oracle, shape, zi):
    if zi not in (-128, 0) and shape[0] * shape[6] * shape[7] > 10000:
        pytest.skip("zero point limits on the small shapes")
    n, k, s, p, co, ci, h, w = shape
    x, f = data(shape)
    oq = out_quant(shape)
    got = run(shape, x, f, zi, -119, oq)
    rc, want = oracle.conv2d_u8(n, CB, k, k, s, p, p, p, p, co, ci, h, w, x, oq_(zi), f, oq_(-119), oq_(oq.zero, oq.multiplier, oq.lshift, oq.rshift))
    assert rc == 0
    assert zi not in (-128,) or len(np.unique(want)) > 3
    assert_equal_exact(got, want, str((shape, zi)))


@pytest.mark.parametrize("oq", [(0, 1 << 30, 0, 0), (7, (1 << 31) - 1, 0, 7), (0, 1 << 30, 3, 14), (0, -(1 << 30), 0, 9)], ids=str)
def test_requantisation_forms(oracle, oq):
    shape = (1, 3, 1, 1, 32, 64, 11, 13)
    x, f = data(shape)
    n, k, s, p, co, ci, h, w = shape
    rc, want = oracle.conv2d_u8(n, CB, k, k, s, p, p, p, p, co, ci, h, w, x, oq_(-128), f, oq_(-128), oq_(*oq))
    assert rc == 0
    assert_equal_exact(run(shape, x, f, -128, -128, hu.q(*oq)), want, str(oq))


@pytest.mark.parametrize("relu", [0, 1])
@pytest.mark.parametrize("with_accum", [False, True])
@pytest.mark.parametrize("shape", [(1, 3, 1, 1, 48, 64, 11, 13), (3, 3, 2, 1, 64, 96, 17, 9)], ids=str)
def test_accum_and_relu(oracle, shape, with_accum, relu):
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


@pytest.mark.parametrize("shape", [(33, 3, 1, 1, 128, 128, 55, 57), (40, 3, 1, 1, 144, 112, 31, 29)], ids=str)
def test_images_of_a_large_batch_alone(shape):
    """Two pixel tiles a wave (first shape) / 64 channels a workgroup; one image takes 32 channels a workgroup."""
    n, k, s, p, co, ci, h, w = shape
    x, f = data(shape)
    oq = out_quant(shape)
    got = run(shape, x, f, -128, -119, oq).reshape(n, -1)
    for i in (0, n // 2, n - 1):
        one = run((1,) + shape[1:], x.reshape(n, -1)[i].copy(), f, -128, -119, oq)
        assert_equal_exact(got[i], one, str((shape, i)))
