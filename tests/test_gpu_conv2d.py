"""HIP general 2-D convolution (xdna_conv2d_*: any kernel, stride, padding) vs the
float64 oracle, to the conv bar: every output within 2 bf16 ulp of the exact sum of the
bf16 operands (floor at ulp(max|ref| * 2^-8)) and relative L2 <= 1e-2.

Shapes: the style network's 9x9 input / output layers and stride-2 encoder convs,
ResNet's 7x7 stride-2 stem and 1x1 stride-2 downsampling, non-square kernels and
strides, odd sizes, channel counts that leave partial 32 / 64 / 128-row tiles, and a
pixel count beyond one 128-column tile row.  The weight gradient is checked for
run-to-run bit equality (fixed-order split reduction).  Forward and input gradient run
in both kernel forms: automatic (the few-channel kernels where they are the faster ones,
else the direct form at stride 1 with <= 32 output and >= 16 input channels of the
direction, up to the widest padded row it stages) and the gather GEMM alone; the
few-channel kernels wherever they apply have a test of their own.
"""
import numpy as np
import pytest

import oracle
from gpu_util import check_bf16, dev, dev_zeros, host, ptr, stream

pytestmark = pytest.mark.gpu

CASES = [
    # B, Cin, Cout, H, W, KH, KW, sh, sw, ph, pw
    (4, 3, 32, 36, 36, 9, 9, 1, 1, 4, 4),     # style: 9x9 3->32
    (4, 32, 3, 36, 36, 9, 9, 1, 1, 4, 4),     # style: 9x9 32->3
    (4, 32, 64, 36, 36, 3, 3, 2, 2, 1, 1),    # style: 3x3 s2 32->64
    (4, 64, 128, 18, 18, 3, 3, 2, 2, 1, 1),   # style: 3x3 s2 64->128
    (2, 3, 64, 32, 32, 7, 7, 2, 2, 3, 3),     # ResNet stem
    (4, 64, 128, 16, 16, 1, 1, 2, 2, 0, 0),   # ResNet 1x1 s2 downsample
    (3, 40, 70, 9, 11, 1, 1, 1, 1, 0, 0),     # 1x1, partial tiles
    (2, 5, 130, 7, 9, 3, 2, 1, 3, 1, 0),      # non-square kernel and stride
    (1, 1, 1, 1, 1, 1, 1, 1, 1, 0, 0),
    (2, 70, 20, 13, 17, 5, 3, 1, 1, 2, 1),    # direct form: 3 channel chunks (partial), 5x3
    (3, 16, 32, 40, 50, 3, 3, 1, 1, 0, 0),    # direct form: no padding, 7 grid blocks
    (2, 16, 5, 30, 90, 7, 7, 1, 1, 3, 3),     # direct form: wide row (12 grid blocks, 95 KB LDS)
    (2, 6, 4, 20, 200, 3, 3, 1, 1, 1, 1),     # too wide for the direct form: gather GEMM
]


@pytest.fixture(params=[0, 1], ids=["auto", "gather"])
def cvar(request, hip):
    assert hip.xdna_conv2d_set_variant(request.param) == 0
    yield request.param
    hip.xdna_conv2d_set_variant(0)


def _data(case, seed):
    B, Cin, Cout, H, W, KH, KW, sh, sw, ph, pw = case
    rng = np.random.default_rng(seed)
    bound = np.sqrt(6.0 / (Cin * KH * KW))
    x = oracle.rng_bf16(rng, (B, Cin, H, W))
    w = oracle.bf16_bits(rng.uniform(-bound, bound, (Cout, Cin, KH, KW)).astype(np.float32))
    b = oracle.bf16_bits(rng.uniform(-0.1, 0.1, (Cout,)).astype(np.float32))
    Ho, Wo = oracle.conv2d_out_size(H, W, KH, KW, sh, sw, ph, pw)
    dy = oracle.rng_bf16(rng, (B, Cout, Ho, Wo))
    return x, w, b, dy, Ho, Wo


@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c)))
def test_forward(hip, case, cvar):
    B, Cin, Cout, H, W, KH, KW, sh, sw, ph, pw = case
    print(f"conv2d fwd {case} variant {cvar}", flush=True)
    x, w, b, _, Ho, Wo = _data(case, sum(case))
    y = dev_zeros((B, Cout, Ho, Wo))
    assert hip.xdna_conv2d_fwd_bf16(ptr(dev(x)), ptr(dev(w)), ptr(dev(b)), ptr(y), B, Cin, Cout, H, W, KH, KW,
                                    sh, sw, ph, pw, stream()) == 0
    check_bf16(host(y), oracle.conv2d_fwd(x, w, b, (sh, sw), (ph, pw)), what=f"fwd {case}")
    y2 = dev_zeros((B, Cout, Ho, Wo))
    assert hip.xdna_conv2d_fwd_bf16(ptr(dev(x)), ptr(dev(w)), None, ptr(y2), B, Cin, Cout, H, W, KH, KW,
                                    sh, sw, ph, pw, stream()) == 0
    check_bf16(host(y2), oracle.conv2d_fwd(x, w, None, (sh, sw), (ph, pw)), what=f"fwd nobias {case}")


@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c)))
def test_dgrad(hip, case, cvar):
    B, Cin, Cout, H, W, KH, KW, sh, sw, ph, pw = case
    print(f"conv2d dgrad {case} variant {cvar}", flush=True)
    _, w, _, dy, Ho, Wo = _data(case, sum(case) + 1)
    dx = dev_zeros((B, Cin, H, W))
    assert hip.xdna_conv2d_dgrad_bf16(ptr(dev(dy)), ptr(dev(w)), ptr(dx), B, Cin, Cout, H, W, KH, KW, sh, sw,
                                      ph, pw, stream()) == 0
    check_bf16(host(dx), oracle.conv2d_dgrad(dy, w, (H, W), (sh, sw), (ph, pw)), what=f"dgrad {case}")


@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c)))
def test_wgrad(hip, case):
    B, Cin, Cout, H, W, KH, KW, sh, sw, ph, pw = case
    print(f"conv2d wgrad {case}", flush=True)
    x, _, _, dy, Ho, Wo = _data(case, sum(case) + 2)
    gw = dev_zeros((Cout, Cin, KH, KW))
    gb = dev_zeros((Cout,))
    dx_, ddy = dev(x), dev(dy)
    assert hip.xdna_conv2d_wgrad_bf16(ptr(dx_), ptr(ddy), ptr(gw), ptr(gb), B, Cin, Cout, H, W, KH, KW, sh, sw,
                                      ph, pw, stream()) == 0
    ref_w, ref_b = oracle.conv2d_wgrad(x, dy, (KH, KW), (sh, sw), (ph, pw))
    got = host(gw)
    check_bf16(got, ref_w, what=f"wgrad {case}")
    check_bf16(host(gb), ref_b, what=f"bias grad {case}")
    gw2 = dev_zeros((Cout, Cin, KH, KW))
    assert hip.xdna_conv2d_wgrad_bf16(ptr(dx_), ptr(ddy), ptr(gw2), None, B, Cin, Cout, H, W, KH, KW, sh, sw,
                                      ph, pw, stream()) == 0
    np.testing.assert_array_equal(host(gw2), got)


# stride-1 layers with few channels on one side (taps beside the few channels): k pads, tile
# and channel remainders, one few channel and four, paddings from none to the full kernel,
# rows from 4 columns to ones that leave no room for a second workgroup
FEW = [
    (3, 8, 1, 5, 4, 3, 3, 1, 1, 1, 1), (2, 33, 3, 13, 11, 9, 9, 1, 1, 4, 4), (2, 70, 4, 9, 30, 5, 7, 1, 1, 2, 3),
    (2, 3, 70, 13, 17, 9, 9, 1, 1, 4, 4), (3, 1, 40, 7, 9, 5, 3, 1, 1, 0, 0), (2, 4, 33, 12, 20, 3, 5, 1, 1, 2, 4),
    (1, 2, 9, 6, 130, 7, 7, 1, 1, 3, 3), (1, 40, 3, 6, 150, 9, 9, 1, 1, 4, 4), (2, 32, 3, 16, 10, 1, 9, 1, 1, 0, 8),
    (5, 3, 64, 20, 27, 3, 3, 1, 1, 1, 1), (2, 9, 2, 11, 12, 16, 9, 1, 1, 8, 4), (700, 3, 16, 4, 4, 3, 3, 1, 1, 1, 1),
    # paddings up to a kernel's width and past it
    (2, 16, 3, 7, 9, 3, 3, 1, 1, 3, 3), (2, 3, 16, 7, 9, 3, 3, 1, 1, 6, 7), (2, 16, 3, 7, 9, 3, 3, 1, 1, 5, 6),
]


@pytest.mark.parametrize("case", FEW, ids=lambda c: "x".join(map(str, c)))
def test_few_channels(hip, case):
    B, Cin, Cout, H, W, KH, KW, sh, sw, ph, pw = case
    print(f"conv2d few channels {case}", flush=True)
    x, w, b, dy, Ho, Wo = _data(case, sum(case) + 3)
    y, dx = dev_zeros((B, Cout, Ho, Wo)), dev_zeros((B, Cin, H, W))
    gw, gb = dev_zeros((Cout, Cin, KH, KW)), dev_zeros((Cout,))
    d = (B, Cin, Cout, H, W, KH, KW, sh, sw, ph, pw, stream())
    xd, wd, dyd = dev(x), dev(w), dev(dy)
    assert hip.xdna_conv2d_fwd_bf16(ptr(xd), ptr(wd), ptr(dev(b)), ptr(y), *d) == 0
    check_bf16(host(y), oracle.conv2d_fwd(x, w, b, (sh, sw), (ph, pw)), what=f"fwd {case}")
    assert hip.xdna_conv2d_dgrad_bf16(ptr(dyd), ptr(wd), ptr(dx), *d) == 0
    check_bf16(host(dx), oracle.conv2d_dgrad(dy, w, (H, W), (sh, sw), (ph, pw)), what=f"dgrad {case}")
    assert hip.xdna_conv2d_wgrad_bf16(ptr(xd), ptr(dyd), ptr(gw), ptr(gb), *d) == 0
    ref_w, ref_b = oracle.conv2d_wgrad(x, dy, (KH, KW), (sh, sw), (ph, pw))
    check_bf16(host(gw), ref_w, what=f"wgrad {case}")
    check_bf16(host(gb), ref_b, what=f"bias grad {case}")


# which kernel applies to each of those, forward, input gradient and weight gradient (1 few outputs,
# 2 few inputs, 3 the weight gradient's, 0 none: paddings past the kernel), and two layers of more
# wide channels than a tile
FEW_ROUTES = [(1, 2, 3)] * 3 + [(2, 1, 3)] * 4 + [(1, 2, 3)] * 2 + [(2, 1, 3), (1, 2, 3), (2, 1, 3), (1, 0, 3), (2, 0, 0), (1, 0, 0)]
FEW_APPLY = list(zip(FEW, FEW_ROUTES)) + [((1, 300, 3, 6, 9, 3, 3, 1, 1, 1, 1), (1, 2, 3)),
                                          ((1, 3, 300, 6, 9, 3, 3, 1, 1, 1, 1), (2, 1, 3))]


@pytest.fixture
def few_everywhere(hip):
    assert hip.xdna_conv2d_set_variant(2) == 0
    yield
    assert hip.xdna_conv2d_set_variant(0) == 0


@pytest.mark.parametrize("case,routes", FEW_APPLY, ids=lambda c: "x".join(map(str, c)))
def test_few_channels_wherever_they_apply(hip, case, routes, few_everywhere):
    """The few-channel kernels at the edges of their tiles, whichever kernels the choice would take."""
    assert tuple(hip.xdna_conv2d_few_pick(op, *case[:7], *case[9:], 1) for op in range(3)) == routes
    test_few_channels(hip, case)


@pytest.mark.parametrize("cin,cout", [(12, 3), (3, 12)])
def test_few_channels_keep_infinities_wherever_they_apply(hip, cin, cout, few_everywhere):
    test_few_channels_keep_infinities_in_their_pairs(hip, cin, cout)


@pytest.mark.parametrize("cin,cout", [(12, 3), (3, 12)])
def test_few_channels_keep_infinities_in_their_pairs(hip, cin, cout):
    """An infinity in x reaches the outputs whose window holds it and the weight gradients of
    its own channel, and nothing else (the kernels multiply padding beside it)."""
    B, H, W, K, p = 2, 9, 13, 9, 4
    rng = np.random.default_rng(cin)
    xf = rng.standard_normal((B, cin, H, W)).astype(np.float32)
    xf[1, 2, 0, W - 1] = np.inf
    x = oracle.bf16_bits(xf)
    w = oracle.bf16_bits(rng.uniform(0.1, 1, (cout, cin, K, K)).astype(np.float32))
    dy = oracle.bf16_bits(rng.uniform(0.1, 1, (B, cout, H, W)).astype(np.float32))
    y, gw = dev_zeros((B, cout, H, W)), dev_zeros((cout, cin, K, K))
    d = (B, cin, cout, H, W, K, K, 1, 1, p, p, stream())
    print(f"few channels with an infinity {cin} -> {cout}", flush=True)
    assert hip.xdna_conv2d_fwd_bf16(ptr(dev(x)), ptr(dev(w)), None, ptr(y), *d) == 0
    assert hip.xdna_conv2d_wgrad_bf16(ptr(dev(x)), ptr(dev(dy)), ptr(gw), None, *d) == 0
    finite = np.ones((B, cout, H, W), bool)
    finite[1, :, :p + 1, W - 1 - p:] = False
    np.testing.assert_array_equal(np.isfinite(oracle.bf16_value(host(y))), finite)
    # tap (ky, kx) pairs x[0][W - 1] with dy[p - ky][W - 1 + p - kx] where that exists
    finite = np.ones((cout, cin, K, K), bool)
    finite[:, 2, :p + 1, p:] = False
    got = oracle.bf16_value(host(gw))
    np.testing.assert_array_equal(np.isfinite(got), finite)
    xf[1, 2, 0, W - 1] = 0
    ref, _ = oracle.conv2d_wgrad(oracle.bf16_bits(xf), dy, (K, K), (1, 1), (p, p))
    check_bf16(np.where(finite, host(gw), 0), np.where(finite, ref, 0), what="weight gradient beside an infinity")


def test_invalid_shapes(hip):
    y = dev_zeros((1,))
    assert hip.xdna_conv2d_fwd_bf16(ptr(y), ptr(y), None, ptr(y), 1, 1, 1, 2, 2, 5, 5, 1, 1, 0, 0, stream()) == -1
    assert "kernel larger" in hip.xdna_hip_last_error().decode()
    assert hip.xdna_conv2d_fwd_bf16(ptr(y), ptr(y), None, ptr(y), 1, 1, 1, 2, 2, 1, 1, 0, 1, 0, 0, stream()) == -1


@pytest.mark.parametrize("variant", [0, 1, 2])
@pytest.mark.parametrize("case", [(2, 20, 30, 9, 13, 5, 3, 1, 1, 2, 1), (2, 3, 40, 8, 11, 3, 3, 1, 1, 1, 1),
                                  (2, 24, 3, 8, 11, 5, 5, 1, 1, 2, 2), (2, 3, 70, 17, 15, 7, 7, 2, 2, 3, 3)],
                         ids=lambda c: "x".join(map(str, c)))
def test_forward_with_relu_is_relu_of_the_forward(hip, case, variant):
    """Every forward kernel's ReLU, bit for bit, a NaN kept."""
    B, Cin, Cout, H, W, KH, KW, sh, sw, ph, pw = case
    print(f"conv2d relu {case} variant {variant}", flush=True)
    x, w, b, dy, Ho, Wo = _data(case, sum(case) + 4)
    x[0, 0, 0, 0] = 0x7FC0
    xd, wd, bd = dev(x), dev(w), dev(b)
    plain, relu = dev_zeros((B, Cout, Ho, Wo)), dev_zeros((B, Cout, Ho, Wo))
    assert hip.xdna_conv2d_set_variant(variant) == 0
    try:
        for bias in (None, ptr(bd)):
            assert hip.xdna_conv2d_fwd_bf16(ptr(xd), ptr(wd), bias, ptr(plain), *case, stream()) == 0
            assert hip.xdna_conv2d_fwd_act_bf16(ptr(xd), ptr(wd), bias, ptr(relu), *case, 1, stream()) == 0
            v = host(plain)
            ref = np.where(oracle.bf16_value(v) <= 0, 0, v)
            assert np.isnan(oracle.bf16_value(v)).any()
            np.testing.assert_array_equal(host(relu), ref)
    finally:
        assert hip.xdna_conv2d_set_variant(0) == 0
