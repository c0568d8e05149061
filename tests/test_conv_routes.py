"""Which kernels the conv dispatch takes, at shapes where both sides were measured on an MI355X
(host functions only: nothing is launched)."""
import pytest

from xdna_train import hip_abi


# op (0 forward, 1 input gradient, 2 weight gradient), B, Cin, Cout, H, W, stride: us of the in-place
# kernel, us of the product
CONV1X1 = [
    # a long k, or short strided rows, on few workgroups: the product
    ((0, 8, 993, 512, 14, 1, 2), 127, 15.7), ((0, 13, 675, 64, 91, 6, 2), 90, 20.9), ((0, 39, 512, 64, 7, 10, 2), 53, 12.2),
    ((0, 114, 2048, 1024, 19, 1, 2), 368, 180), ((0, 5, 512, 256, 3, 3, 2), 21.3, 10.7), ((0, 2, 512, 64, 27, 24, 2), 29.8, 9.4),
    ((1, 12, 85, 2048, 2, 2, 1), 101, 13.5), ((1, 2, 64, 2048, 10, 87, 1), 87, 14.6), ((1, 4, 128, 2048, 11, 11, 1), 45, 11.5),
    ((1, 71, 1024, 12, 73, 4, 2), 92, 33), ((1, 36, 30, 512, 2, 2, 1), 27, 10.6),
    ((2, 256, 1935, 256, 3, 3, 2), 273, 59), ((2, 184, 324, 799, 4, 11, 2), 104, 36), ((2, 48, 512, 544, 1, 1, 1), 23, 10),
    ((0, 50, 1024, 2048, 16, 16, 1), 127, 90), ((0, 32, 1024, 1024, 32, 32, 1), 160, 96),
    # many workgroups, short k, planes that fill no product tile: in place
    ((0, 128, 64, 128, 64, 64, 2), 19, 37), ((1, 128, 64, 128, 64, 64, 2), 23, 31), ((2, 128, 64, 128, 64, 64, 2), 21, 85),
    ((0, 128, 64, 256, 56, 56, 1), 57, 137), ((1, 128, 64, 256, 56, 56, 1), 48, 47), ((2, 128, 64, 256, 56, 56, 1), 57, 241),
    ((0, 109, 574, 512, 2, 2, 1), 22, 59), ((1, 48, 2048, 2039, 2, 4, 1), 52, 188), ((1, 190, 1024, 1483, 4, 2, 1), 81, 275),
    ((1, 43, 256, 1024, 16, 16, 1), 21.5, 73), ((2, 3, 1024, 743, 87, 87, 1), 160, 359), ((0, 2, 64, 128, 9, 9, 1), None, None),
]


@pytest.mark.parametrize("shape,here,product", CONV1X1, ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else "")
def test_conv1x1_takes_the_faster_form(shape, here, product):
    want = 1 if here is None or here < 1.05 * product else 0
    assert hip_abi.load().xdna_conv1x1_pick(*shape) == want


# op (0 forward, 1 input gradient, 2 weight gradient, 3 the 3x3 input gradient against the packed-rows
# conv), B, Cin, Cout, H, W, K, padding, bias: us of the few-channel kernel, us of the other
FEW = [
    # batches of planes that fill no tile; one input channel; taps of one k-tile; long chains of chunks
    ((0, 1859, 3, 102, 4, 4, 3, 1, 0), 45, 9.2), ((0, 445, 1, 254, 4, 4, 7, 3, 0), 46, 11.3),
    ((0, 2091, 4, 336, 8, 8, 3, 0, 1), 171, 60), ((1, 430, 194, 1, 2, 2, 9, 4, 0), 65, 12.8),
    ((1, 73, 228, 1, 63, 9, 9, 4, 0), 40.5, 23.0), ((0, 32, 1, 52, 102, 107, 5, 2, 0), 34.5, 23.3),
    ((0, 84, 3, 238, 34, 31, 3, 1, 0), 32.4, 24.2), ((0, 3, 1, 9, 24, 109, 3, 0, 0), 5.7, 4.6),
    ((0, 2032, 9, 3, 5, 5, 3, 0, 0), 15.8, 8.0), ((2, 1266, 3, 254, 4, 4, 5, 2, 0), 94, 29),
    ((2, 4, 3, 22, 45, 22, 9, 4, 0), 14.8, 10.3), ((2, 773, 1, 127, 5, 5, 3, 1, 1), 51.7, 34.8),
    ((3, 1, 3, 163, 23, 30, 3, 1, 0), 17.5, 11.0), ((3, 74, 1, 416, 8, 8, 3, 1, 0), 38, 21),
    ((3, 733, 3, 57, 4, 4, 3, 1, 0), 19.6, 13.6), ((3, 1, 3, 233, 10, 87, 3, 1, 0), 26.6, 13.9),
    # the layers they were made for
    ((0, 40, 3, 32, 36, 36, 9, 4, 1), 8.5, 23.1), ((1, 40, 3, 32, 36, 36, 9, 4, 0), 11.4, 25.9),
    ((2, 40, 3, 32, 36, 36, 9, 4, 1), 17.8, 33.0), ((0, 40, 32, 3, 36, 36, 9, 4, 1), 11.7, 27.7),
    ((1, 40, 32, 3, 36, 36, 9, 4, 0), 8.2, 21.4), ((2, 40, 32, 3, 36, 36, 9, 4, 1), 20.8, 51.0),
    ((0, 128, 3, 64, 64, 64, 3, 1, 0), 30, 44), ((3, 128, 3, 64, 64, 64, 3, 1, 0), 51, 82),
    ((2, 128, 3, 64, 64, 64, 3, 1, 0), 76, 153), ((0, 2233, 335, 3, 5, 5, 7, 3, 0), 190, 1180),
    ((0, 40, 3, 138, 10, 71, 3, 1, 1), 8.8, 18.0), ((3, 40, 3, 64, 36, 36, 3, 1, 0), 9.8, 13.3),
]


@pytest.mark.parametrize("shape,here,other", FEW, ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else "")
def test_few_channel_convs_take_the_faster_form(shape, here, other):
    op, B, cin, cout, H, W, K, p, bias = shape
    got = hip_abi.load().xdna_conv2d_few_pick(op, B, cin, cout, H, W, K, K, p, p, bias)
    assert (got > 0) == (here < other)


# op (0 / 1 stride-1 / stride-2 forward against the packed-rows kernels, 5 / 6 with the pack against the one that
# reads NCHW in place), B, Cin, Cout, H, W: us of the real-pixel kernel, us of the other
PX = [
    ((6, 19, 32, 16, 26, 26), 11.4, 6.9), ((6, 14, 64, 128, 4, 4), 9.0, 6.5), ((6, 1, 16, 512, 28, 28), 10.8, 6.7),
    ((6, 6, 512, 64, 16, 16), 14.3, 10.8), ((6, 572, 128, 16, 3, 3), 16.2, 9.2), ((6, 68, 128, 64, 2, 2), 12.6, 10.7),
    ((1, 1, 9, 128, 37, 5), 10.2, 8.6), ((1, 3, 7, 256, 24, 24), 11.0, 9.5),
    ((6, 40, 64, 128, 18, 18), None, None), ((1, 128, 64, 128, 64, 64), 57, 72), ((1, 40, 32, 64, 36, 36), None, None),
    ((5, 6, 512, 5, 6, 6), 13.0, 8.5), ((5, 82, 256, 32, 16, 16), 28.7, 20.9), ((5, 1909, 256, 64, 2, 2), 30.6, 20.7),
    ((5, 1, 256, 128, 35, 35), 14.2, 11.2), ((5, 4, 512, 64, 10, 7), 13.1, 8.9), ((0, 26, 512, 23, 3, 3), 9.1, 8.1),
    ((5, 40, 256, 256, 9, 9), 16.1, 19.3), ((5, 40, 512, 256, 4, 4), 16.8, 23.1), ((0, 40, 256, 256, 9, 9), 12.5, 13.4),
    ((0, 40, 512, 256, 4, 4), 11.4, 16.8), ((0, 40, 128, 128, 9, 9), 10.1, 7.0),
]


@pytest.mark.parametrize("shape,here,other", PX, ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else "")
def test_conv3x3_forwards_take_the_faster_form(shape, here, other):
    want = 1 if here is None or here < other else 0
    assert hip_abi.load().xdna_conv3x3_px_pick(*shape, 1) == want


def test_grids_past_the_launch_limit_stay_off_the_few_channel_kernels():
    """A workgroup per image of 256 threads: 2^24 of them are more threads than a launch takes."""
    lib = hip_abi.load()
    pick = lambda op, *a: lib.xdna_conv2d_few_pick(op, *a, 3, 3, 1, 1, 1)  # noqa: E731
    assert pick(0, 1 << 24, 8, 3, 1, 4) == 0 and pick(0, 1 << 24, 3, 8, 1, 4) == 0 and pick(1, 1 << 24, 3, 8, 1, 4) == 0
    assert lib.xdna_conv1x1_pick(0, 1 << 24, 8, 8, 1, 4, 1) == 0


def test_stride2_layers_within_the_offset_limits_take_the_real_pixel_kernels():
    """The weight gradient's limits are those of x's and of the half-resolution dY's packed rows; past
    them (2 GB) the layer takes the stride-1 form."""
    pick = hip_abi.load().xdna_conv3x3_px_pick
    assert pick(4, 128, 128, 512, 128, 128, 1) == 1 and pick(2, 128, 512, 128, 128, 128, 1) == 1
    assert pick(4, 128, 1024, 64, 128, 128, 1) == 0  # x's rows 4.4 GB
    assert pick(4, 500, 64, 512, 128, 128, 1) == 0   # dY's 2.3 GB
    assert pick(3, 500, 64, 64, 128, 128, 1) == 0    # pixels: more than a plan holds
