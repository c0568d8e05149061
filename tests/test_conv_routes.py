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
