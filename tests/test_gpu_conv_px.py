"""The 3x3 convs over real output pixels (xdna_conv3x3_px_*): stride 1 and 2, forward, input
gradient and weight gradient, against the float64 oracle to the conv bar, at the edges of
their tiles and lattices; every tile and split of K, both row layouts, bit equality of
repeated calls, and the choice through aten."""
import numpy as np
import pytest
import torch

import oracle
import xdna_train
from gpu_util import check_bf16, dev, dev_zeros, host, ptr, stream

pytestmark = pytest.mark.gpu

# B, Cin, Cout, H, W: one pixel, odd and even sizes (parities without pixels), one and two
# strips, partial channel chunks and tiles, more pixel tiles than one, a channel count that
# splits K
SHAPES = [(1, 1, 1, 1, 1), (2, 5, 7, 2, 3), (3, 70, 130, 13, 11), (2, 64, 64, 9, 40), (5, 33, 20, 16, 16),
          (1, 300, 66, 5, 4), (2, 130, 260, 7, 73)]


def _ids(s):
    return "x".join(map(str, s))


def _data(shape, stride):
    B, cin, cout, H, W = shape
    rng = np.random.default_rng(sum(shape) + stride)
    bound = np.sqrt(6.0 / (9 * cin))
    x = oracle.rng_bf16(rng, (B, cin, H, W))
    w = oracle.bf16_bits(rng.uniform(-bound, bound, (cout, cin, 3, 3)).astype(np.float32))
    b = oracle.bf16_bits(rng.uniform(-0.1, 0.1, (cout,)).astype(np.float32))
    dy = oracle.rng_bf16(rng, (B, cout, (H - 1) // stride + 1, (W - 1) // stride + 1))
    return x, w, b, dy


def _pack(hip, bits, layout):
    B, C, H, W = bits.shape
    buf = dev(np.full((hip.xdna_conv3x3_layout_packed_bytes(B, C, H, W, layout) // 2,), 0xBEEF, np.uint16))
    assert hip.xdna_conv3x3_layout_pack_bf16(ptr(dev(bits)), ptr(buf), B, C, H, W, layout, stream()) == 0
    return buf


def _prepared(hip, w, dgrad):
    cout, cin = w.shape[:2]
    a, b = (cout, cin) if dgrad else (cin, cout)
    wt = dev_zeros((hip.xdna_conv3x3_prepared_weight_bytes(a, b) // 2,))
    assert hip.xdna_conv3x3_prepare_weights_bf16(ptr(dev(w)), ptr(wt), cout, cin, int(dgrad), stream()) == 0
    return wt


# (tiles 5 and 6: the stride-2 input gradient in column pairs)
@pytest.mark.parametrize("stride,tile", [(s, t) for s in (1, 2) for t in range(5 if s == 1 else 7)])
@pytest.mark.parametrize("layout", [0, 1])
@pytest.mark.parametrize("shape", SHAPES, ids=_ids)
def test_forward_and_input_gradient(hip, shape, stride, layout, tile):
    B, cin, cout, H, W = shape
    print(f"conv px {shape} stride {stride} layout {layout} tile {tile}", flush=True)
    x, w, b, dy = _data(shape, stride)
    y = dev(np.full(dy.shape, 0x7F7F, np.uint16))
    xp = _pack(hip, x, layout)
    for act in (0, 1):
        assert hip.xdna_conv3x3_px_bf16(stride - 1, ptr(xp), ptr(_prepared(hip, w, False)), ptr(dev(b)), ptr(y), B, cin,
                                        cout, H, W, layout, act, min(tile, 4), stream()) == 0
        ref = oracle.conv2d_fwd(x, w, b, (stride, stride), (1, 1))
        check_bf16(host(y), np.maximum(ref, 0) if act else ref, what=f"fwd {shape}")
    dx = dev(np.full(x.shape, 0x7F7F, np.uint16))
    assert hip.xdna_conv3x3_px_bf16(0 if stride == 1 else 2, ptr(_pack(hip, dy, layout)), ptr(_prepared(hip, w, True)),
                                    None, ptr(dx), B, cout, cin, H, W, layout, 0, tile, stream()) == 0
    check_bf16(host(dx), oracle.conv2d_dgrad(dy, w, (H, W), (stride, stride), (1, 1)), what=f"dgrad {shape}")


@pytest.mark.parametrize("splits", [0, 1, 5, 8, 64])
@pytest.mark.parametrize("layout", [0, 1])
@pytest.mark.parametrize("stride", [1, 2])
@pytest.mark.parametrize("shape", SHAPES, ids=_ids)
def test_weight_gradient(hip, shape, stride, layout, splits):
    B, cin, cout, H, W = shape
    print(f"conv px wgrad {shape} stride {stride} layout {layout} splits {splits}", flush=True)
    x, _, _, dy = _data(shape, stride)
    xp, dp = _pack(hip, x, layout), _pack(hip, dy, layout)
    assert hip.xdna_conv3x3_set_wgrad_splits(splits) == 0
    try:
        n = hip.xdna_conv3x3_px_wgrad_workspace_bytes(stride - 1, B, cin, cout, H, W)
        ws = dev(np.full((n // 2,), 0x7FC0, np.uint16))  # NaN: every partial that is read was written
        out = []
        for with_bias in (True, False):
            gw, gb = dev_zeros((cout, cin, 3, 3)), dev_zeros((cout,))
            assert hip.xdna_conv3x3_px_wgrad_bf16(stride - 1, ptr(xp), ptr(dp), ptr(gw), ptr(gb) if with_bias else None,
                                                  B, cin, cout, H, W, layout, ptr(ws), n, stream()) == 0
            out.append((host(gw), host(gb)))
        assert hip.xdna_conv3x3_px_wgrad_bf16(stride - 1, ptr(xp), ptr(dp), ptr(gw), None, B, cin, cout, H, W, layout,
                                              ptr(ws), n - 1, stream()) == -1
    finally:
        assert hip.xdna_conv3x3_set_wgrad_splits(0) == 0
    ref_w, ref_b = oracle.conv2d_wgrad(x, dy, (3, 3), (stride, stride), (1, 1))
    check_bf16(out[0][0], ref_w, what=f"wgrad {shape}")
    check_bf16(out[0][1], ref_b, what=f"bias grad {shape}")
    np.testing.assert_array_equal(out[1][0], out[0][0])


def test_pick(hip):
    """The choice: stride-2 convs and small layers' weight gradients take these kernels, large
    stride-1 grids the window kernels; forcing one of those turns it off; operands past 32-bit
    offsets are refused."""
    pick = hip.xdna_conv3x3_px_pick
    assert [pick(op, 128, 64, 128, 64, 64, 1) for op in (1, 2, 4)] == [1, 1, 1]
    assert pick(0, 40, 256, 256, 9, 9, 1) == 1 and pick(0, 40, 128, 128, 9, 9, 1) == 0
    assert pick(0, 64, 512, 512, 72, 72, 1) == 0 and pick(3, 64, 512, 512, 72, 72, 1) == 0
    assert pick(3, 40, 128, 128, 9, 9, 1) == 1
    assert pick(1, 4096, 512, 64, 64, 64, 1) == 0  # more than 2 GiB of packed rows
    assert hip.xdna_conv3x3_px_bf16(1, 1, 1, None, 1, 4096, 512, 64, 64, 64, 1, 0, 0, stream()) == -1
    assert pick(3, 160, 64, 64, 64, 64, 1) == 1 and pick(3, 64, 64, 512, 64, 64, 1) == 0
    assert pick(3, 1024, 512, 512, 8, 8, 1) == 1 and pick(3, 64, 512, 512, 36, 36, 1) == 0
    # the weight gradient: more pixels than its splits hold
    assert pick(4, 40, 16, 16, 512, 512, 1) == 1 and pick(4, 41, 16, 16, 512, 512, 1) == 0
    ws = hip.xdna_conv3x3_px_wgrad_workspace_bytes
    assert ws(0, 40, 64, 64, 256, 256) > 0 and ws(0, 64, 64, 64, 256, 256) == 0
    assert hip.xdna_conv3x3_px_wgrad_bf16(0, 1, 1, 1, None, 64, 64, 64, 256, 256, 1, 1, 1 << 40, stream()) == -1
    assert hip.xdna_conv3x3_set_rows_variant(9) == 0
    assert pick(1, 128, 64, 128, 64, 64, 1) == 0
    assert hip.xdna_conv3x3_set_rows_variant(0) == 0


def test_stride2_weight_gradient_near_the_offset_limit(hip):
    """A layer whose output gradient packs to 0.6 GB as it is and to 2.4 GB spread onto the stride-1 grid: the
    real-pixel kernels take it, and their offsets hold (first and last channels against float64)."""
    B, cin, cout, H, W = 128, 128, 512, 128, 128
    assert [hip.xdna_conv3x3_px_pick(op, B, *((cout, cin) if op == 2 else (cin, cout)), H, W, 1) for op in (1, 2, 4)] == [1] * 3
    print("conv px wgrad 128 -> 512 on 128 x 128 x 128", flush=True)
    g = torch.Generator(device="cuda").manual_seed(5)
    x = torch.randn(B, cin, H, W, generator=g, device="cuda").bfloat16()
    dy = torch.randn(B, cout, H // 2, W // 2, generator=g, device="cuda").bfloat16()

    def pack(t):
        b, c, h, w = t.shape
        buf = torch.empty(hip.xdna_conv3x3_layout_packed_bytes(b, c, h, w, 1) // 2, dtype=torch.int16, device="cuda")
        assert hip.xdna_conv3x3_layout_pack_bf16(t.data_ptr(), buf.data_ptr(), b, c, h, w, 1, stream()) == 0
        return buf

    xp, dp = pack(x), pack(dy)
    n = hip.xdna_conv3x3_px_wgrad_workspace_bytes(1, B, cin, cout, H, W)
    ws = torch.empty(n, dtype=torch.uint8, device="cuda")
    gw = torch.empty(cout, cin, 3, 3, dtype=torch.bfloat16, device="cuda")
    assert hip.xdna_conv3x3_px_wgrad_bf16(1, xp.data_ptr(), dp.data_ptr(), gw.data_ptr(), None, B, cin, cout, H, W, 1,
                                          ws.data_ptr(), n, stream()) == 0
    some = [0, 1, 255, 256, 510, 511]
    ref = torch.zeros(len(some), cin, 3, 3, dtype=torch.float64, device="cuda")
    for b in range(0, B, 16):
        xd = torch.nn.functional.pad(x[b:b + 16].double(), [1] * 4)
        d = dy[b:b + 16, some].double().flatten(2)
        for i in range(3):
            for j in range(3):
                t = xd[:, :, i:i + H:2, j:j + W:2].flatten(2).transpose(1, 2).contiguous()
                ref[:, :, i, j] += torch.matmul(d, t).sum(0)
    got = gw[some].double()
    # one bf16 rounding beside fp32 sums of 524288 products
    assert float((got - ref).norm() / ref.norm()) < 4e-3


@pytest.mark.parametrize("need_dx", [True, False])
@pytest.mark.parametrize("trainable", [True, False])
def test_aten_stride2(trainable, need_dx):
    """Every combination of gradients a stride-2 layer is asked for, against the oracle."""
    torch.manual_seed(3)
    conv = torch.nn.Conv2d(20, 40, 3, stride=2, padding=1).bfloat16().to("xdna").requires_grad_(trainable)
    x = torch.randn(3, 20, 15, 38).bfloat16()
    dy = torch.randn(3, 40, 8, 19).bfloat16()
    xd = x.to("xdna").requires_grad_(need_dx)
    y = conv(xd)
    bits = lambda t: t.detach().cpu().contiguous().view(torch.int16).numpy().view(np.uint16)  # noqa: E731
    xb, wb, bb, db = bits(x), bits(conv.weight), bits(conv.bias), bits(dy)
    check_bf16(bits(y), oracle.conv2d_fwd(xb, wb, bb, (2, 2), (1, 1)), what="fwd")
    if not (trainable or need_dx):
        return
    y.backward(dy.to("xdna"))
    xdna_train.synchronize()
    if need_dx:
        check_bf16(bits(xd.grad), oracle.conv2d_dgrad(db, wb, (15, 38), (2, 2), (1, 1)), what="dgrad")
    if trainable:
        gw, gb = oracle.conv2d_wgrad(xb, db, (3, 3), (2, 2), (1, 1))
        check_bf16(bits(conv.weight.grad), gw, what="wgrad")
        check_bf16(bits(conv.bias.grad), gb, what="bias grad")
