"""1x1 convolutions (stride 1 and 2, no padding: ResNet's downsampling shortcut) on the
HIP GEMM path through aten.convolution(_backward): forward, input, weight and bias
gradients against the float64 oracle (oracle.conv2d_*, pinned by brute force and
PyTorch's CPU conv in tests/test_oracle_conv2d.py), with the conv bar (2 bf16 ulp with the
ulp(max|ref| 2^-8) floor, relative L2 <= 1e-2), on odd sizes and at BASELINE config 5's
full shapes.  Path counters prove the HIP path ran (no MIOpen)."""
import numpy as np
import pytest
import torch

import oracle
import xdna_train
from gpu_util import check_bf16

pytestmark = pytest.mark.gpu
X = torch.device("xdna")


def bits(t):
    return t.detach().cpu().contiguous().view(torch.int16).numpy().view(np.uint16)


@pytest.mark.parametrize("B,Ci,Co,H,W,s,bias", [
    (4, 64, 128, 16, 16, 2, False),
    (3, 32, 48, 9, 7, 2, True),      # odd planes: ceil(H/2) outputs
    (2, 128, 64, 8, 8, 1, True),
    (5, 24, 40, 5, 11, 1, False),
    (128, 64, 128, 64, 64, 2, False),   # config 5 shortcuts
    (128, 128, 256, 32, 32, 2, False),
    (128, 256, 512, 16, 16, 2, False),
])
def test_conv1x1_matches_oracle(B, Ci, Co, H, W, s, bias):
    print(f"conv1x1 B{B} {Ci}->{Co} {H}x{W} s{s} bias={bias}", flush=True)
    g = torch.Generator().manual_seed(B * 7 + Ci + s)
    x = torch.randn(B, Ci, H, W, generator=g).bfloat16()
    w = (torch.randn(Co, Ci, 1, 1, generator=g) / Ci ** 0.5).bfloat16()
    b = (torch.randn(Co, generator=g) * 0.1).bfloat16() if bias else None
    Ho, Wo = (H - 1) // s + 1, (W - 1) // s + 1
    dy = torch.randn(B, Co, Ho, Wo, generator=g).bfloat16()
    xd = x.to(X).requires_grad_()
    wd = w.to(X).requires_grad_()
    bd = b.to(X).requires_grad_() if bias else None
    xdna_train.reset_mapped_cpu_stats()
    y = torch.nn.functional.conv2d(xd, wd, bd, stride=s)
    y.backward(dy.to(X))
    st = xdna_train.mapped_cpu_stats()
    for k in ("hip_conv1x1.fwd.run", "hip_conv1x1.bwd.run"):
        assert st.get(k, {}).get("calls", 0) == 1, (k, st)
    assert not any(k.startswith("aten::convolution") for k in st), st
    xb, wb, dyb = bits(x), bits(w), bits(dy)
    bb = bits(b) if bias else None
    check_bf16(bits(y), oracle.conv2d_fwd(xb, wb, bb, stride=(s, s)), what="1x1 fwd")
    check_bf16(bits(xd.grad), oracle.conv2d_dgrad(dyb, wb, (H, W), stride=(s, s)), what="1x1 dgrad")
    gw, gb = oracle.conv2d_wgrad(xb, dyb, (1, 1), stride=(s, s))
    check_bf16(bits(wd.grad), gw, what="1x1 wgrad")
    if bias:
        check_bf16(bits(bd.grad), gb, what="1x1 bias grad")


# The kernels that sample and spread in place: both output-channel widths (up to 64, more), the
# step of 64 channels and pixels and its remainders, rows of 8-pixel pieces, rows that a piece
# crosses once and twice, odd planes, whose last even row has none below, single pixels, operands
# 2 bytes off a 4-byte address, a bias, and one split or several of the weight gradient.
@pytest.mark.parametrize("B,Ci,Co,H,W,s,off", [
    (2, 64, 128, 16, 32, 2, 0),
    (3, 65, 64, 13, 34, 2, 1),
    (2, 130, 129, 17, 19, 2, 0),
    (5, 7, 9, 7, 7, 2, 1),
    (2, 3, 70, 5, 3, 2, 0),
    (4, 9, 5, 1, 1, 2, 0),
    (1, 64, 64, 2, 260, 2, 0),
    (3, 64, 200, 8, 8, 1, 0),
    (2, 100, 33, 9, 15, 1, 1),
    (1, 1, 1, 1, 3, 1, 0),
    (40, 63, 65, 11, 12, 2, 1),
])
def test_conv1x1_in_place_kernels(B, Ci, Co, H, W, s, off):
    from xdna_train import hip_abi
    import ctypes

    print(f"conv1x1 direct B{B} {Ci}->{Co} {H}x{W} s{s} off {off}", flush=True)
    lib = hip_abi.load()
    g = torch.Generator().manual_seed(B * 31 + Ci + H)
    Ho, Wo = (H + s - 1) // s, (W + s - 1) // s

    def dev(t):  # `off` elements into a buffer of its own
        buf = torch.zeros(t.numel() + off + 8, dtype=t.dtype, device="cuda")
        buf[off:off + t.numel()] = t.reshape(-1).cuda()
        return buf[off:off + t.numel()].view(t.shape)

    x = dev(torch.randn(B, Ci, H, W, generator=g).bfloat16())
    w = dev((torch.randn(Co, Ci, 1, 1, generator=g) / Ci ** 0.5).bfloat16())
    b = dev((torch.randn(Co, generator=g) * 0.1).bfloat16())
    dy = dev(torch.randn(B, Co, Ho, Wo, generator=g).bfloat16())
    y, dx, gw = dev(torch.full((B, Co, Ho, Wo), 7.0).bfloat16()), dev(torch.full((B, Ci, H, W), 7.0).bfloat16()), dev(
        torch.full((Co, Ci, 1, 1), 7.0).bfloat16())
    ws = torch.empty(lib.xdna_conv1x1_wgrad_workspace_bytes(B, Ci, Co, H, W, s), dtype=torch.uint8, device="cuda")
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    assert lib.xdna_conv1x1_fwd_bf16(p(x), p(w), p(b), p(y), B, Ci, Co, H, W, s, st) == 0
    assert lib.xdna_conv1x1_dgrad_bf16(p(dy), p(w), p(dx), B, Ci, Co, H, W, s, st) == 0
    assert lib.xdna_conv1x1_wgrad_bf16(p(x), p(dy), p(gw), B, Ci, Co, H, W, s, p(ws), ws.numel(), st) == 0
    assert lib.xdna_conv1x1_wgrad_bf16(p(x), p(dy), p(gw), B, Ci, Co, H, W, s, p(ws), ws.numel() - 1, st) != 0
    torch.cuda.synchronize()
    check_bf16(bits(y), oracle.conv2d_fwd(bits(x), bits(w), bits(b), stride=(s, s)), what="1x1 fwd")
    check_bf16(bits(dx), oracle.conv2d_dgrad(bits(dy), bits(w), (H, W), stride=(s, s)), what="1x1 dgrad")
    check_bf16(bits(gw), oracle.conv2d_wgrad(bits(x), bits(dy), (1, 1), stride=(s, s))[0], what="1x1 wgrad")
