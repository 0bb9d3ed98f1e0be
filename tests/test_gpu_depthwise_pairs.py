"""Depthwise quantized::conv2d, 3 x 3 at stride 1, two output columns a lane: odd and single columns, strips that end inside, channel
counts off the dword grid, every epilogue, against the direct kernel."""
import pytest
import torch

from gpu_util import say
from torch_musa_amd import cabi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("b,h,w,c,pad", [(20, 40, 41, 256, 1), (3, 33, 270, 280, 1), (172, 17, 2, 1022, 1),
                                         (3, 100, 101, 290, 2), (25, 30, 44, 273, 0), (162, 8, 8, 820, 1)])
@pytest.mark.parametrize("signed", [False, True])
def test_pairs(b, h, w, c, pad, signed):
    say("depthwise pairs", b, h, w, c, pad, signed)
    g = torch.Generator(device="cuda").manual_seed(b + h + w + c)
    lo, hi, dt = (-128, 128, torch.int8) if signed else (0, 256, torch.uint8)
    geom = cabi.conv_geom((b, h, w, c), (c, 3, 3), (1, 1), (pad, pad), (1, 1), c)
    oh, ow = cabi.conv_out_hw(geom)
    assert b * -(-oh // 8) * ow * -(-c // 4) >= 262144       # (the size from which on a lane has two columns)
    x = torch.randint(lo, hi, (b, h, w, c), generator=g, device="cuda").to(dt)
    pw = cabi.PackedConv2d(torch.randint(-127, 128, (c, 3, 3, 1), generator=g, device="cuda").to(torch.int8), geom)
    scales = torch.rand(c, generator=g, device="cuda") * 1e-3 + 1e-4
    bias = torch.randn(c, generator=g, device="cuda")
    rest = torch.randint(lo, hi, (b, oh, ow, c), generator=g, device="cuda").to(dt)
    calls = [lambda: cabi.conv2d_acc32(x, pw, geom, 3),
             lambda: cabi.conv2d(x, pw, geom, 0.05, 3, scales, bias, 0.02, 10, relu=True),
             lambda: cabi.conv2d_fused(x, pw, geom, 0.05, 3, scales, bias, 0.02, 10, accum=rest, accum_scale=0.01, accum_zp=4, activation="relu")]
    for call in calls:
        got = call()
        cabi.force_conv_path(3)
        try:
            assert torch.equal(got, call())
        finally:
            cabi.force_conv_path(-1)
