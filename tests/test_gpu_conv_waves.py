"""quantized::conv2d on one round of tiles of 32 pixels whose waves walk K in pieces: the automatic choice at the edges of tiles,
pieces and of the sizes it is taken for, windows over every border, against the direct kernel and the implicit GEMM."""
import pytest
import torch

from gpu_util import say
from torch_musa_amd import cabi


def _operands(b, h, w, ic, oc, k, signed, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    lo, hi, dt = (-128, 128, torch.int8) if signed else (0, 256, torch.uint8)
    x = torch.randint(lo, hi, (b, h, w, ic), generator=g, device="cuda").to(dt)
    wq = torch.randint(-127, 128, (oc, k, k, ic), generator=g, device="cuda").to(torch.int8)
    scales = torch.rand(oc, generator=g, device="cuda") * 1e-3 + 1e-4
    return x, wq, scales, torch.randn(oc, generator=g, device="cuda"), g, (lo, hi, dt)


def _on(path, call):
    cabi.force_conv_path(path)
    try:
        return call()
    finally:
        cabi.force_conv_path(-1)


@pytest.mark.gpu
@pytest.mark.parametrize("b,h,w,ic,oc,k,stride,pad,dil", [
    (1, 5, 6, 64, 31, 3, 1, 1, 1), (1, 4, 8, 64, 33, 3, 1, 1, 1), (3, 7, 5, 80, 65, 3, 2, 1, 1),      # a tile and its edges
    (2, 9, 9, 112, 48, 3, 1, 0, 1), (1, 12, 12, 128, 40, 3, 1, 2, 2), (2, 11, 13, 64, 20, 3, 3, 2, 1),  # no pad, dilation, wide pad
    (1, 6, 7, 1024, 24, 1, 2, 0, 1), (1, 9, 10, 48, 50, 5, 1, 2, 1), (1, 9, 7, 32, 36, 7, 2, 3, 1),     # other kernels, up to 49 taps
    (1, 7, 7, 512, 72, 3, 1, 1, 1), (1, 8, 8, 464, 16, 3, 1, 1, 1),                                   # waves with three and four pieces
    (1, 32, 32, 64, 256, 3, 1, 1, 1), (1, 32, 33, 64, 256, 3, 1, 1, 1),                               # 256 tiles of 32 channels and more
    (1, 64, 32, 80, 256, 3, 1, 1, 1), (1, 64, 33, 80, 256, 3, 1, 1, 1), (2, 10, 10, 40, 24, 3, 1, 1, 1)])  # ... of 64; padded channels
@pytest.mark.parametrize("signed", [False, True])
def test_automatic_choice(b, h, w, ic, oc, k, stride, pad, dil, signed):
    say("conv waves", b, h, w, ic, oc, k, stride, pad, dil, signed)
    x, wq, scales, bias, g, (lo, hi, dt) = _operands(b, h, w, ic, oc, k, signed, b + h + w + ic + oc)
    geom = cabi.conv_geom(x.shape, (oc, k, k), (stride, stride), (pad, pad), (dil, dil), 1)
    pw = cabi.PackedConv2d(wq, geom)
    scale = 0.4 * (ic * k * k / 1000) ** 0.5
    plain = lambda relu: cabi.conv2d(x, pw, geom, 0.05, 3, scales, bias, scale, 10, relu=relu)  # noqa: E731
    for relu in (False, True):
        assert torch.equal(plain(relu), _on(3, lambda: plain(relu)))
    # the same epilogue behind the implicit GEMM: the same bytes
    rest = torch.randint(lo, hi, tuple(cabi.conv_out_hw(geom)) + (oc,), generator=g, device="cuda").to(dt)
    rest = rest.unsqueeze(0).repeat(b, 1, 1, 1)
    for kw in (dict(activation="silu"), dict(accum=rest, accum_scale=0.1, accum_zp=4, activation="relu"),
               dict(accum=rest, accum_scale=0.1, accum_zp=4, activation="silu")):
        fused = lambda: cabi.conv2d_fused(x, pw, geom, 0.05, 3, scales, bias, scale, 10, **kw)  # noqa: B023,E731
        assert torch.equal(fused(), _on(2 if ic % 16 == 0 else 8, fused)), kw


def test_scratch():
    ask = lambda *s: cabi.lib().tmq_conv2d_scratch_bytes(cabi.conv_geom(s[:4], s[4:7], (1, 1), (1, 1), (1, 1), 1))  # noqa: E731
    assert ask(1, 7, 7, 512, 512, 3, 3) == 0
    assert ask(1, 7, 7, 512, 8250, 3, 3) == 49 * 4608          # more than a round: patch rows
    assert ask(2, 20, 20, 40, 40, 3, 3) == 2 * 400 * 48        # padded channels
