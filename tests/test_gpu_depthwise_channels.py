"""Depthwise convolutions over channel counts off the dword grid, against PyTorch's CPU operators: the last four channels
of a pixel overlap the four before them."""
import numpy as np
import pytest
import torch
import torch_musa_amd  # noqa: F401

import oracle
from gpu_util import dev, host, say
from test_gpu_conv import LSB_TOL, _conv_case, cabi  # noqa: F401

pytestmark = pytest.mark.gpu
OPS = torch.ops.quantized


@pytest.mark.parametrize("channels", [17, 18, 31, 270, 1030])
@pytest.mark.parametrize("kernel,stride,dilation", [(3, 1, 1), (3, 2, 1), (5, 1, 1), (7, 2, 1), (2, 1, 2)])
def test_off_the_dword_grid(channels, kernel, stride, dilation):
    """Exact integer sums and the requantisation of the CPU operator: the same bytes."""
    gen = torch.Generator().manual_seed(channels * 64 + kernel * 8 + stride)
    w = torch.randn(channels, 1, kernel, kernel, generator=gen) / kernel
    qw = torch.quantize_per_channel(w, w.abs().flatten(1).amax(1).double() / 127, torch.zeros(channels, dtype=torch.long),
                                    0, torch.qint8)
    bias = torch.randn(channels, generator=gen) * 0.1
    x = torch.randn(2, channels, 13, 19, generator=gen).contiguous(memory_format=torch.channels_last)
    qx = torch.quantize_per_tensor(x, 0.03, 119, torch.quint8)
    args = ([stride] * 2, [kernel // 2] * 2, [dilation] * 2, channels)
    want = OPS.conv2d_relu(qx, OPS.conv2d_prepack(qw, bias, *args), 0.04, 3)
    print("[case]", channels, kernel, stride, flush=True)
    packed = OPS.conv2d_prepack(qw.cuda(), bias.cuda(), *args)
    got = OPS.conv2d_relu(qx.cuda(), packed, 0.04, 3)
    assert torch.equal(got.int_repr().cpu(), want.int_repr())


def _at(a, offset):
    """A device copy of `a` that begins `offset` elements into its storage."""
    t = dev(a)
    return torch.empty(t.numel() + offset, dtype=t.dtype, device="cuda")[offset:].view(t.shape).copy_(t)


@pytest.mark.parametrize("channels,kernel,stride,dilation", [
    (17, 3, 1, 1), (18, 3, 2, 1), (31, 5, 1, 1), (270, 3, 1, 1), (1030, 3, 2, 1), (22, 7, 1, 1), (19, 2, 1, 2),
])
@pytest.mark.parametrize("x_signed", [False, True])
@pytest.mark.parametrize("offset", [0, 1])
def test_off_the_dword_grid_sums_residual_and_silu(cabi, channels, kernel, stride, dilation, x_signed, offset):  # noqa: F811
    """The kernel's other outputs at such counts: int32 sums, a residual and SiLU, with the input, the residual and the
    output at addresses of no grid, against the oracle."""
    say("depthwise", channels, kernel, stride, dilation, x_signed, offset)
    c = _conv_case(2, 13, 11, channels, channels, kernel, stride, kernel // 2, dilation, channels,
                   seed=channels + kernel, x_signed=x_signed)
    args = (c["stride"], c["padding"], c["dilation"], c["groups"])
    g = cabi.conv_geom(c["xq"].shape, c["wq"].shape, *args)
    pw = cabi.PackedConv2d(dev(c["wq"]), g)
    ws, bias, x = dev(c["w_scales"].astype(np.float32)), dev(c["bias"]), _at(c["xq"], offset)
    cabi.force_conv_path(7)
    try:
        sums = host(cabi.conv2d_acc32(x, pw, g, c["x_zp"]))
        np.testing.assert_array_equal(sums, oracle.conv2d_acc32(c["xq"], c["wq"], *args, c["x_zp"], nthreads=8))
        rng = np.random.default_rng(channels)
        for activation, residual, signed in (("none", True, True), ("relu", True, False), ("silu", False, True),
                                             ("silu", True, False)):
            lo, hi = (-128, 128) if signed else (0, 256)
            dt = np.int8 if signed else np.uint8
            acc = rng.integers(lo, hi, sums.shape, dtype=dt) if residual else None
            zp, acc_zp = (-20, -7) if signed else (30, 110)
            want = oracle.conv2d_fused(c["xq"], c["x_scale"], c["x_zp"], c["wq"], c["w_scales"], c["bias"], *args,
                                       c["out_scale"], zp, accum=acc, accum_scale=0.35, accum_zp=acc_zp,
                                       activation=activation, out_signed=signed, nthreads=8)
            out = _at(np.zeros(sums.shape, dt), offset)
            got = host(cabi.conv2d_fused(x, pw, g, c["x_scale"], c["x_zp"], ws, bias, c["out_scale"], zp,
                                         accum=None if acc is None else _at(acc, offset), accum_scale=0.35,
                                         accum_zp=acc_zp, activation=activation, out_signed=signed, out=out))
            d = np.abs(got.astype(np.int32) - want.astype(np.int32))
            if activation == "silu":   # expf on the device and on the host may differ in the last bit
                assert d.max() <= LSB_TOL and np.count_nonzero(d) <= max(2, 0.001 * d.size), (d.max(), np.count_nonzero(d))
            else:
                assert d.max() == 0, (activation, np.count_nonzero(d), d.max())
    finally:
        cabi.force_conv_path(-1)
