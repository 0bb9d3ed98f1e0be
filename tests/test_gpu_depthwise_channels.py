"""Depthwise convolutions over channel counts off the dword grid, against PyTorch's CPU operators: the last four channels
of a pixel overlap the four before them."""
import pytest
import torch
import torch_musa_amd  # noqa: F401

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
