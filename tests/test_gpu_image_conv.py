"""Convolutions over images of three channels against the oracle: operand alignments (odd and even strides), groups
of four pixels over the image's edges and the tensor's ends, channel tails, one and several k-steps, tiles in columns."""
import numpy as np
import pytest
import torch

import oracle
from gpu_util import say
from test_gpu_conv import _check, _conv_case, _run, cabi  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("spec", [
    # batch, height, width, channels in, out, kernel, stride, padding, dilation, groups
    (1, 2, 2, 3, 5, 2, 1, 0, 1, 1),       # twelve bytes in all, one k-step
    (1, 3, 3, 3, 1, 3, 1, 1, 1, 1),
    (3, 5, 7, 3, 17, 3, 1, 1, 1, 1),      # odd stride, width of no group, a few channels
    (2, 9, 13, 3, 24, 3, 2, 0, 1, 1),     # the last group of a row reaches into the next
    (2, 11, 6, 3, 48, 4, 3, 2, 1, 1),     # odd stride beyond one
    (2, 20, 33, 3, 64, 5, 2, 2, 1, 1),    # two k-steps and a half
    (1, 31, 30, 3, 70, 7, 2, 3, 1, 1),    # four k-steps, a second channel block of six
    (1, 17, 19, 3, 130, 8, 1, 3, 1, 1),   # eight taps: a run of exactly 32 bytes
    (1, 6, 900, 3, 32, 3, 1, 1, 1, 1),    # rows split into columns
    (1, 40, 4, 3, 16, 7, 1, 6, 1, 1),     # more padding than image
    (40, 33, 35, 3, 96, 3, 2, 1, 1, 1),   # several tiles per block
])
@pytest.mark.parametrize("x_signed", [False, True])
def test_image_conv(cabi, spec, x_signed):  # noqa: F811
    say("image conv", spec, x_signed)
    c = _conv_case(*spec, seed=sum(spec), x_signed=x_signed, relu=not x_signed)
    y, acc, _ = _run(cabi, c)
    args = (c["stride"], c["padding"], c["dilation"], c["groups"])
    np.testing.assert_array_equal(acc, oracle.conv2d_acc32(c["xq"], c["wq"], *args, c["x_zp"], nthreads=8))
    want = oracle.conv2d(c["xq"], c["x_scale"], c["x_zp"], c["wq"], c["w_scales"], c["bias"], *args, c["out_scale"],
                         c["out_zp"], relu=c["relu"], nthreads=8)
    _check(y, want, "image conv")


@pytest.mark.parametrize("size", [(1, 3, 5), (1, 4, 4), (2, 1, 17), (3, 7, 11), (2, 64, 48), (1, 3, 4099)])
@pytest.mark.parametrize("at", [0, 1])
def test_planes_to_pixels(cabi, size, at):
    b, h, w = size
    x = torch.randint(0, 256, (b * 3 * h * w + at,), dtype=torch.uint8).cuda()[at:].view(b, 3, h, w)
    print("[case]", size, at, flush=True)
    y = torch.full((b, h, w, 3), 77, dtype=torch.uint8, device="cuda")
    rc = cabi.lib().tmq_planes_to_pixels(x.data_ptr(), y.data_ptr(), b, h * w, cabi.stream_ptr())
    assert rc == (0 if h * w >= 16 else 2)  # fewer than 16 pixels are refused
    assert torch.equal(y, x.permute(0, 2, 3, 1)) if rc == 0 else bool((y == 77).all())


def test_image_in_nchw_memory_gives_the_same_bytes(cabi):
    x = torch.quantize_per_tensor(torch.randn(2, 3, 33, 29).cuda(), 0.03, 128, torch.quint8)
    w = torch.quantize_per_tensor(torch.randn(24, 3, 3, 3).cuda(), 0.02, 0, torch.qint8)
    packed = torch.ops.quantized.conv2d_prepack(w, None, [2, 2], [1, 1], [1, 1], 1)
    y = torch.ops.quantized.conv2d(x, packed, 0.1, 100)
    z = torch.ops.quantized.conv2d(x.contiguous(memory_format=torch.channels_last), packed, 0.1, 100)
    assert torch.equal(y.int_repr(), z.int_repr())
