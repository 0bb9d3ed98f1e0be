"""Max pooling over channel counts and addresses off the 16-byte grid, against the CPU oracle: the last group of 16
channels overlaps the one before it; fewer than 16 channels go one by one."""
import numpy as np
import oracle
import pytest
import torch
from gpu_util import dev, host
from torch_musa_amd import cabi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("channels", [1, 15, 16, 17, 24, 31, 33, 40])
@pytest.mark.parametrize("kernel,stride,padding", [((3, 3), (2, 2), (1, 1)), ((2, 5), (1, 2), (0, 2))])
@pytest.mark.parametrize("signed", [False, True])
def test_any_channel_count(channels, kernel, stride, padding, signed):
    rng = np.random.default_rng(channels)
    x = rng.integers(-128 if signed else 0, 128 if signed else 256, (2, 13, 18, channels)).astype(
        np.int8 if signed else np.uint8)
    want = oracle.qmaxpool2d(x, kernel, stride, padding)
    print("[case]", channels, kernel, signed, flush=True)
    args = (kernel, stride, padding, (1, 1), want.shape[1:3])
    np.testing.assert_array_equal(host(cabi.qmaxpool2d(dev(x), *args)), want)
    moved = torch.empty(x.size + 1, dtype=dev(x).dtype, device="cuda")[1:].view(x.shape).copy_(dev(x))
    np.testing.assert_array_equal(host(cabi.qmaxpool2d(moved, *args)), want)
