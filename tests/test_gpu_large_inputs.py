"""Inputs past the lines that a size draws: the same bytes as the same input in smaller pieces (whose results the other
tests compare with the oracle).  Pointwise convolutions over more than 2 GiB and 4 GiB; the quantizer on either side of
the codes that it still writes with ordinary stores."""
import numpy as np
import pytest
import torch

from gpu_util import dev, say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch,channels,residual", [
    (33, 256, False),    # 2 214 592 512 bytes, four k-steps
    (65, 256, False),    # 4 362 076 160 bytes
    (129, 64, True),     # 2 164 260 864 bytes, one k-step and a residual
])
def test_pointwise_beyond_32_bits(batch, channels, residual):
    from torch_musa_amd import cabi
    say("pointwise", batch, channels, residual)
    h = w = 512
    oc = 16
    rng = np.random.default_rng(batch)
    wq = rng.integers(-127, 128, (oc, 1, 1, channels), dtype=np.int8)
    pw = cabi.PackedConv2d(dev(wq), cabi.conv_geom((1, h, w, channels), wq.shape, (1, 1), (0, 0), (1, 1), 1))
    ws = dev((0.001 + 0.002 * rng.random(oc)).astype(np.float32))
    gen = torch.Generator("cuda").manual_seed(batch)
    x = torch.randint(0, 256, (batch, h, w, channels), dtype=torch.uint8, device="cuda", generator=gen)
    accum = torch.randint(0, 256, (batch, h, w, oc), dtype=torch.uint8, device="cuda", generator=gen) if residual else None
    out_scale = float(np.float32(3 * 74.0 * 74.0 * 0.03 * 0.002 * np.sqrt(channels) / 128))

    def run(lo, hi):
        g = cabi.conv_geom((hi - lo, h, w, channels), wq.shape, (1, 1), (0, 0), (1, 1), 1)
        if residual:
            return cabi.conv2d_fused(x[lo:hi], pw, g, 0.03, 60, ws, None, out_scale, 128, accum=accum[lo:hi],
                                     accum_scale=0.35, accum_zp=110, activation="relu")
        return cabi.conv2d(x[lo:hi], pw, g, 0.03, 60, ws, None, out_scale, 128)

    whole = run(0, batch)
    torch.cuda.synchronize()
    step = (2**31 - 1) // (h * w * channels)
    for lo in range(0, batch, step):
        hi = min(lo + step, batch)
        assert torch.equal(whole[lo:hi], run(lo, hi)), (lo, hi)
    assert whole[0].unique().numel() > 100


@pytest.mark.parametrize("n", [2**28, 2**28 + 4, 2**28 + 1031])
@pytest.mark.parametrize("dtype", [torch.quint8, torch.qint8])
def test_quantize_around_a_cache_of_codes(n, dtype):
    say("quantize", n, dtype)
    gen = torch.Generator("cuda").manual_seed(n % 9973)
    x = torch.randn(n, device="cuda", generator=gen)
    whole = torch.quantize_per_tensor(x, 0.03, 5, dtype).int_repr()
    cut = 2**27 + 12  # off the blocks' grid
    assert torch.equal(whole[:cut], torch.quantize_per_tensor(x[:cut], 0.03, 5, dtype).int_repr())
    assert torch.equal(whole[cut:], torch.quantize_per_tensor(x[cut:], 0.03, 5, dtype).int_repr())
