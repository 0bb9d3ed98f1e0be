"""Float outputs of quantized::linear whose rows end anywhere: four values leave in one store at any address, and nothing between or
behind the rows is written.  Against the plain kernel, for every kernel that the sizes choose."""
import ctypes as C

import pytest
import torch

from gpu_util import say
from torch_musa_amd import cabi

pytestmark = pytest.mark.gpu


def _f32(x, pw, scales, bias, pitch, config):
    rows = x.shape[0]
    y = torch.full((rows * pitch + 8,), 77.0, device="cuda")
    cabi.force_linear_config(config)
    try:
        d = cabi._linear_desc(x, pw, 0.05, 3, scales, bias, 1.0, 0, False, False, None)
        cabi.check(cabi.lib().tmq_linear_f32(C.byref(d), None, y[3:].data_ptr(), pitch, cabi.stream_ptr()), "tmq_linear_f32")
    finally:
        cabi.force_linear_config(-1)
    return y


@pytest.mark.parametrize("m,k", [(1, 64), (16, 1040), (40, 144), (200, 256), (300, 1040), (600, 2064), (1300, 192), (1030, 4112)])
@pytest.mark.parametrize("n", [1, 3, 6, 65, 131, 1022])
@pytest.mark.parametrize("gap", [0, 5])
def test_f32_rows(m, k, n, gap):
    say("float rows", m, k, n, gap)
    g = torch.Generator(device="cuda").manual_seed(m + k + n)
    x = torch.randint(0, 256, (m, k), generator=g, device="cuda").to(torch.uint8)
    pw = cabi.PackedLinear(torch.randint(-127, 128, (n, k), generator=g, device="cuda").to(torch.int8))
    scales = torch.rand(n, generator=g, device="cuda") * 1e-3 + 1e-4
    bias = torch.randn(n, generator=g, device="cuda")
    got, want = (_f32(x, pw, scales, bias, n + gap, config) for config in (-1, 9))
    assert torch.equal(got, want)
    rows = got[3:3 + m * (n + gap)].view(m, n + gap)
    assert bool((rows[:, n:] == 77).all()) and bool((got[:3] == 77).all()) and bool((got[3 + m * (n + gap):] == 77).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("m,k,n", [(17, 64, 5), (100, 320, 131), (300, 1040, 1022), (700, 192, 3001)])
def test_16_bit_rows(m, k, n, dtype):
    say("16-bit rows", m, k, n, dtype)
    gen = torch.Generator().manual_seed(m + n)
    x = torch.randint(0, 256, (m, k), dtype=torch.uint8, generator=gen).cuda()
    w = torch.randint(-127, 128, (k, n), dtype=torch.int8, generator=gen).cuda()
    ws, wz = (torch.rand(n, generator=gen) * 1e-3).cuda(), torch.zeros(n, dtype=torch.long).cuda()
    call = lambda out: torch.ops.quantized.linear_per_tensor(x, 0.02, 120, w, ws, wz, None, 1.0, 0, out, "none", [], "")  # noqa: E731
    assert torch.equal(call(dtype), call(torch.float32).to(dtype))
