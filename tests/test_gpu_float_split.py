"""16-bit float outputs of products that are split along K: the partial sums stay 32-bit words, and the results are the fp32 ones
rounded once, as every other kernel writes them."""
import ctypes as C

import pytest
import torch

from gpu_util import say
from torch_musa_amd import cabi

pytestmark = pytest.mark.gpu

KINDS = {torch.float32: 0, torch.bfloat16: 1, torch.float16: 2}


def _product(x, pw, scales, bias, pitch, dtype, config):
    m = x.shape[0]
    room = torch.empty(max(cabi.lib().tmq_linear_workspace_bytes(m, pw.N, pw.K), 16), dtype=torch.uint8, device="cuda").fill_(0x55)
    y = torch.full((m, pitch), 77.0, dtype=dtype, device="cuda")
    d = cabi._linear_desc(x, pw, 0.02, 131, scales, bias, 1.0, 0, False, False, None)
    d.workspace, d.workspace_bytes, d.kernel = room.data_ptr(), room.numel(), config + 1
    cabi.check(cabi.lib().tmq_linear_float(C.byref(d), None, C.c_void_p(y.data_ptr()), C.c_int64(pitch), KINDS[dtype],
                                           C.c_void_p(cabi.stream_ptr())), "tmq_linear_float")
    return y


@pytest.mark.parametrize("m,n,k", [(26, 7, 12704), (65, 130, 8208), (128, 4200, 8240), (300, 300, 8192), (1193, 5, 12960)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_split(m, n, k, dtype):
    say("16-bit split", m, n, k, dtype)
    g = torch.Generator(device="cuda").manual_seed(m + n)
    x = torch.randint(0, 256, (m, k), generator=g, device="cuda").to(torch.uint8)
    pw = cabi.PackedLinear(torch.randint(-127, 128, (n, k), generator=g, device="cuda").to(torch.int8))
    scales = torch.rand(n, generator=g, device="cuda") * 1e-3 + 1e-4
    bias = torch.randn(n, generator=g, device="cuda")
    exact = _product(x, pw, scales, bias, n, torch.float32, 2)              # (not split)
    for config in (13, -1):
        for pitch in (n, n + 3):
            y = _product(x, pw, scales, bias, pitch, dtype, config)
            assert torch.equal(y[:, :n], exact.to(dtype)), (config, pitch)
            assert bool((y[:, n:] == 77).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_operator(dtype):
    m, k, n = 128, 8240, 4200
    assert cabi.linear_kernel_choice(m, n, k, out="f32", workspace=True)["kernel"] - 1 == 13
    say("16-bit split, operator", dtype)
    gen = torch.Generator().manual_seed(3)
    x = torch.randint(0, 256, (m, k), dtype=torch.uint8, generator=gen).cuda()
    w = torch.randint(-127, 128, (k, n), dtype=torch.int8, generator=gen).cuda()
    ws, wz = (torch.rand(n, generator=gen) * 1e-4).cuda(), torch.zeros(n, dtype=torch.long).cuda()
    call = lambda out: torch.ops.quantized.linear_per_tensor(x, 0.02, 120, w, ws, wz, None, 1.0, 0, out, "none", [], "")  # noqa: E731
    assert torch.equal(call(dtype), call(torch.float32).to(dtype))
