"""quantized::linear and linear_dynamic on feature counts and pointers off the 16-byte grid, against PyTorch's CPU
operators: the streaming kernel on unaligned rows, the copy onto the grid, the one-launch dynamic kernels."""
import pytest
import torch
import torch_musa_amd  # noqa: F401

pytestmark = pytest.mark.gpu
OPS = torch.ops.quantized

SHAPES = [(1, 16, 5), (1, 17, 3), (16, 31, 16), (2, 63, 17), (7, 65, 33), (16, 1000, 40), (3, 4100, 64), (5, 8191, 20),
          (1, 1, 4), (16, 15, 9), (17, 7, 5), (17, 17, 18), (33, 100, 64), (64, 129, 63), (65, 1000, 130),
          (130, 2051, 100), (517, 1000, 2051), (70, 8200, 96), (300, 72, 1000)]


def _weight(n, k, per_channel, gen):
    w = torch.randn(n, k, generator=gen) * 0.02
    if per_channel:
        return torch.quantize_per_channel(w, w.abs().amax(1).double().clamp_min(1e-6) / 127,
                                          torch.zeros(n, dtype=torch.long), 0, torch.qint8)
    return torch.quantize_per_tensor(w, float(w.abs().max()) / 127, 0, torch.qint8)


@pytest.mark.parametrize("m,k,n", SHAPES)
@pytest.mark.parametrize("per_channel", [True, False])
def test_static(m, k, n, per_channel):
    gen = torch.Generator().manual_seed(m * 7919 + k * 31 + n)
    w, b = _weight(n, k, per_channel, gen), torch.randn(n, generator=gen)
    x = torch.quantize_per_tensor(torch.randn(m, k, generator=gen), 0.03, 121, torch.quint8)
    scale = 0.03 * max(k, 4) ** 0.5
    op = OPS.linear_relu if m % 2 else OPS.linear
    want = op(x, OPS.linear_prepack(w, b), scale, 99).int_repr()
    packed = OPS.linear_prepack(w.cuda(), b.cuda())
    print("[case]", m, k, n, per_channel, flush=True)
    got = op(x.cuda(), packed, scale, 99).int_repr().cpu()
    assert torch.equal(got, want)
    # the same rows one byte into their storage
    codes = torch.empty(m * k + 1, dtype=torch.uint8, device="cuda")[1:].view(m, k).copy_(x.int_repr().cuda())
    view = torch._make_per_tensor_quantized_tensor(codes, 0.03, 121)
    assert torch.equal(op(view, packed, scale, 99).int_repr().cpu(), want)


@pytest.mark.parametrize("m,k,n", SHAPES + [(16, 1022, 33), (16, 2047, 20), (4, 8190, 33), (1, 16383, 17)])
def test_dynamic(m, k, n):
    gen = torch.Generator().manual_seed(m * 104729 + k * 17 + n)
    w, b = _weight(n, k, m % 3 == 0, gen), torch.randn(n, generator=gen)
    x = torch.randn(m, k, generator=gen) + 0.5
    want = OPS.linear_dynamic(x, OPS.linear_prepack(w, b), False)
    print("[case]", m, k, n, flush=True)
    packed = OPS.linear_prepack(w.cuda(), b.cuda())
    got = OPS.linear_dynamic(x.cuda(), packed, False).cpu()
    assert torch.allclose(got, want, rtol=1e-5, atol=1e-5 * float(want.abs().max()) + 1e-7)
    view = torch.empty(m * k + 1, device="cuda")[1:].view(m, k).copy_(x.cuda())
    assert torch.equal(OPS.linear_dynamic(view, packed, False).cpu(), got)


@pytest.mark.parametrize("m,k,n", [(1, 64, 5), (7, 100, 33), (100, 320, 18), (300, 1024, 257), (64, 4096, 96),
                                   (512, 64, 4099), (2600, 320, 1920)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_plain_tensor_linear_in_16_bits(m, k, n, dtype):
    """The 16-bit outputs are the fp32 output rounded once."""
    gen = torch.Generator().manual_seed(m + k + n)
    x = torch.randint(0, 256, (m, k), dtype=torch.uint8, generator=gen).cuda()
    w = torch.randint(-127, 128, (k, n), dtype=torch.int8, generator=gen).cuda()
    ws, wz = (torch.rand(n, generator=gen) * 1e-3).cuda(), torch.zeros(n, dtype=torch.long).cuda()
    call = lambda out: OPS.linear_per_tensor(x, 0.02, 120, w, ws, wz, None, 1.0, 0, out, "relu", [], "")  # noqa: E731
    assert torch.equal(call(dtype), call(torch.float32).to(dtype))


@pytest.mark.parametrize("m,k,n", [
    # an odd or short run of stages shared by two wave groups: 20, 21 (the last one 16 bytes), 33, 103 stages
    (64, 1280, 64), (130, 1296, 100), (517, 2064, 70), (266, 6592, 130),
    # 64 x 128 tiles with all of K in LDS: one chunk, two to four phases, edges of tiles
    (129, 16, 10000), (1030, 272, 1001), (384, 768, 3072), (500, 784, 3000), (65, 1024, 16100),
    # rows read where they lie: the last chunk 1 ... 15 bytes, one stage, one and two wave groups, edges of tiles
    (17, 17, 65), (129, 65, 1), (65, 127, 64), (400, 1279, 66), (64, 1281, 65), (70, 2049, 129), (300, 8191, 67)])
@pytest.mark.parametrize("relu", [False, True])
def test_tiles_of_64_rows(m, k, n, relu):
    """Exact integer sums and the requantisation of the CPU operator: the same bytes."""
    gen = torch.Generator().manual_seed(m * 7919 + k * 31 + n)
    w, b = _weight(n, k, n % 2 == 0, gen), torch.randn(n, generator=gen)
    x = torch.quantize_per_tensor(torch.randn(m, k, generator=gen), 0.03, 121, torch.quint8)
    scale = 0.03 * max(k, 4) ** 0.5
    op = OPS.linear_relu if relu else OPS.linear
    want = op(x, OPS.linear_prepack(w, b), scale, 99).int_repr()
    packed = OPS.linear_prepack(w.cuda(), b.cuda())
    print("[case]", m, k, n, relu, flush=True)
    for at in (0, 1, 8):  # the rows at this byte of their storage
        codes = torch.empty(m * k + at, dtype=torch.uint8, device="cuda")[at:].view(m, k).copy_(x.int_repr().cuda())
        view = torch._make_per_tensor_quantized_tensor(codes, 0.03, 121)
        assert torch.equal(op(view, packed, scale, 99).int_repr().cpu(), want)
