"""Per-channel conversions where the channels lie differently in memory (columns, whole rows, rows that no 16-byte
access divides), and the values the device reports to the host before a kernel ends, against PyTorch's CPU operators."""
import threading

import pytest
import torch
import torch_musa_amd  # noqa: F401
from torch_musa_amd import cabi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("outer,channels,inner", [
    (1, 1, 1), (5, 3, 1), (33, 4, 1), (7, 257, 1), (50, 1028, 1), (129, 1030, 1), (3, 4099, 1),   # columns
    (1, 9, 64), (2, 5, 4100), (3, 7, 516),                                                        # whole rows
    (1, 11, 27), (2, 6, 63), (1, 5, 65), (3, 3, 2049), (2, 2, 5411), (40, 50, 5), (9, 1, 12), (600, 2, 4),  # flat
    (4, 5, 2), (6, 7, 3),                                                                         # elements
])
@pytest.mark.parametrize("kind", ["qint8", "quint8", "float"])
def test_per_channel(outer, channels, inner, kind):
    torch.manual_seed(outer * 131 + channels * 7 + inner)
    dt = torch.qint8 if kind == "qint8" else torch.quint8
    lo, hi = (-128, 127) if kind == "qint8" else (0, 255)
    x = torch.randn(outer, channels, inner) * 3
    s = torch.rand(channels, dtype=torch.double) * 0.05 + 0.01
    z = torch.randint(lo, hi + 1, (channels,))
    if kind == "float":
        s, z = s.float(), z.float() + torch.rand(channels) * 0 + 0.25
        z = z.clamp(lo, hi)
    want = torch.quantize_per_channel(x, s, z, 1, dt)
    for offset in (0, 1):   # a view one element into its storage leaves the 16-byte grid
        xg = torch.empty(x.numel() + offset, device="cuda")[offset:].view(x.shape).copy_(x.cuda())
        got = torch.quantize_per_channel(xg, s.cuda(), z.cuda(), 1, dt)
        assert torch.equal(got.int_repr().cpu(), want.int_repr())
        assert torch.equal(got.dequantize().cpu(), want.dequantize())
    bad = z.clone()
    bad[channels - 1] = hi + 1
    with pytest.raises(RuntimeError, match="zero point"):
        torch.quantize_per_channel(x.cuda(), s.cuda(), bad.cuda(), 1, dt)


@pytest.mark.parametrize("n", [1, 3, 1000, 32768, 32769, 131072, (1 << 25) + 4])
def test_dynamic_range_report(n):
    x = torch.randn(n, generator=torch.Generator().manual_seed(n)) * 2
    want = torch.quantize_per_tensor_dynamic(x, torch.quint8, False)
    got = torch.quantize_per_tensor_dynamic(x.cuda(), torch.quint8, False)
    assert got.q_scale() == want.q_scale() and got.q_zero_point() == want.q_zero_point()
    assert torch.equal(got.int_repr().cpu(), want.int_repr())
    assert torch.equal(got.dequantize().cpu(), want.dequantize())
    with pytest.raises(RuntimeError, match="min should be"):
        torch.quantize_per_tensor_dynamic(torch.full((n,), float("nan"), device="cuda"), torch.quint8, False)


@pytest.mark.parametrize("n,offset", [
    (98305, 0), (1 << 21, 0),                                           # by each block of the range pass
    ((1 << 21) + 4, 0), ((1 << 21) + 7, 0), ((1 << 24) + 1, 0), (1 << 25, 0),  # by the quantizer's first block
    (98305, 1), ((1 << 21) + 6, 1),                                     # values off the 16-byte grid: by the pass between
])
@pytest.mark.parametrize("dtype", [torch.quint8, torch.qint8])
def test_dynamic_range_report_by_each_pass(n, offset, dtype):
    x = torch.randn(n, generator=torch.Generator().manual_seed(n)) * 2
    x[n - 1], x[n // 2] = 31.0, -47.0    # the range's ends: the last value and one in the middle
    xg = torch.empty(n + offset, device="cuda")[offset:].copy_(x.cuda())
    want = torch.quantize_per_tensor_dynamic(x, dtype, False)
    got = torch.quantize_per_tensor_dynamic(xg, dtype, False)
    assert got.q_scale() == want.q_scale() and got.q_zero_point() == want.q_zero_point()
    assert torch.equal(got.int_repr().cpu(), want.int_repr())
    with pytest.raises(RuntimeError, match="min should be"):
        torch.quantize_per_tensor_dynamic(xg.fill_(float("nan")), dtype, False)


@pytest.mark.parametrize("n,offset", [(1, 0), (65537, 0), (98304, 0),            # by the one launch, from 32769 on by its first block once it has
                                      (98305, 0), (200003, 0), (1 << 21, 0),     # all ranges
                                      ((1 << 21) + 1, 0), (98305, 1)])           # (off the grid: by the launch behind the range pass)
def test_range_reported_as_a_whole(n, offset):
    """The C entry point whose range comes in one piece at every size."""
    x = torch.randn(n, generator=torch.Generator().manual_seed(n)) * 2
    x[n - 1], x[n // 2] = 31.0, -47.0
    xg = torch.empty(n + offset, device="cuda")[offset:].copy_(x.cuda())
    want = torch.quantize_per_tensor_dynamic(x, torch.quint8, False)
    report = torch.zeros(2, dtype=torch.int64).pin_memory()
    for ticket in (7, 8):     # the slot is ready for the next call
        q, qp = cabi.quantize_per_tensor_dynamic_report(xg, False, False, report, ticket, 63)
        torch.cuda.synchronize()
        assert [w >> 32 for w in report.tolist()] == [ticket, ticket]
        bits = torch.tensor([w & 0xffffffff for w in report.tolist()], dtype=torch.int64).to(torch.uint32)
        assert bits.view(torch.float32).tolist() == [x.min().item(), x.max().item()]
        assert cabi.read_qparams(qp) == (want.q_scale(), want.q_zero_point())
        assert torch.equal(q.cpu(), want.int_repr())


def test_dynamic_keeps_the_memory_format():
    x = torch.randn(2, 5, 6, 7).contiguous(memory_format=torch.channels_last)
    got = torch.quantize_per_tensor_dynamic(x.cuda(), torch.qint8, True)
    want = torch.quantize_per_tensor_dynamic(x, torch.qint8, True)
    assert got.is_contiguous(memory_format=torch.channels_last) and got.q_scale() == want.q_scale()
    assert torch.equal(got.int_repr().cpu(), want.int_repr())


def test_reports_of_several_threads_and_streams():
    xs = [torch.randn(1000 + 777 * i) * (i + 1) for i in range(6)]
    wants = [torch.quantize_per_tensor_dynamic(x, torch.quint8, False).q_scale() for x in xs]
    failed = []

    def work(i):
        with torch.cuda.stream(torch.cuda.Stream()):
            x = xs[i].cuda()
            for _ in range(50):
                if torch.quantize_per_tensor_dynamic(x, torch.quint8, False).q_scale() != wants[i]:
                    failed.append(i)
            torch.cuda.current_stream().synchronize()

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(xs))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed
