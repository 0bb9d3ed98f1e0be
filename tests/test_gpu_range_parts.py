"""quantize_per_tensor_dynamic where the range reaches the host in parts: sizes around a block, a round of blocks and both
ends of the range, extremes at either end, NaNs and infinities, threads, against the CPU op."""
import threading

import pytest
import torch

from gpu_util import say

import torch_musa_amd  # noqa: F401

pytestmark = pytest.mark.gpu

SIZES = [65536, 65537, 65539, 81920, 98304, 98305, 98306, 98307, 98308, 128 * 1024, 262144 - 1, 262144, 262144 + 5, 262144 + 4096 * 4 + 3, 1 << 20, (1 << 21) - 3, 1 << 21, (1 << 21) + 1]


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("dtype", [torch.quint8, torch.qint8])
def test_sizes_and_places(n, dtype):
    say("range parts", n, dtype)
    x = torch.randn(n, generator=torch.Generator().manual_seed(n))
    for at in (0, 1, n // 2, n - 4, n - 3, n - 2, n - 1):
        y = x.clone()
        y[at] = 37.5
        y[(at + n // 3) % n] = -21.25
        want = torch.quantize_per_tensor_dynamic(y, dtype, False)
        got = torch.quantize_per_tensor_dynamic(y.cuda(), dtype, False)
        assert got.q_scale() == want.q_scale() and got.q_zero_point() == want.q_zero_point(), at
        assert torch.equal(got.int_repr().cpu(), want.int_repr()), at


@pytest.mark.parametrize("n", [98308, 300001])
def test_nan_and_no_number(n):
    say("range parts, NaN", n)
    x = torch.randn(n)
    x[::7] = float("nan")
    x[5], x[n - 2] = 9.0, -4.0
    q = torch.quantize_per_tensor_dynamic(x.cuda(), torch.quint8, False)
    clean = torch.where(torch.isnan(x), torch.zeros(()), x)
    want = torch.quantize_per_tensor_dynamic(clean, torch.quint8, False)
    assert q.q_scale() == want.q_scale() and q.q_zero_point() == want.q_zero_point()
    with pytest.raises(RuntimeError, match="min should be less than or equal to max"):
        torch.quantize_per_tensor_dynamic(torch.full((n,), float("nan"), device="cuda"), torch.quint8, False)
    q = torch.quantize_per_tensor_dynamic(clean.cuda(), torch.quint8, False)   # the slot serves the next call
    assert q.q_scale() == want.q_scale()


def test_threads_and_streams():
    say("range parts, threads")
    xs = [torch.randn(131072 + 64 * i, generator=torch.Generator().manual_seed(i)) * (i + 1) for i in range(6)]
    want = [torch.quantize_per_tensor_dynamic(x, torch.quint8, False) for x in xs]
    bad = []

    def work(i):
        x = xs[i].cuda()
        torch.cuda.synchronize()
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(40):
                q = torch.quantize_per_tensor_dynamic(x, torch.quint8, False)
                if q.q_scale() != want[i].q_scale() or q.q_zero_point() != want[i].q_zero_point():
                    bad.append(i)
            torch.cuda.current_stream().synchronize()
            if not torch.equal(q.int_repr().cpu(), want[i].int_repr()):
                bad.append(-i)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(6)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad, bad
