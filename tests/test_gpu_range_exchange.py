"""Dynamic quantization in the launch whose blocks exchange their ranges: around every step of what a thread holds, rows and
dense, blocks that find the missing ranges themselves, streams at once, a captured stream; against the oracle."""
import threading

import numpy as np
import pytest
import torch

import oracle
from gpu_util import dev, host, say

from torch_musa_amd import cabi

pytestmark = pytest.mark.gpu

BLOCK = 512 * 4        # values a block reads at a time
CHIP = 256 * BLOCK     # ... and all of them


def check(x, pitch, q, qp, signed, reduce_range, fused):
    mn, mx = oracle.minmax(x.ravel(), nthreads=8)
    scale, zp = oracle.choose_qparams(mn, mx, signed, reduce_range)
    assert cabi.read_qparams(qp) == (scale, zp)
    want = (oracle.quantize_per_tensor_fused if fused else oracle.quantize_per_tensor)(x.ravel(), scale, zp, signed, nthreads=8)
    np.testing.assert_array_equal(host(q)[:, :x.shape[1]], want.reshape(x.shape))


def values(m, k, seed, low, high):
    x = (np.random.default_rng(seed).standard_normal((m, k)) * 2.5 + 0.4).astype(np.float32)
    x.ravel()[low], x.ravel()[high] = -31.5, 23.25
    return x


@pytest.mark.parametrize("n", [4, 7, BLOCK - 1, BLOCK, BLOCK + 3, CHIP - 1, CHIP, CHIP + 1, 2 * CHIP + 5, 3 * CHIP + BLOCK + 2,
                               6 * CHIP + 1, 8 * CHIP + 4, 13 * CHIP + 3, 16 * CHIP, 16 * CHIP + 7, 24 * CHIP + 1, 32 * CHIP - 2,
                               32 * CHIP + 1, 49 * CHIP + 6])
@pytest.mark.parametrize("signed,fused", [(False, True), (False, False), (True, False)])
def test_dense(n, signed, fused):
    say("exchange dense", n, signed, fused)
    for low, high in [(0, n - 1), (n - 2, n // 2)]:
        x = values(1, n, n, low, high)
        q, qp = cabi.quantize_dynamic_exchange(dev(x), n, signed, n % 2 == 1, fused)
        check(x, n, q, qp, signed, n % 2 == 1, fused)


@pytest.mark.parametrize("m,k", [(1, 4), (3, 5), (64, 513), (2000, 17), (257, 1001), (266, 6578), (3906, 550), (2100, 4090), (4100, 4099)])
def test_rows(m, k):
    say("exchange rows", m, k)
    pitch = (k + 15) // 16 * 16
    x = values(m, k, m * k, m * k - 1, k - 1)
    q, qp = cabi.quantize_dynamic_exchange(dev(x), pitch, False, False, True)
    check(x, pitch, q, qp, False, False, True)


@pytest.mark.parametrize("m,k,pitch", [(1, 5 * CHIP + 3, 0), (1, BLOCK * 40, 0), (700, 1003, 1008)])
@pytest.mark.parametrize("blocks", [1, 3, 64, 65, 256])
def test_blocks_that_do_not_wait(m, k, pitch, blocks):
    # no poll: whatever a block does not see at once it finds itself, as it does behind blocks that cannot run yet
    say("exchange, no polls", m, k, blocks)
    x = values(m, k, k, 0, m * k - 1)
    q, qp = cabi.quantize_dynamic_exchange(dev(x), pitch or k, False, False, True, blocks=blocks, polls=0)
    check(x, pitch or k, q, qp, False, False, True)


def test_no_numbers_and_infinities():
    say("exchange, NaN and infinity")
    x = values(1, 200001, 1, 17, 150000)
    x[0, ::7] = np.nan
    q, qp = cabi.quantize_dynamic_exchange(dev(x), 200001, False, False, False)
    assert cabi.read_qparams(qp) == oracle.choose_qparams(*(float(v) for v in (np.nanmin(x), np.nanmax(x))), False, False)
    clean = np.nan_to_num(x, nan=0.0)
    want = oracle.quantize_per_tensor(clean.ravel(), *cabi.read_qparams(qp), False)
    numbers = ~np.isnan(x.ravel())
    np.testing.assert_array_equal(host(q).ravel()[numbers], want[numbers])
    # all of both, and an infinity: as the launches that do not exchange ranges have it (a captured stream takes those)
    for bad in (np.full((1, 70000), np.nan, np.float32), np.where(np.arange(70000) == 69999, np.inf, 1.0).astype(np.float32)[None]):
        xd = dev(bad)
        q, qp = cabi.quantize_dynamic_exchange(xd, 70000, False, False, True)
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            q2, qp2 = cabi.quantize_per_tensor_dynamic_dev(xd, False, False, fused=True)
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(qp.cpu(), qp2.cpu()) and torch.equal(q.cpu(), q2.cpu())


def test_streams_at_once():
    say("exchange, streams")
    sizes = [40000, 300000, CHIP * 3 + 1, CHIP * 9]
    xs = [dev(values(1, n, n, 5, n - 5)) for n in sizes]
    torch.cuda.synchronize()
    want = [cabi.quantize_dynamic_exchange(x, x.shape[1], False, False, True) for x in xs]
    torch.cuda.synchronize()
    bad = []

    def work(i):
        x = xs[i]
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(30):
                q, qp = cabi.quantize_dynamic_exchange(x, x.shape[1], False, False, True)
            torch.cuda.current_stream().synchronize()
        if not (torch.equal(q, want[i][0]) and torch.equal(qp, want[i][1])):
            bad.append(i)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(xs))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad, bad


def test_captured_stream_takes_launches_without_exchange():
    say("exchange, captured")
    x = dev(values(1, 400000, 3, 9, 11))
    with pytest.raises(RuntimeError, match="tmq_quantize_dynamic_exchange"):
        with torch.cuda.graph(torch.cuda.CUDAGraph()):
            cabi.quantize_dynamic_exchange(x, 400000, False, False, True)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        q, qp = cabi.quantize_per_tensor_dynamic_dev(x, False, False)
    for scale in (1.0, 2.0, 0.5):
        x.mul_(scale)
        g.replay()
        torch.cuda.synchronize()
        q2, qp2 = cabi.quantize_per_tensor_dynamic_dev(x, False, False)
        assert torch.equal(q, q2) and torch.equal(qp, qp2)
