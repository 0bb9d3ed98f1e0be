"""Dynamic quantization in the launches that no block waits in: what captured streams, operands off the grid and C callers with a
workspace off it take.  A workspace on the 8-byte and not the 16-byte grid pins them; against the oracle."""
import numpy as np
import pytest
import torch

import oracle
from gpu_util import dev, host, say

from torch_musa_amd import cabi

pytestmark = pytest.mark.gpu


def values(shape, seed):
    x = (np.random.default_rng(seed).standard_normal(shape) * 2.5 + 0.4).astype(np.float32)
    x.ravel()[-1], x.ravel()[x.size // 2] = 31.5, -23.25
    return x


def workspace():
    room = torch.empty(cabi.lib().tmq_minmax_workspace_bytes(0) + 8, dtype=torch.uint8, device="cuda")
    assert room.data_ptr() % 16 == 0
    return room, room.data_ptr() + 8, room.numel() - 8


def check(x, q, qp, signed, reduce_range, fused):
    scale, zp = oracle.choose_qparams(*oracle.minmax(x.ravel(), nthreads=8), signed, reduce_range)
    assert cabi.read_qparams(qp) == (scale, zp)
    want = (oracle.quantize_per_tensor_fused if fused else oracle.quantize_per_tensor)(x.ravel(), scale, zp, signed, nthreads=8)
    np.testing.assert_array_equal(host(q), want.reshape(x.shape))


# one launch whose blocks read everything; two from 98305 values on, with a tail, the last one of several turns of the grid's loop that
# ends inside a chunk; three past 2^25
@pytest.mark.parametrize("n", [32769, 98304, 98305, 98307, 200003, 1 << 20, (1 << 20) + 3, (1 << 23) + 1029, 1 << 25, (1 << 25) + 5])
@pytest.mark.parametrize("signed", [False, True])
@pytest.mark.parametrize("fused", [False, True])
def test_dense(n, signed, fused):
    say("range launches", n, signed, fused)
    x = values(n, n)
    xd, (room, ws, ws_bytes) = dev(x), workspace()
    for reduce_range in (False, True):
        q = torch.empty(n, dtype=torch.int8 if signed else torch.uint8, device="cuda")
        qp = torch.empty(16, dtype=torch.uint8, device="cuda")
        cabi.check(cabi.lib().tmq_quantize_per_tensor_dynamic_dev(xd.data_ptr(), q.data_ptr(), n, int(signed), int(reduce_range),
                                                                  int(fused), qp.data_ptr(), ws, ws_bytes, cabi.stream_ptr()), "dense")
        check(x, q, qp, signed, reduce_range, fused)
    del room


@pytest.mark.parametrize("m,k", [(30000, 3), (40000, 4), (25001, 5), (7000, 15), (130, 1003), (131, 1001), (517, 1002), (1033, 2052), (4100, 4099)])
@pytest.mark.parametrize("signed,fused", [(False, True), (False, False), (True, False), (True, True)])
def test_rows(m, k, signed, fused):
    say("range launches, rows", m, k, signed, fused)
    pitch = (k + 15) // 16 * 16
    x = values((m, k), m + k)
    xd, (room, ws, ws_bytes) = dev(x), workspace()
    q = torch.empty((m, pitch), dtype=torch.int8 if signed else torch.uint8, device="cuda")
    qp = torch.empty(16, dtype=torch.uint8, device="cuda")
    status = cabi.lib().tmq_quantize_rows_dynamic_dev(xd.data_ptr(), q.data_ptr(), m, k, pitch, int(signed), 0, int(fused),
                                                      qp.data_ptr(), ws, ws_bytes, cabi.stream_ptr())
    cabi.check(status, "rows")
    check(x, q[:, :k].contiguous(), qp, signed, False, fused)
    del room


@pytest.mark.parametrize("n", [98305, 200003, 1 << 21, (1 << 21) + 1, (1 << 25) + 5])
def test_report_by_the_range_pass(n):
    # its last block to arrive up to 2^21 values, the pass behind it beyond; twice: the slot's block count is ready again
    say("range launches, report", n)
    x = values(n, n)
    xd, (room, ws, ws_bytes) = dev(x), workspace()
    report = torch.zeros(2, dtype=torch.int64).pin_memory()
    for ticket in (7, 8):
        q, qp = torch.empty(n, dtype=torch.uint8, device="cuda"), torch.empty(16, dtype=torch.uint8, device="cuda")
        cabi.check(cabi.lib().tmq_quantize_per_tensor_dynamic_report(xd.data_ptr(), q.data_ptr(), n, 0, 0, 0, qp.data_ptr(), ws, ws_bytes,
                                                                     report.data_ptr(), ticket, 62, cabi.stream_ptr()), "report")
        torch.cuda.synchronize()
        assert [w >> 32 for w in report.tolist()] == [ticket, ticket]
        bits = torch.tensor([w & 0xffffffff for w in report.tolist()], dtype=torch.int64).to(torch.uint32)
        assert bits.view(torch.float32).tolist() == [float(x.min()), float(x.max())]
        check(x, q, qp, False, False, False)
    del room


@pytest.mark.parametrize("m,k,n", [(130, 1003, 40), (600, 515, 33), (517, 1002, 64), (100, 2053, 24)])
def test_captured_dynamic_linear_off_the_grid(m, k, n):
    say("range launches, captured", m, k, n)
    rng = np.random.default_rng(m)
    w = rng.integers(-127, 128, (n, k), dtype=np.int8)
    bias = rng.standard_normal(n).astype(np.float32)
    wq = torch._make_per_tensor_quantized_tensor(torch.from_numpy(w), 0.0123, 0)
    packed = torch.ops.quantized.linear_prepack(wq.cuda(), dev(bias))
    xd = dev(values((m, k), 1))
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.cuda.stream(stream):
        torch.ops.quantized.linear_dynamic(xd, packed, False)
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=stream):
        y = torch.ops.quantized.linear_dynamic(xd, packed, False)
    for seed in (2, 3, 4):
        x = values((m, k), seed) * np.float32(seed)
        xd.copy_(torch.from_numpy(x))
        graph.replay()
        torch.cuda.synchronize()
        np.testing.assert_array_equal(host(y), oracle.linear_dynamic(x, w, np.array([0.0123]), bias))
        assert torch.equal(y, torch.ops.quantized.linear_dynamic(xd, packed, False))
