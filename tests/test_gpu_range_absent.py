"""Launches whose blocks exchange their ranges where not all of them are on the chip together, and where another launch writes the
same words: every block ends, with the same codes, parameters and products as alone."""
import ctypes as C
import threading

import pytest
import torch

from gpu_util import say

from torch_musa_amd import cabi

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def neighbour():
    """Queues a product on a stream of its own whose blocks have 64 / 128 / 224 CUs to themselves for some 160 us."""
    pw = cabi.PackedLinear(torch.randint(-127, 128, (4096, 16384), device="cuda").to(torch.int8))
    x = torch.randint(0, 255, (3584, 16384), device="cuda").to(torch.uint8)
    scale, stream = torch.ones(1, device="cuda"), torch.cuda.Stream()
    torch.cuda.synchronize()

    def busy(cus):
        with torch.cuda.stream(stream):
            cabi.force_linear_config(6)             # tiles of 256 x 256, one on a CU
            try:
                return cabi.linear(x[:cus * 16], pw, 1.0, 3, scale, None, 1e6, 0)
            finally:
                cabi.force_linear_config(-1)
    return busy


@pytest.mark.parametrize("cus", [64, 128, 224])
@pytest.mark.parametrize("m,k", [(1, 70001), (1, (1 << 23) + 7), (1, 12 << 20), (1, 1 << 24), (1, (1 << 25) + 5), (3906, 4099)])
def test_quantize_beside_a_neighbour(neighbour, cus, m, k):
    say("range beside a neighbour", cus, m, k)
    x = torch.randn(m, k, generator=torch.Generator(device="cuda").manual_seed(k), device="cuda")
    x.view(-1)[m * k - 1], x.view(-1)[m * k // 3] = 19.0, -23.0
    pitch = k if m == 1 else (k + 15) // 16 * 16
    want, params = cabi.quantize_dynamic_exchange(x, pitch, False, False, True)
    torch.cuda.synchronize()
    for polls in (32, 0):
        keep = neighbour(cus)
        q, qp = cabi.quantize_dynamic_exchange(x, pitch, False, False, True, polls=polls)
        torch.cuda.synchronize()
        assert torch.equal(qp, params) and torch.equal(q[:, :k], want[:, :k]), polls
        del keep


@pytest.mark.parametrize("cus", [64, 128, 224])
@pytest.mark.parametrize("m,n,k", [(2000, 250, 2048), (1001, 500, 1022), (2999, 180, 512)])
def test_dynamic_tiles_beside_a_neighbour(neighbour, cus, m, n, k):
    say("dynamic tiles beside a neighbour", cus, m, n, k)
    x = torch.randn(m, k, generator=torch.Generator(device="cuda").manual_seed(m), device="cuda")
    x[m - 1, k - 1], x[m // 3, 0] = 19.0, -23.0
    pw = cabi.PackedLinear(torch.randint(-127, 128, (n, k), device="cuda").to(torch.int8))
    scale, y = torch.full((1,), 1e-3, device="cuda"), torch.empty(2, m, n, device="cuda")
    need = cabi.lib().tmq_linear_dynamic_tiles_workspace(m, n, k)
    words = torch.zeros(need, dtype=torch.uint8, device="cuda")
    d = cabi.LinearDesc()
    d.M, d.N, d.K = m, n, k
    d.w_packed, d.w_colsum, d.w_scales = pw.packed.data_ptr(), pw.colsum.data_ptr(), scale.data_ptr()
    d.workspace, d.workspace_bytes = words.data_ptr(), need

    def call(out, polls):
        cabi.check(cabi.lib().tmq_linear_dynamic_tiles(C.byref(d), x.data_ptr(), k, 0, out.data_ptr(), n, polls, cabi.stream_ptr()),
                   "tmq_linear_dynamic_tiles")
    call(y[0], -1)
    torch.cuda.synchronize()
    for polls in (-1, 0):
        keep = neighbour(cus)
        call(y[1], polls)
        torch.cuda.synchronize()
        assert torch.equal(y[0], y[1]), polls
        del keep


def test_two_streams_one_workspace():
    # (what up to 98304 values long needed no workspace may still be given one that is shared)
    say("range words shared")
    sizes = [40001, 60000, 98304, 98300]
    xs = [torch.randn(n, generator=torch.Generator(device="cuda").manual_seed(n), device="cuda") * (i + 1) for i, n in enumerate(sizes)]
    want = [cabi.quantize_per_tensor_dynamic_dev(x, False, False) for x in xs]
    words = torch.zeros(cabi.lib().tmq_minmax_workspace_bytes(0), dtype=torch.uint8, device="cuda")
    got = [(torch.empty_like(q), torch.empty_like(p)) for q, p in want]
    torch.cuda.synchronize()
    bad = []

    def work(i):
        stream = torch.cuda.Stream()
        for _ in range(100):
            q, qp = got[i]
            cabi.check(cabi.lib().tmq_quantize_per_tensor_dynamic_dev(
                xs[i].data_ptr(), q.data_ptr(), sizes[i], 0, 0, 0, qp.data_ptr(), words.data_ptr(), words.numel(),
                stream.cuda_stream), "tmq_quantize_per_tensor_dynamic_dev")
        stream.synchronize()
        if not (torch.equal(got[i][0], want[i][0]) and torch.equal(got[i][1], want[i][1])):
            bad.append(sizes[i])

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(sizes))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad, bad
