"""quantized::linear_dynamic of more than 16 rows in one launch: rows, channels and K at the edges of tiles and of the waves' shares,
blocks that wait for the others' ranges and blocks that find them themselves, against the oracle and the launches that quantize the
rows first (which exchange ranges themselves above 32768 values)."""
import ctypes as C

import numpy as np
import pytest
import torch

import oracle
from gpu_util import dev, host, say
from torch_musa_amd import cabi


def _call(x, pw, scales, bias, relu, reduce_range, polls, garbage, short=0):
    m, k = x.shape
    need = cabi.lib().tmq_linear_dynamic_tiles_workspace(m, pw.N, k)
    d = cabi.LinearDesc()
    d.M, d.N, d.K = m, pw.N, k
    d.w_packed, d.w_colsum, d.w_scales = pw.packed.data_ptr(), pw.colsum.data_ptr(), scales.data_ptr()
    d.w_per_channel, d.relu, d.bias = int(scales.numel() > 1), int(relu), None if bias is None else bias.data_ptr()
    words = torch.full((max(need, 16),), garbage, dtype=torch.uint8, device="cuda")
    d.workspace, d.workspace_bytes = words.data_ptr(), need - short
    y = torch.full((m, pw.N + 3), 77.0, device="cuda")
    status = cabi.lib().tmq_linear_dynamic_tiles(C.byref(d), x.data_ptr(), x.stride(0), int(reduce_range), y.data_ptr(), pw.N + 3, polls,
                                                 cabi.stream_ptr())
    return status, y


@pytest.mark.gpu
@pytest.mark.parametrize("m,n", [(17, 1), (32, 33), (33, 31), (64, 65), (257, 70), (96, 2700), (97, 7900), (4100, 64)])
@pytest.mark.parametrize("k", [16, 19, 100, 256, 257, 512, 515, 1024, 1026, 2047, 2048])
def test_edges(m, n, k):
    say("dynamic tiles", m, n, k)
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    wide = torch.randn(m, k + 5, generator=g, device="cuda") + 0.3
    wide[m - 1, k - 1], wide[m // 2, 0] = 9.0, -7.0          # the range sits in the last row's last value and in one tile's first
    x = wide[:, :k] if m % 2 else wide[:, :k].contiguous()   # (rows of a wider tensor as well)
    pw = cabi.PackedLinear(torch.randint(-127, 128, (n, k), generator=g, device="cuda").to(torch.int8))
    scales = torch.rand(n if n % 2 else 1, generator=g, device="cuda") * 1e-3 + 1e-4
    bias = torch.randn(n, generator=g, device="cuda") if k % 3 else None
    want = cabi.linear_dynamic(x.contiguous(), pw, scales, bias, relu=bool(m & 1), reduce_range=bool(k & 1))
    need = cabi.lib().tmq_linear_dynamic_tiles_workspace(m, n, k)
    assert (need < 0) == (n == 7900 and k > 512)             # (two blocks a CU up to there)
    for polls in (-1, 0, 1) if need >= 0 else ():
        status, y = _call(x, pw, scales, bias, m & 1, k & 1, polls, 0xff * (polls & 1))
        assert status == 0
        assert torch.equal(y[:, :n], want), polls
        assert bool((y[:, n:] == 77).all())


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(17, 33, 2048), (33, 70, 1026), (64, 65, 515), (257, 70, 1024), (97, 129, 2047), (1100, 40, 256),
                                   (4100, 64, 19), (2000, 250, 100)])
def test_against_the_oracle(m, n, k):
    say("dynamic tiles, oracle", m, n, k)
    rng = np.random.default_rng(m * n + k)
    x = rng.standard_normal((m, k)).astype(np.float32) + np.float32(0.3)
    x[m - 1, k - 1], x[m // 2, 0] = 9.0, -7.0
    w = rng.integers(-127, 128, (n, k), dtype=np.int8)
    scales = (rng.random(n) * 1e-3 + 1e-4).astype(np.float32)
    bias = rng.standard_normal(n).astype(np.float32) if k % 3 else None
    want = oracle.linear_dynamic(x, w, scales.astype(np.float64), bias, bool(m & 1), bool(k & 1))
    pw, xd, sd, bd = cabi.PackedLinear(dev(w)), dev(x), dev(scales), None if bias is None else dev(bias)
    for polls in (-1, 0):
        status, y = _call(xd, pw, sd, bd, m & 1, k & 1, polls, 0)
        assert status == 0
        np.testing.assert_array_equal(host(y)[:, :n], want)


@pytest.mark.gpu
def test_values_without_order():
    """Infinities, zeros and NaN among the rows: what the separate launches make of them."""
    g = torch.Generator(device="cuda").manual_seed(5)
    pw = cabi.PackedLinear(torch.randint(-127, 128, (40, 96), generator=g, device="cuda").to(torch.int8))
    scales = torch.rand(40, generator=g, device="cuda") * 1e-3
    for fill in (0.0, -0.0, 1e-38, 3e38, float("nan"), float("inf")):
        x = torch.randn(70, 96, generator=g, device="cuda")
        x[:] = fill if abs(fill) < 1 else x
        x[40, 3] = fill
        say("dynamic tiles, values", fill)
        status, y = _call(x, pw, scales, None, 0, 0, -1, 0)
        want = cabi.linear_dynamic(x, pw, scales, None)
        assert status == 0 and torch.equal(torch.nan_to_num(y[:, :40], 7.0), torch.nan_to_num(want, 7.0)), fill


@pytest.mark.gpu
def test_refused_and_captured():
    pw = cabi.PackedLinear(torch.ones(64, 128, dtype=torch.int8, device="cuda"))
    scales, x = torch.ones(1, device="cuda"), torch.randn(100, 128, device="cuda")
    unsupported = _call(x[:16], pw, scales, None, 0, 0, -1, 0)[0]
    assert unsupported != 0 and _call(x, pw, scales, None, 0, 0, -1, 0, short=1)[0] == unsupported
    # under capture: the launches before it, and every replay of new values
    w = torch.quantize_per_tensor(torch.randn(64, 128), 0.02, 0, torch.qint8)
    packed = torch.ops.quantized.linear_prepack(w.cuda(), torch.randn(64, device="cuda"))
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        torch.ops.quantized.linear_dynamic(x, packed, False)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        y = torch.ops.quantized.linear_dynamic(x, packed, False)
    for i in range(4):
        x.normal_(std=i + 1.0)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, torch.ops.quantized.linear_dynamic(x, packed, False))


def test_sizes():
    ask = cabi.lib().tmq_linear_dynamic_tiles_workspace
    for m, n, k, want in ((16, 64, 64, -1), (17, 64, 64, 0), (32, 8192, 64, 0), (32, 32768, 512, 0), (32, 32769, 512, -1), (32, 16384, 513, 0), (32, 16385, 513, -1), (33, 64, 15, -1),
                          (33, 64, 16, 32), (33, 64, 2048, 32), (33, 64, 2049, -1), (8192, 64, 64, 4096), (8193, 64, 64, -1), (64, 0, 64, -1)):
        assert ask(m, n, k) == want, (m, n, k)
