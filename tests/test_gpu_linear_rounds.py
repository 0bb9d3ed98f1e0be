"""quantized::linear on tiles copied straight into LDS: K around the copies' rings of three and six stages, tile edges, rounds
beyond one; and the automatic choice by rounds against the plain kernel."""
import numpy as np
import pytest
import torch

import oracle
from gpu_util import dev, host, say
from test_gpu_linear import _check, _run, _tile_case, cabi  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cfg", [1, 2])   # 128 x 128 and 64 x 64 tiles
@pytest.mark.parametrize("k", [112, 128, 144, 192, 208, 320, 336, 400, 1040])
@pytest.mark.parametrize("m,n", [(1, 1), (63, 65), (65, 64), (129, 130), (64 * 17, 64 * 16)])
def test_ring_and_tile_edges(cabi, cfg, k, m, n):  # noqa: F811
    say("linear copies", cfg, m, n, k)
    c = _tile_case(m, n, k, seed=m + n + k + cfg, x_signed=bool(k & 16), relu=bool(m & 2))
    y, acc, pw = _run(cabi, c, cfg)
    np.testing.assert_array_equal(acc, oracle.linear_acc32(c["xq"], c["wq"]))
    _check(y, oracle.linear(c["xq"], c["x_scale"], c["x_zp"], c["wq"], c["w_scales"], c["bias"], c["out_scale"], c["out_zp"],
                            relu=c["relu"]), "copies")
    cabi.force_linear_config(cfg)
    try:
        f = host(cabi.linear_f32(dev(c["xq"]), pw, c["x_scale"], c["x_zp"], dev(c["w_scales"].astype(np.float32)),
                                 dev(c["bias"])))
    finally:
        cabi.force_linear_config(-1)
    sums = acc.astype(np.int64) - c["x_zp"] * c["wq"].astype(np.int64).sum(1)
    exact = sums * (np.float32(c["x_scale"]) * c["w_scales"].astype(np.float32)).astype(np.float64) + c["bias"]
    # one rounding of the integer sum to 24 bits and one of the fused multiply-add
    bound = 2.0 ** -23 * (np.abs(exact - c["bias"]) + np.abs(exact)) + 1e-30
    assert np.all(np.abs(f - exact) <= bound)


@pytest.mark.parametrize("m,n,k", [(757, 3456, 64), (1690, 2616, 112), (941, 5056, 192), (603, 2304, 768), (642, 2304, 1920),
                                   (2417, 832, 1344), (843, 1088, 2688), (2496, 820, 1456), (19800, 320, 640),
                                   (3430, 1728, 656)])
@pytest.mark.parametrize("x_signed", [False, True])
def test_choice_by_rounds(cabi, m, n, k, x_signed):  # noqa: F811
    say("linear by rounds", m, n, k, x_signed)
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    lo, hi, dt = (-128, 128, torch.int8) if x_signed else (0, 256, torch.uint8)
    x = torch.randint(lo, hi, (m, k), generator=g, device="cuda").to(dt)
    w = torch.randint(-127, 128, (n, k), generator=g, device="cuda").to(torch.int8)
    ws = torch.rand(n, generator=g, device="cuda") * 1e-3 + 1e-4
    bias = torch.randn(n, generator=g, device="cuda")
    pw = cabi.PackedLinear(w)
    outs = []
    for cfg in (-1, 9):
        cabi.force_linear_config(cfg)
        try:
            outs.append((cabi.linear(x, pw, 0.05, 3, ws, bias, 0.4, 10), cabi.linear_f32(x, pw, 0.05, 3, ws, bias)))
        finally:
            cabi.force_linear_config(-1)
    assert torch.equal(outs[0][0], outs[1][0])
    assert torch.equal(outs[0][1], outs[1][1])
