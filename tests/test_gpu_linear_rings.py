"""quantized::linear on 64 x 128, 128 x 64 and 128 x 128 tiles with a block per CU: rings of six stages and eight waves, K around
the rings' turns, tile edges, one round of tiles and more; and the automatic choice where it names them."""
import numpy as np
import pytest
import torch

import oracle
from gpu_util import dev, host, say
from test_gpu_linear import _check, _run, _tile_case, cabi  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cfg", [7, 22, 23])   # 128 x 128, 128 x 64, 64 x 128
# five stages and a chunk, six, an odd number, one turn of the ring and each remainder; from 1536 on a ring under 128 x 128
@pytest.mark.parametrize("k", [336, 384, 400, 448, 512, 640, 704, 1520, 1536, 1552, 1600, 1664])
@pytest.mark.parametrize("m,n", [(1, 1), (63, 129), (129, 63), (200, 260)])
def test_ring_and_tile_edges(cabi, cfg, k, m, n):  # noqa: F811
    say("linear rings", cfg, m, n, k)
    c = _tile_case(m, n, k, seed=m + n + k + cfg, x_signed=bool(k & 64), relu=bool(m & 2), per_channel=n != 63)
    y, acc, pw = _run(cabi, c, cfg)
    np.testing.assert_array_equal(acc, oracle.linear_acc32(c["xq"], c["wq"], nthreads=8))
    _check(y, oracle.linear(c["xq"], c["x_scale"], c["x_zp"], c["wq"], c["w_scales"], c["bias"], c["out_scale"], c["out_zp"],
                            relu=c["relu"], nthreads=8), "rings")
    cabi.force_linear_config(cfg)
    try:
        f = host(cabi.linear_f32(dev(c["xq"]), pw, c["x_scale"], c["x_zp"], dev(c["w_scales"].astype(np.float32)),
                                 dev(c["bias"])))
    finally:
        cabi.force_linear_config(-1)
    np.testing.assert_array_equal(f, oracle.linear_f32(c["xq"], c["x_scale"], c["x_zp"], c["wq"], c["w_scales"], c["bias"],
                                                       nthreads=8))


@pytest.mark.parametrize("m,n,k", [
    (2048, 1024, 1280), (2049, 1024, 1280), (2048, 1024, 1264), (1280, 1700, 1296),      # a round of 64 x 128 tiles, 64 x 64 in two
    (1024, 1024, 1280), (1025, 1024, 1280),                                              # ... in one
    (422, 3904, 5824), (422, 3904, 5808), (133, 4100, 4112),                             # 128 x 64
    (512, 8192, 1536), (513, 8192, 1536), (500, 8100, 1520), (254, 11264, 1552),         # 128 x 128, a round and more
    (1535, 2900, 4112), (1537, 2900, 4112), (1537, 2900, 8208), (887, 5280, 2576), (575, 8100, 4112), (577, 8100, 4112),       # ... or 128 x 256, half a round
    (900, 8100, 1088), (900, 8100, 1104)])
@pytest.mark.parametrize("x_signed", [False, True])
def test_the_choice(cabi, m, n, k, x_signed):  # noqa: F811
    say("linear rings, the choice", m, n, k, x_signed)
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    lo, hi, dt = (-128, 128, torch.int8) if x_signed else (0, 256, torch.uint8)
    x = torch.randint(lo, hi, (m, k), generator=g, device="cuda").to(dt)
    w = torch.randint(-127, 128, (n, k), generator=g, device="cuda").to(torch.int8)
    ws = torch.rand(n, generator=g, device="cuda") * 1e-3 + 1e-4
    bias = torch.randn(n, generator=g, device="cuda")
    pw = cabi.PackedLinear(w)
    outs = []
    for cfg in (9, -1):
        cabi.force_linear_config(cfg)
        try:
            outs.append((cabi.linear(x, pw, 0.05, 3, ws, bias, 0.4, 10), cabi.linear_f32(x, pw, 0.05, 3, ws, bias)))
        finally:
            cabi.force_linear_config(-1)
    assert torch.equal(outs[0][0], outs[1][0])
    assert torch.equal(outs[0][1], outs[1][1])
