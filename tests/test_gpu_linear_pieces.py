"""quantized::linear on tiles of 32 rows whose waves walk their shares of a long K in pieces: piece and tile edges against the
oracle, and the automatic choice on either side of its lines against the plain kernel."""
import numpy as np
import pytest
import torch

import oracle
from gpu_util import dev, host, say
from test_gpu_linear import _check, _run, _tile_case, cabi  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cfg", [29, 30])   # 32 x 32 and 32 x 64 tiles, pieces of 256 and 128 bytes
# one chunk; waves without work; the eight waves' first pieces, one more; an odd last piece; the ends of the range it is taken for
@pytest.mark.parametrize("k", [16, 112, 128, 144, 1024, 1040, 2048, 2064, 4112, 4480, 12288])
@pytest.mark.parametrize("m,n", [(1, 1), (31, 33), (33, 31), (64, 64), (70, 129)])
def test_piece_and_tile_edges(cabi, cfg, k, m, n):  # noqa: F811
    say("linear pieces", cfg, m, n, k)
    c = _tile_case(m, n, k, seed=m + n + k + cfg, x_signed=bool(k & 16), relu=bool(m & 2), bias=m != 33, per_channel=n != 64)
    y, acc, pw = _run(cabi, c, cfg)
    np.testing.assert_array_equal(acc, oracle.linear_acc32(c["xq"], c["wq"], nthreads=8))
    _check(y, oracle.linear(c["xq"], c["x_scale"], c["x_zp"], c["wq"], c["w_scales"], c["bias"], c["out_scale"], c["out_zp"],
                            relu=c["relu"], nthreads=8), "pieces")
    cabi.force_linear_config(cfg)
    try:
        f = host(cabi.linear_f32(dev(c["xq"]), pw, c["x_scale"], c["x_zp"], dev(c["w_scales"].astype(np.float32)),
                                 None if c["bias"] is None else dev(c["bias"])))
    finally:
        cabi.force_linear_config(-1)
    sums = acc.astype(np.int64) - c["x_zp"] * c["wq"].astype(np.int64).sum(1)
    bias = 0.0 if c["bias"] is None else c["bias"]
    exact = sums * (np.float32(c["x_scale"]) * c["w_scales"].astype(np.float32)).astype(np.float64) + bias
    # one rounding of the integer sum to 24 bits and one of the fused multiply-add
    bound = 2.0 ** -23 * (np.abs(exact - bias) + np.abs(exact)) + 1e-30
    assert np.all(np.abs(f - exact) <= bound)


@pytest.mark.parametrize("m,n,k", [
    (48, 320, 4112), (49, 320, 4112), (49, 320, 4096), (64, 4096, 4400), (64, 4128, 4400),        # few rows
    (256, 1024, 4112), (257, 1024, 4112), (2048, 128, 12288), (300, 700, 12304),                  # 256 tiles of 32 x 32, the end of K
    (512, 1024, 5120), (513, 1024, 5120), (288, 1800, 6400), (288, 1800, 7168),                   # 256 of 32 x 64
    (100, 3740, 8960), (100, 3750, 8960), (100, 2270, 9216), (100, 2280, 9216),                   # 32 and 20 Mi weights
    (32, 320, 7680), (33, 320, 7680), (33, 320, 7664),                                            # more than 32 rows
    # off the 16-byte grid: the copy comes first where the padded shape is one of these
    (49, 33, 4097), (840, 192, 8155), (513, 70, 4111), (300, 500, 12287), (300, 500, 12290),
    # ... or 64 x 128 tiles in a ring
    (700, 1500, 2303), (700, 1500, 2305), (500, 3900, 4100),
    # tiles dealt to the XCDs in runs, on either side of 900 KB of weights, of all row tiles' remainders
    (129, 3040, 656), (129, 3072, 656), (64, 1360, 672), (64, 1376, 672), (33, 1376, 672), (300, 950, 1024),
    (70, 5184, 1280), (65, 950, 1040), (129, 1100, 2064), (1129, 448, 3072), (40, 4200, 4096)])
@pytest.mark.parametrize("x_signed", [False, True])
def test_the_choice(cabi, m, n, k, x_signed):  # noqa: F811
    say("linear pieces, the choice", m, n, k, x_signed)
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    lo, hi, dt = (-128, 128, torch.int8) if x_signed else (0, 256, torch.uint8)
    pitch = k + (16 if m % 2 else 0)          # rows of a wider tensor as well
    x = torch.randint(lo, hi, (m, pitch), generator=g, device="cuda").to(dt)[:, :k]
    w = torch.randint(-127, 128, (n, k), generator=g, device="cuda").to(torch.int8)
    ws = torch.rand(n, generator=g, device="cuda") * 1e-3 + 1e-4
    bias = torch.randn(n, generator=g, device="cuda")
    pw = cabi.PackedLinear(w)
    outs = []
    scratch = cabi.lib().tmq_linear_scratch_bytes(m, n, k, int(k % 16 == 0))
    for cfg, room in ((9, 0), (-1, 0), (-1, scratch)):
        cabi.force_linear_config(cfg)
        work = torch.full((room,), 0xab, dtype=torch.uint8, device="cuda") if room else None
        cabi.linear_workspace, cabi.use_linear_workspace = work, room > 0
        try:
            outs.append((cabi.linear(x, pw, 0.05, 3, ws, bias, 0.4, 10), cabi.linear_f32(x, pw, 0.05, 3, ws, bias)))
        finally:
            cabi.force_linear_config(-1)
            cabi.linear_workspace, cabi.use_linear_workspace = None, True
        if room and k % 16:                    # the rows were copied onto the grid first
            pitch = (k + 15) // 16 * 16
            assert torch.equal(work[:m * pitch].view(dt).view(m, pitch)[:, :k], x)
    for bytes_, floats in outs[1:]:
        assert torch.equal(bytes_, outs[0][0])
        assert torch.equal(floats, outs[0][1])
