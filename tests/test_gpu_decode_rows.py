"""One to five rows on the weight-streaming kernel, where a request for activations brings four k-blocks of 64 bytes for up
to four rows: k-block counts around the waves' shares (8 waves, 8 k-blocks each) and rows on and off the 16-byte grid,
against the oracle."""
import numpy as np
import pytest

import oracle
from gpu_util import dev, host, say
from test_gpu_linear import _tile_case, cabi  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("k", [16, 48, 64, 80, 512, 528, 2048, 2064, 4096, 4112, 8208, 17, 33, 75, 515, 1000, 4099])
@pytest.mark.parametrize("x_signed", [False, True])
def test_rows(cabi, m, k, x_signed):  # noqa: F811
    say("decode rows", m, k, x_signed)
    n = 50
    c = _tile_case(m, n, k, seed=m * 100000 + k, x_signed=x_signed)
    pw = cabi.PackedLinear(dev(c["wq"]))
    ws, b, x = dev(c["w_scales"].astype(np.float32)), dev(c["bias"]), dev(c["xq"])
    # (K on the 16-byte grid: pinned, others take this kernel up to 16 rows by themselves)
    cabi.force_linear_config(8 if k % 16 == 0 else -1)
    try:
        acc = oracle.linear_acc32(c["xq"], c["wq"])
        np.testing.assert_array_equal(host(cabi.linear_acc32(x, pw)), acc)
        want = oracle.linear(c["xq"], c["x_scale"], c["x_zp"], c["wq"], c["w_scales"], c["bias"], c["out_scale"], c["out_zp"])
        got = host(cabi.linear(x, pw, c["x_scale"], c["x_zp"], ws, b, c["out_scale"], c["out_zp"], out_signed=x_signed))
        np.testing.assert_array_equal(got, want)
        raw = acc.astype(np.int64) - c["x_zp"] * c["wq"].astype(np.int64).sum(1)
        real = raw * (np.float64(np.float32(c["x_scale"])) * c["w_scales"].astype(np.float32).astype(np.float64)) + c["bias"]
        f = host(cabi.linear_f32(x, pw, c["x_scale"], c["x_zp"], ws, b))
        # the product of the scales and the fused multiply-add round once each
        np.testing.assert_allclose(f, real, rtol=3 * 2.0 ** -24, atol=3 * 2.0 ** -24 * np.abs(real).max())
    finally:
        cabi.force_linear_config(-1)
