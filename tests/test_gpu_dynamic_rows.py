"""quantized::linear_dynamic of up to 16 rows, which a block holds as float values: rows whose length is no multiple of four,
groups that end with a thread's last one, the most values it can hold, against the oracle."""
import numpy as np
import pytest

import oracle
from gpu_util import dev, host, say
from test_gpu_linear import cabi  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,k,n", [(1, 16, 20), (16, 17, 40), (3, 1363, 33), (16, 1023, 64), (16, 1024, 48), (5, 3275, 100),
                                   (7, 4679, 70), (16, 2047, 130), (16, 2048, 130), (4, 8192, 20),               # up to 8 groups a thread
                                   (9, 3641, 10240), (16, 4093, 10250), (16, 4096, 10300), (8, 8191, 10241), (13, 5036, 12000)])   # up to 16
@pytest.mark.parametrize("pin", [0, 9, 29])
def test_rows(cabi, m, k, n, pin):  # noqa: F811
    groups = m * ((k + 3) // 4)
    if (pin == 9 and 4 * groups > 16384) or (pin == 29 and k < 64):
        pytest.skip("not this kernel's")
    say("dynamic rows", m, k, n, pin)
    rng = np.random.default_rng(m * k + n)
    x = (rng.standard_normal((m, k)) * 1.5 + 0.3).astype(np.float32)
    x[m - 1, k - 1], x[0, k - 1] = 14.25, -11.5           # the extremes in rows' last groups
    w = rng.integers(-127, 128, (n, k)).astype(np.int8)
    ws = (rng.random(n) * 1e-3 + 1e-4).astype(np.float32)
    b = rng.standard_normal(n).astype(np.float32)
    assert cabi.lib().tmq_linear_dynamic_small_takes(m, n, k) == 1
    pw = cabi.PackedLinear(dev(w))
    y = np.empty((m, n), dtype=np.float32)
    yd = dev(y)
    d = cabi.LinearDesc()
    d.M, d.N, d.K, d.kernel = m, n, k, pin
    xd, wsd, bd = dev(x), dev(ws), dev(b)
    d.w_packed, d.w_colsum, d.w_scales, d.w_per_channel, d.bias = pw.packed.data_ptr(), pw.colsum.data_ptr(), wsd.data_ptr(), 1, bd.data_ptr()
    cabi.check(cabi.lib().tmq_linear_dynamic_small(d, xd.data_ptr(), k, 0, yd.data_ptr(), n, cabi.stream_ptr()), "dynamic rows")
    np.testing.assert_array_equal(host(yd), oracle.linear_dynamic(x, w, ws.astype(np.float64), b, False, False))
