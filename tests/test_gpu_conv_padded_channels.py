"""The copy with padded channels in front of the matrix kernels: tensors whose last blocks would be read past their end, and
block counts around a thread's four, against the oracle."""
import numpy as np
import pytest

import oracle
from gpu_util import say
from test_gpu_conv import _check, _conv_case, _run, cabi  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ic", [1, 3, 15, 17, 31, 40, 97])
@pytest.mark.parametrize("batch,height,width", [(1, 1, 16), (1, 3, 7), (1, 16, 16), (3, 19, 18)])
@pytest.mark.parametrize("x_signed", [False, True])
def test_padded_copy(cabi, ic, batch, height, width, x_signed):  # noqa: F811
    say("padded channels", ic, batch, height, width, x_signed)
    c = _conv_case(batch, height, width, ic, 20, 3, 1, 1, 1, 1, seed=ic + width, x_signed=x_signed)
    cabi.force_conv_path(8)
    try:
        y, acc, _ = _run(cabi, c)
    finally:
        cabi.force_conv_path(-1)
    args = (c["stride"], c["padding"], c["dilation"], c["groups"])
    np.testing.assert_array_equal(acc, oracle.conv2d_acc32(c["xq"], c["wq"], *args, c["x_zp"], nthreads=8))
    _check(y, oracle.conv2d(c["xq"], c["x_scale"], c["x_zp"], c["wq"], c["w_scales"], c["bias"], *args, c["out_scale"],
                            c["out_zp"], relu=c["relu"], nthreads=8), "padded")
