"""The implicit GEMM's k order in a table: channel blocks that do not fill a stage, strides, dilations, groups, the table's
limits (63 taps, 16 KiB of K) and what lies beyond them, against the oracle."""
import numpy as np
import pytest

import oracle
from gpu_util import say
from test_gpu_conv import _check, _conv_case, _run, cabi  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("spec,wave_groups,tile_rows", [
    # batch, height, width, channels in, out, kernel, stride, padding, dilation, groups
    ((1, 5, 7, 16, 16, 2, 1, 0, 1, 1), 0, 0),        # one stage: shorter than the pipeline
    ((1, 5, 7, 16, 16, 3, 1, 3, 1, 1), 0, 0),        # windows wholly in the padding
    ((2, 9, 11, 32, 70, 3, 2, 1, 1, 1), 0, 0),       # two blocks per tap
    ((2, 9, 11, 48, 64, 3, 1, 2, 2, 1), 0, 0),       # three
    ((1, 13, 9, 160, 48, 3, 3, 0, 1, 2), 0, 0),      # five, two groups, stride 3
    ((1, 12, 12, 80, 64, 5, 1, 6, 3, 1), 0, 0),      # dilation 3: outer taps outside for every window
    ((3, 8, 8, 64, 64, 4, 1, 2, 1, 1), 2, 0),
    ((3, 8, 8, 64, 130, 4, 1, 2, 1, 1), 4, 0),
    ((3, 8, 8, 64, 64, 4, 2, 2, 1, 1), 2, 128),
    ((1, 9, 9, 320, 64, 7, 1, 3, 1, 1), 0, 0),       # 980 chunks
    ((1, 4, 5, 1024, 20, 4, 1, 2, 1, 1), 4, 0),      # 1024: the whole table
    ((1, 4, 5, 1040, 20, 4, 1, 2, 1, 1), 4, 0),      # 1040: past it
    ((1, 9, 9, 16, 64, 8, 1, 4, 1, 1), 2, 0),        # 64 taps: past it
])
@pytest.mark.parametrize("x_signed", [False, True])
def test_conv_gemm_table(cabi, spec, wave_groups, tile_rows, x_signed):  # noqa: F811
    say("conv gemm table", spec, wave_groups, tile_rows, x_signed)
    c = _conv_case(*spec, seed=sum(spec), x_signed=x_signed, relu=x_signed)
    cabi.force_conv_path(2)
    cabi.force_conv_tile(tile_rows, wave_groups)
    try:
        y, acc, _ = _run(cabi, c)
    finally:
        cabi.force_conv_path(-1)
        cabi.force_conv_tile(0, 0)
    args = (c["stride"], c["padding"], c["dilation"], c["groups"])
    np.testing.assert_array_equal(acc, oracle.conv2d_acc32(c["xq"], c["wq"], *args, c["x_zp"], nthreads=8))
    _check(y, oracle.conv2d(c["xq"], c["x_scale"], c["x_zp"], c["wq"], c["w_scales"], c["bias"], *args, c["out_scale"],
                            c["out_zp"], relu=c["relu"], nthreads=8), "table")
