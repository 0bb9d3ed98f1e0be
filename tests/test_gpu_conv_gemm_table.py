"""The implicit GEMM's k order in a table: channel blocks that do not fill a stage, strides, dilations, groups, the table's
limits (63 taps, 8128 chunks of 16 bytes) and what lies beyond them, against the oracle."""
import numpy as np
import pytest

import oracle
from gpu_util import dev, host, say
from test_gpu_conv import LSB_TOL, _check, _conv_case, _run, cabi  # noqa: F401

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
    ((1, 9, 9, 160, 70, 3, 1, 1, 1, 1), 1, 0),       # copies into LDS, 64 x 64 tiles
    ((5, 7, 7, 48, 130, 3, 1, 1, 1, 1), 0, 128),     # 128 x 128: three images per tile, channels one past the tile
    ((140, 3, 3, 64, 33, 3, 3, 1, 1, 1), 0, 128),    # an image per row and partly padding
    ((3, 9, 10, 64, 257, 3, 2, 1, 1, 1), 0, 256),    # 128 x 256
    ((1, 12, 11, 208, 250, 1, 1, 0, 1, 1), 0, 256),  # one tap, rows and channels just past and short of the tile
    ((2, 11, 12, 96, 96, 3, 1, 2, 1, 2), 0, 256),    # two groups
    ((1, 13, 10, 144, 16, 1, 1, 0, 1, 1), 0, 128),   # three stages, the copies' ring
    ((1, 13, 10, 128, 16, 1, 1, 0, 1, 1), 0, 128),   # two: the cursor
    ((1, 9, 9, 320, 64, 7, 1, 3, 1, 1), 0, 0),       # 980 chunks
    ((1, 4, 5, 1024, 20, 4, 1, 2, 1, 1), 4, 0),      # 1024
    ((1, 4, 5, 1040, 20, 4, 1, 2, 1, 1), 4, 0),      # 1040
    ((1, 4, 5, 2048, 70, 3, 1, 2, 2, 1), 0, 128),    # 1152: dilated, direct copies
    ((1, 3, 4, 8128, 20, 4, 1, 2, 1, 1), 4, 0),      # 8128: the whole table
    ((1, 3, 4, 8128, 20, 4, 1, 2, 1, 1), 0, 256),    # ... beside the largest tile's stages
    ((1, 3, 4, 8144, 20, 4, 1, 2, 1, 1), 4, 0),      # 8144: past it
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


@pytest.mark.parametrize("ic,oc,height,tile_rows", [(272, 70, 9, 0), (464, 256, 17, 128), (1024, 40, 8, 256),
                                                    (304, 130, 11, -1), (320, 320, 57, -1), (464, 300, 81, -1), (784, 64, 129, -1)])
@pytest.mark.parametrize("residual,activation", [(False, "relu"), (False, "silu"), (True, "relu"), (True, "silu")])
def test_wide_pointwise(cabi, ic, oc, height, tile_rows, residual, activation):  # noqa: F811
    """Wide pointwise layers with residual and SiLU in the GEMM's epilogue: pinned, and (-1) by the rule's own choice."""
    say("wide pointwise", ic, oc, height, tile_rows, residual, activation)
    rng = np.random.default_rng(ic + oc)
    c = _conv_case(1, height, 131, ic, oc, 1, 1, 0, 1, 1, seed=ic)
    acc = rng.integers(0, 256, (1, height, 131, oc), dtype=np.uint8) if residual else None
    g = cabi.conv_geom(c["xq"].shape, c["wq"].shape, (1, 1), (0, 0), (1, 1), 1)
    pw = cabi.PackedConv2d(dev(c["wq"]), g)
    if tile_rows >= 0:
        cabi.force_conv_path(2)
        cabi.force_conv_tile(tile_rows, 0)
    try:
        y = host(cabi.conv2d_fused(dev(c["xq"]), pw, g, c["x_scale"], c["x_zp"], dev(c["w_scales"].astype(np.float32)),
                                   dev(c["bias"]), c["out_scale"], 20, accum=None if acc is None else dev(acc),
                                   accum_scale=0.35, accum_zp=110, activation=activation))
    finally:
        cabi.force_conv_path(-1)
        cabi.force_conv_tile(0, 0)
    want = oracle.conv2d_fused(c["xq"], c["x_scale"], c["x_zp"], c["wq"], c["w_scales"], c["bias"], (1, 1), (0, 0), (1, 1), 1,
                               c["out_scale"], 20, accum=acc, accum_scale=0.35, accum_zp=110, activation=activation, nthreads=8)
    d = np.abs(y.astype(np.int32) - want.astype(np.int32))
    if activation == "silu":  # expf on the device and on the host may differ in the last bit
        assert d.max() <= LSB_TOL and np.count_nonzero(d) <= max(2, 0.001 * d.size), (d.max(), np.count_nonzero(d))
    else:
        assert d.max() == 0, (np.count_nonzero(d), d.max())


@pytest.mark.parametrize("spec", [
    # layers without a table, by the rule's own choice
    (1, 9, 9, 32, 20, 9, 1, 4, 1, 1),          # 41 stages: four wave groups, ten stages each and eleven
    (2, 10, 9, 64, 70, 9, 2, 4, 1, 2),         # the same over two groups
    (1, 6, 7, 32, 33, 8, 1, 6, 2, 1),          # 32 stages, windows reaching past the image on all sides
    (5, 36, 34, 32, 130, 8, 1, 3, 1, 1),       # 5775 pixels x 130 channels: 128 x 64 tiles, two groups of 16 stages
    (5, 36, 34, 32, 130, 9, 1, 4, 1, 1),       # the same of 21 and 20
    (1, 40, 52, 48, 72, 9, 1, 4, 1, 1),        # 61 stages
    (1, 30, 31, 16, 40, 8, 1, 4, 1, 1),        # 16 stages: one group
    (1, 129, 130, 32, 70, 1, 1, 0, 1, 1),      # one stage, 128 x 128 tiles
    (1, 257, 257, 32, 48, 1, 1, 0, 1, 1),      # one stage, 256 x 64 tiles
    (1, 513, 515, 112, 64, 1, 2, 0, 1, 1),     # two, every second pixel
])
@pytest.mark.parametrize("x_signed", [False, True])
def test_conv_gemm_walk(cabi, spec, x_signed):  # noqa: F811
    say("conv gemm walk", spec, x_signed)
    c = _conv_case(*spec, seed=sum(spec), x_signed=x_signed, relu=x_signed)
    cabi.force_conv_path(2)
    try:
        y, acc, _ = _run(cabi, c)
    finally:
        cabi.force_conv_path(-1)
    args = (c["stride"], c["padding"], c["dilation"], c["groups"])
    np.testing.assert_array_equal(acc, oracle.conv2d_acc32(c["xq"], c["wq"], *args, c["x_zp"], nthreads=8))
    _check(y, oracle.conv2d(c["xq"], c["x_scale"], c["x_zp"], c["wq"], c["w_scales"], c["bias"], *args, c["out_scale"],
                            c["out_zp"], relu=c["relu"], nthreads=8), "walk")


@pytest.mark.parametrize("spec,wave_groups,tile_rows", [
    ((1, 9, 9, 64, 64, 3, 1, 1, 1, 1), 4, 128),    # no such tile
    ((1, 9, 9, 128, 64, 3, 1, 1, 1, 1), 2, 256),   # 128 x 256: one group
    ((1, 9, 9, 64, 64, 3, 1, 1, 1, 1), 0, 64),     # no such height
    ((1, 9, 9, 64, 64, 3, 1, 1, 1, 1), 0, 192),
    ((1, 9, 9, 192, 64, 3, 1, 1, 1, 1), 3, 0),     # three groups
    ((1, 9, 9, 64, 64, 3, 1, 1, 1, 1), 2, 0),      # nine stages
    ((1, 9, 9, 32, 64, 9, 1, 4, 1, 1), 2, 0),      # 41, without a table
    ((1, 9, 9, 16, 64, 8, 1, 4, 1, 1), 0, 256),    # 128 x 256 without a table
    ((1, 9, 9, 128, 64, 1, 1, 0, 1, 1), 0, 256),
])
def test_conv_gemm_pins_refused(cabi, spec, wave_groups, tile_rows):  # noqa: F811
    say("conv gemm pins refused", spec, wave_groups, tile_rows)
    c = _conv_case(*spec, seed=sum(spec))
    cabi.force_conv_path(2)
    cabi.force_conv_tile(tile_rows, wave_groups)
    try:
        with pytest.raises(cabi.TmqError):
            _run(cabi, c)
    finally:
        cabi.force_conv_path(-1)
        cabi.force_conv_tile(0, 0)


@pytest.mark.parametrize("wave_groups,tile_rows", [(1, 0), (2, 0), (4, 0), (2, 128), (1, 128)])
def test_conv_gemm_walk_pinned(cabi, wave_groups, tile_rows):  # noqa: F811
    say("conv gemm walk pinned", wave_groups, tile_rows)
    c = _conv_case(2, 11, 12, 80, 70, 8, 1, 4, 1, 1, seed=wave_groups + tile_rows)
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
                            c["out_zp"], relu=c["relu"], nthreads=8), "walk pinned")


@pytest.mark.parametrize("spec", [
    (1, 7, 9, 320, 33, 3, 1, 1, 1, 1),     # 45 stages: two wave groups, 23 and 22
    (2, 9, 10, 448, 70, 3, 2, 2, 2, 2),    # 32 stages each (31.5) over two groups
    (1, 8, 9, 192, 40, 7, 1, 3, 1, 1),     # 147: four, 37, 37, 37 and 36
    (1, 7, 7, 912, 20, 3, 1, 1, 1, 1),     # 129 (128.25): 33, 32, 32 and 32
    (5, 35, 33, 320, 130, 3, 1, 1, 1, 1),  # 45 over 128 x 64 tiles
])
@pytest.mark.parametrize("x_signed", [False, True])
def test_conv_gemm_uneven_groups(cabi, spec, x_signed):  # noqa: F811
    """Stage counts that the wave groups do not divide, by the rule's own choice."""
    say("conv gemm uneven groups", spec, x_signed)
    c = _conv_case(*spec, seed=sum(spec), x_signed=x_signed, relu=x_signed)
    cabi.force_conv_path(2)
    try:
        y, acc, _ = _run(cabi, c)
    finally:
        cabi.force_conv_path(-1)
    args = (c["stride"], c["padding"], c["dilation"], c["groups"])
    np.testing.assert_array_equal(acc, oracle.conv2d_acc32(c["xq"], c["wq"], *args, c["x_zp"], nthreads=8))
    _check(y, oracle.conv2d(c["xq"], c["x_scale"], c["x_zp"], c["wq"], c["w_scales"], c["bias"], *args, c["out_scale"],
                            c["out_zp"], relu=c["relu"], nthreads=8), "uneven groups")
