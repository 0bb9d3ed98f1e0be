"""Pointwise convolutions around the ends of a piece of 16 pixels, of a block of 64 (32) channels and of the tensor, against
the oracle: most pieces are read without a check, the tensor's last bytes with one."""
import numpy as np
import pytest

import oracle
from gpu_util import dev, host, say
from test_gpu_conv import LSB_TOL, _conv_case, cabi  # noqa: F401
from test_gpu_depthwise_channels import _at

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("height,width", [(1, 15), (1, 16), (1, 17), (3, 11), (48, 1), (53, 61), (113, 450)])
@pytest.mark.parametrize("ic,oc", [(16, 64), (3, 24), (24, 144), (5, 7), (93, 130), (64, 200), (255, 40), (256, 33)])
@pytest.mark.parametrize("x_signed,offset", [(False, 0), (True, 3)])
def test_pieces(cabi, height, width, ic, oc, x_signed, offset):  # noqa: F811
    if height * width > 5000 and ic * oc > 4000:
        pytest.skip("the oracle takes long; the smaller images have the same edges")
    say("pointwise", height, width, ic, oc, x_signed, offset)
    c = _conv_case(1, height, width, ic, oc, 1, 1, 0, 1, 1, seed=height + ic + oc, x_signed=x_signed)
    args = (c["stride"], c["padding"], c["dilation"], c["groups"])
    if c["xq"].size < 16:
        pytest.skip("the kernel wants 16 bytes")
    g = cabi.conv_geom(c["xq"].shape, c["wq"].shape, *args)
    pw = cabi.PackedConv2d(dev(c["wq"]), g)
    ws, bias, x = dev(c["w_scales"].astype(np.float32)), dev(c["bias"]), _at(c["xq"], offset)
    rng = np.random.default_rng(ic)
    cabi.force_conv_path(9)
    try:
        sums = host(cabi.conv2d_acc32(x, pw, g, c["x_zp"]))
        np.testing.assert_array_equal(sums, oracle.conv2d_acc32(c["xq"], c["wq"], *args, c["x_zp"], nthreads=8))
        for activation, residual, signed in (("none", False, x_signed), ("relu", True, False), ("none", True, True),
                                             ("silu", False, False), ("silu", True, True)):
            lo, hi = (-128, 128) if signed else (0, 256)
            dt = np.int8 if signed else np.uint8
            acc = rng.integers(lo, hi, sums.shape, dtype=dt) if residual else None
            zp, acc_zp = (-128 if residual else -20, -7) if signed else (0 if residual else 30, 110)
            want = oracle.conv2d_fused(c["xq"], c["x_scale"], c["x_zp"], c["wq"], c["w_scales"], c["bias"], *args,
                                       c["out_scale"], zp, accum=acc, accum_scale=0.35, accum_zp=acc_zp,
                                       activation=activation, out_signed=signed, nthreads=8)
            out = _at(np.zeros(sums.shape, dt), offset)
            got = host(cabi.conv2d_fused(x, pw, g, c["x_scale"], c["x_zp"], ws, bias, c["out_scale"], zp,
                                         accum=None if acc is None else _at(acc, offset), accum_scale=0.35,
                                         accum_zp=acc_zp, activation=activation, out_signed=signed, out=out))
            d = np.abs(got.astype(np.int32) - want.astype(np.int32))
            if activation == "silu":   # expf on the device and on the host may differ in the last bit
                assert d.max() <= LSB_TOL and np.count_nonzero(d) <= max(2, 0.001 * d.size), (d.max(), np.count_nonzero(d))
            else:
                assert d.max() == 0, (activation, np.count_nonzero(d), d.max())
    finally:
        cabi.force_conv_path(-1)


@pytest.mark.parametrize("ic,oc,height,width", [(24, 512, 1, 17), (24, 513, 9, 31), (100, 1030, 40, 41),  # eight channel blocks and more
                                                (96, 512, 59, 118), (16, 570, 73, 75),  # ... a piece more for some groups
                                                (16, 24576, 7, 19), (16, 32770, 5, 23),  # eight groups, and five
                                                (192, 320, 30, 30), (144, 768, 40, 45), (150, 190, 91, 91),  # three k-steps
                                                (200, 200, 128, 128), (256, 330, 127, 129), (256, 512, 33, 31)])  # four
def test_many_blocks_and_choice(cabi, ic, oc, height, width):  # noqa: F811
    """Waves placed by XCD, and wide layers by the automatic choice, against the oracle."""
    say("pointwise blocks", ic, oc, height, width)
    c = _conv_case(1, height, width, ic, oc, 1, 1, 0, 1, 1, seed=ic + oc, relu=True)
    args = (c["stride"], c["padding"], c["dilation"], c["groups"])
    g = cabi.conv_geom(c["xq"].shape, c["wq"].shape, *args)
    pw, ws, bias = cabi.PackedConv2d(dev(c["wq"]), g), dev(c["w_scales"].astype(np.float32)), dev(c["bias"])
    want = oracle.conv2d(c["xq"], c["x_scale"], c["x_zp"], c["wq"], c["w_scales"], c["bias"], *args, c["out_scale"],
                         c["out_zp"], relu=True, nthreads=8)
    for path in (9, -1):
        cabi.force_conv_path(path)
        try:
            got = host(cabi.conv2d(dev(c["xq"]), pw, g, c["x_scale"], c["x_zp"], ws, bias, c["out_scale"], c["out_zp"],
                                   relu=True))
        finally:
            cabi.force_conv_path(-1)
        np.testing.assert_array_equal(got, want)
