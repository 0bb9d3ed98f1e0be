"""quantized::linear on one round of tiles of 32 rows whose activation rows lie off the 16-byte grid: tile and piece edges and a
last chunk of 1 to 15 bytes, rows of any pitch and address with the storage's ends at the first and last byte, against the oracle."""
import numpy as np
import pytest
import torch

import oracle
from gpu_util import dev, host, say
from test_gpu_linear import _check, _run, _tile_case, cabi  # noqa: F401


def _in_place(cabi, m, n, k):
    return cabi.lib().tmq_linear_rows_in_place(m, n, k)


@pytest.mark.gpu
# less than a chunk per wave; pieces of 128 and 256 bytes on either side of eight waves' shares; a last chunk of
# 1, 8 and 15 bytes; the end of the range
@pytest.mark.parametrize("k", [129, 255, 257, 511, 513, 1000, 1025, 2047, 2049, 2305, 4095, 4097, 12287])
@pytest.mark.parametrize("m,n", [(17, 1), (31, 33), (33, 64), (65, 129)])
def test_edges(cabi, k, m, n):  # noqa: F811
    assert _in_place(cabi, m, n, k) == 1
    say("ragged pieces", m, n, k)
    c = _tile_case(m, n, k, seed=m + n + k, x_signed=bool(k & 2), relu=bool(m & 2), bias=m != 33, per_channel=n != 64)
    want = oracle.linear(c["xq"], c["x_scale"], c["x_zp"], c["wq"], c["w_scales"], c["bias"], c["out_scale"], c["out_zp"],
                         relu=c["relu"], nthreads=8)
    cabi.use_linear_workspace = False
    try:
        y, acc, pw = _run(cabi, c, -1)
        np.testing.assert_array_equal(acc, oracle.linear_acc32(c["xq"], c["wq"], nthreads=8))
        _check(y, want, "ragged pieces")
        # an odd pitch and address: the last row ends where the storage does
        wide = torch.empty(m * (k + 3) + 1 - 3, dtype=dev(c["xq"]).dtype, device="cuda")
        rows = torch.as_strided(wide, (m, k), (k + 3, 1), 1).copy_(dev(c["xq"]))
        bias = None if c["bias"] is None else dev(c["bias"])
        scales = dev(c["w_scales"].astype(np.float32))
        args = (pw, c["x_scale"], c["x_zp"], scales, bias)
        _check(host(cabi.linear(rows, *args, c["out_scale"], c["out_zp"], relu=c["relu"])), want, "ragged pieces, odd pitch")
        assert torch.equal(cabi.linear_f32(rows, *args), cabi.linear_f32(dev(c["xq"]), *args))
    finally:
        cabi.use_linear_workspace = True


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(256, 1024, 1000), (257, 1024, 1000), (512, 1024, 1000), (513, 1024, 1000), (512, 1024, 501),
                                   (300, 700, 12289), (16, 300, 1001), (64, 130, 127), (64, 512, 4100), (40, 64, 9001)])
def test_either_side_of_the_lines(cabi, m, n, k):  # noqa: F811
    """The route and the plain kernel: the same bytes."""
    say("ragged pieces, lines", m, n, k)
    c = _tile_case(m, n, k, seed=m + n + k, x_signed=bool(m & 1), relu=False, bias=True, per_channel=True)
    want, _, _ = _run(cabi, c, 9)
    for workspace in (False, True):
        cabi.use_linear_workspace = workspace
        try:
            got, _, _ = _run(cabi, c, -1)
        finally:
            cabi.use_linear_workspace = True
        np.testing.assert_array_equal(got, want)


def test_route():
    from torch_musa_amd import cabi
    for m, n, k, one in ((16, 64, 1001, 0), (17, 64, 1001, 1), (17, 64, 127, 0), (17, 64, 129, 1), (512, 1024, 1000, 1),
                         (513, 1024, 1000, 0), (64, 64, 12287, 1), (64, 64, 12289, 0), (0, 64, 1001, 0)):
        assert _in_place(cabi, m, n, k) == one, (m, n, k)


FEW_ROWS = [(17, 2600, 6001, 1), (24, 64, 8001, 1), (24, 1000, 11001, 1), (24, 300, 7001, 1), (28, 2600, 10002, 1),
            (29, 2600, 6001, 0), (25, 300, 7001, 0), (24, 2600, 5631, 0), (24, 64, 8193, 0), (24, 300, 10002, 0), (24, 2600, 8004, 0), (17, 17, 12001, 0)]


def test_few_long_rows_are_copied_first():
    from torch_musa_amd import cabi
    for m, n, k, copied in FEW_ROWS:
        assert _in_place(cabi, m, n, k) == 1 - copied, (m, n, k)
        room = cabi.lib().tmq_linear_scratch_bytes(m, n, k, 0)
        assert room == (-(-(m * (-(-k // 16) * 16)) // 256) * 256 if copied else 0), (m, n, k, room)


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [s[:3] for s in FEW_ROWS[:5]])
def test_few_long_rows(cabi, m, n, k):  # noqa: F811
    """With the room for a copy and, read where they lie, without: the plain kernel's bytes."""
    say("few long rows", m, n, k)
    c = _tile_case(m, n, k, seed=m + n + k, x_signed=bool(m & 1), relu=False, bias=True, per_channel=True)
    want, _, _ = _run(cabi, c, 9)
    got, _, _ = _run(cabi, c, -1)
    np.testing.assert_array_equal(got, want)
    keep, cabi.linear_workspace = cabi.linear_workspace, torch.empty(cabi.lib().tmq_linear_scratch_bytes(m, n, k, 0), dtype=torch.uint8, device="cuda")
    try:
        got, _, _ = _run(cabi, c, -1)
    finally:
        cabi.linear_workspace = keep
    np.testing.assert_array_equal(got, want)
