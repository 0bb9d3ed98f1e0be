"""quantized::linear on tiles of 64 x 128, 128 x 128 and 128 x 256 whose activation rows lie off the 16-byte grid: edges of tiles, last
chunks of 1 to 15 bytes, either side of the lines between them, rows of any pitch and address, every output type, against the oracle."""
import numpy as np
import pytest
import torch

import oracle
from gpu_util import dev, host, say
from test_gpu_linear import _check, _run, _tile_case, cabi  # noqa: F401


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [
    # one round of 64 x 128: just past a tile, the last chunk 1, 15 and 8 bytes; at the line (K = 1200 stays with 64 x 64)
    (1025, 1030, 1201), (1087, 1023, 1215), (1030, 1025, 2056), (1025, 1030, 1199), (96, 16321, 1249), (1025, 1030, 1537),
    # one round of 128 x 128: one row and channel past a tile, two stages and a byte; 288 and 289 tiles of 64 x 128 at K = 639, 641, 289 at 329, 331
    (1470, 2049, 129), (1025, 2049, 331), (1025, 2049, 329), (1030, 2060, 1000), (1150, 2047, 2063), (1152, 2048, 639), (1152, 2048, 641),
    (1088, 2049, 639), (3000, 1000, 377),
    # one round of 128 x 256, 64 x 128 below K = 480 up to 700 tiles of those
    (2049, 2049, 481), (2170, 2303, 1001), (2049, 2049, 479), (2881, 2049, 200),
    # more than that: 128 x 128 from K = 250 to 640, else a copy
    (2113, 4097, 249), (2113, 4097, 251), (2120, 4100, 639), (2113, 4097, 641),
    # few channels, few rows: as before
    (16640, 65, 300), (3000, 383, 1249), (3000, 384, 1249), (95, 16500, 1249)])
def test_edges(cabi, m, n, k):  # noqa: F811
    say("ragged tiles", m, n, k)
    c = _tile_case(m, n, k, seed=m + n + k, x_signed=bool(k & 2), relu=bool(m & 2), bias=m != 1030, per_channel=n != 2049)
    want = oracle.linear(c["xq"], c["x_scale"], c["x_zp"], c["wq"], c["w_scales"], c["bias"], c["out_scale"], c["out_zp"],
                         relu=c["relu"], nthreads=16)
    y, acc, pw = _run(cabi, c, -1)
    np.testing.assert_array_equal(acc, oracle.linear_acc32(c["xq"], c["wq"], nthreads=16))
    _check(y, want, "ragged tiles")
    # an odd pitch and address: the last row ends where the storage does
    wide = torch.empty(m * (k + 3) + 1 - 3, dtype=dev(c["xq"]).dtype, device="cuda")
    rows = torch.as_strided(wide, (m, k), (k + 3, 1), 1).copy_(dev(c["xq"]))
    bias = None if c["bias"] is None else dev(c["bias"])
    args = (pw, c["x_scale"], c["x_zp"], dev(c["w_scales"].astype(np.float32)), bias)
    _check(host(cabi.linear(rows, *args, c["out_scale"], c["out_zp"], relu=c["relu"])), want, "ragged tiles, odd pitch")
    # fp32: the rows where they lie and, padded with zeros onto the grid, on the kernels for those
    padded = torch.full((m, (k + 15) // 16 * 16), int(c["x_zp"]), dtype=wide.dtype, device="cuda")
    padded[:, :k] = rows
    wq = np.zeros((n, padded.shape[1]), c["wq"].dtype)
    wq[:, :k] = c["wq"]
    pw_padded = cabi.PackedLinear(dev(wq))
    assert torch.equal(cabi.linear_f32(rows, *args), cabi.linear_f32(padded, pw_padded, *args[1:]))


def test_room_for_a_copy():
    """0: the rows are read where they lie; else the copy and what follows it."""
    from torch_musa_amd import cabi
    for m, n, k, copies in ((1025, 1030, 1201, 0), (1025, 2049, 1000, 0), (1152, 2048, 639, 0), (2049, 2049, 1001, 0), (2113, 4097, 400, 0),
                            (2113, 4097, 1000, 1), (2113, 4097, 200, 1), (1025, 1030, 4001, 1), (2049, 2049, 3301, 1), (1025, 2049, 3301, 1), (256, 9000, 2001, 1), (256, 9000, 1999, 0),
                            (512, 11000, 2001, 1), (512, 11000, 1999, 0), (513, 11000, 2001, 0), (512, 8192, 2001, 0), (512, 8193, 2001, 1),
                            (2034, 6687, 637, 1), (2034, 6687, 399, 0), (2034, 6401, 401, 1), (2034, 6400, 401, 0),
                           
                            (17000, 65, 1001, 1), (17000, 65, 701, 0)):
        assert (cabi.lib().tmq_linear_scratch_bytes(m, n, k, 0) > 0) == bool(copies), (m, n, k)


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(300, 11010, 2003), (1290, 10505, 405)])
def test_copied_where_there_is_room(cabi, m, n, k):  # noqa: F811
    """The same bytes as the plain kernel's with the room for a copy and, in the tiles that need none, without it."""
    room = cabi.lib().tmq_linear_scratch_bytes(m, n, k, 0)
    assert room > 0
    say("ragged tiles, room", m, n, k)
    c = _tile_case(m, n, k, seed=m + n + k, x_signed=bool(m & 1), relu=False, bias=True, per_channel=True)
    want, _, _ = _run(cabi, c, 9)
    keep = cabi.linear_workspace
    try:
        for given in (None, torch.empty(room, dtype=torch.uint8, device="cuda")):
            cabi.linear_workspace = given
            got, _, _ = _run(cabi, c, -1)
            np.testing.assert_array_equal(got, want)
    finally:
        cabi.linear_workspace = keep
