"""Tiles of 32 rows whose waves walk their shares of K in pieces: the host's choice of them stays inside what the kernel's
index arithmetic and the measured range allow, and no scratch memory is asked for beside them."""
import numpy as np

from torch_musa_amd import cabi


def _ceil(a, b):
    return -(-a // b)


def test_choice_and_scratch():
    rng = np.random.default_rng(5)
    seen = set()
    for _ in range(20000):
        m = int(2 ** rng.uniform(4, 12.5))
        n = int(2 ** rng.uniform(0, 13.5))
        k = 16 * int(2 ** rng.uniform(7.5, 10))
        c = cabi.linear_kernel_choice(m, n, k, workspace=True)
        if c["kernel"] - 1 not in (29, 30):
            assert not (m > (32 if k >= 7680 else 48) and 5632 <= k <= 12288 and _ceil(m, 32) * _ceil(n, 32) <= 256), (m, n, k, c)
            continue
        what = (m, n, k, c)
        assert m > 32 and 4096 < k <= 12288 and c["tile_channels"] == 32 * (c["kernel"] - 29) and c["waves"] == 8 and c["splits"] == 1, what
        assert c["blocks"] == c["tiles"] == _ceil(m, 32) * _ceil(n, c["tile_channels"]) <= 256, what
        assert cabi.linear_kernel_choice(m, n, k, workspace=True, forced=c["kernel"]) == c, what
        assert cabi.lib().tmq_linear_scratch_bytes(m, n, k, 1) == 0, what
        # off the grid: room for the copy, and for nothing else
        assert cabi.lib().tmq_linear_scratch_bytes(m, n, k - 1, 0) == _ceil(m * k, 256) * 256, what
        seen.add(c["tile_channels"])
    assert seen == {32, 64}
