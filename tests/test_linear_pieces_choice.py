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
            streamed = m <= 40 and n * k > 17 << 20 and k < 10240
            assert not (m > (32 if k >= 7680 else 48) and 5632 <= k <= 12288 and _ceil(m, 32) * _ceil(n, 32) <= 256
                        and not streamed), (m, n, k, c)
            continue
        what = (m, n, k, c)
        assert not (m <= 40 and n * k > 17 << 20 and k < 10240), what
        assert m > 32 and 4096 < k <= 12288 and c["tile_channels"] == 32 * (c["kernel"] - 29) and c["waves"] == 8 and c["splits"] == 1, what
        assert c["blocks"] == c["tiles"] == _ceil(m, 32) * _ceil(n, c["tile_channels"]) <= 256, what
        assert cabi.linear_kernel_choice(m, n, k, workspace=True, forced=c["kernel"]) == c, what
        assert cabi.lib().tmq_linear_scratch_bytes(m, n, k, 1) == 0, what
        # off the grid: room for the copy, and for nothing else
        assert cabi.lib().tmq_linear_scratch_bytes(m, n, k - 1, 0) == _ceil(m * k, 256) * 256, what
        seen.add(c["tile_channels"])
    assert seen == {32, 64}


def test_lines_between_128_x_128_and_128_x_256_tiles():
    # (just past a round of the former, of many rows: the shapes that were measured on either side)
    for m, n, k, kernel in ((1779, 2544, 7424, 7), (2018, 2432, 7616, 7), (1732, 2768, 7168, 7), (1979, 2496, 6528, 7),
                            (1751, 2496, 5824, 19), (2613, 1792, 6800, 19), (3379, 1344, 7760, 19), (2798, 1536, 4160, 19),
                            (1234, 3440, 4992, 7), (1650, 2512, 8960, 7), (479, 9984, 2816, 19), (640, 8192, 4096, 7)):
        assert cabi.linear_kernel_choice(m, n, k, workspace=True)["kernel"] - 1 == kernel, (m, n, k)


def test_split_along_k_where_the_ring_of_phases_would_run():
    # (us, split | phases: 34.5 | 35.6, 26.2 | 32.1, 27.2 | 29.0, 35.7 | 40.6, 23.4 | 26.5; the others, split | lone tiles' ring: 28.4 | 21.1,
    # 25.9 | 21.3, 27.2 | 23.3)
    for m, n, k in ((128, 7038, 10960), (114, 4815, 10576), (119, 6172, 9056), (123, 7505, 13184), (128, 4200, 8240)):
        assert cabi.linear_kernel_choice(m, n, k, workspace=True)["kernel"] - 1 == 13, (m, n, k)
        assert cabi.linear_kernel_choice(m, n, k, workspace=False)["kernel"] - 1 == 21, (m, n, k)
    for m, n, k in ((661, 1408, 8544), (478, 1152, 8736), (168, 4736, 8656)):
        for workspace in (False, True):
            assert cabi.linear_kernel_choice(m, n, k, workspace=workspace)["kernel"] - 1 == 2, (m, n, k)
    # rows too far apart for the ring's copies: the split, as a workspace asks for
    assert cabi.linear_kernel_choice(478, 1152, 8736, ldx=2 ** 23 + 16, workspace=True)["kernel"] - 1 == 13


def test_no_room_for_a_split_that_is_not_made():
    rng = np.random.default_rng(11)
    asked = spared = 0
    for _ in range(20000):
        m, n, k = int(2 ** rng.uniform(4, 12)), int(2 ** rng.uniform(4, 14)), 16 * int(2 ** rng.uniform(6, 10))
        plan = cabi.lib().tmq_linear_workspace_bytes(m, n, k)
        uses = any(cabi.linear_kernel_choice(m, n, k, out=out, workspace=True)["kernel"] !=
                   cabi.linear_kernel_choice(m, n, k, out=out, workspace=False)["kernel"] for out in ("bytes", "f32"))
        assert cabi.lib().tmq_linear_scratch_bytes(m, n, k, 1) == (plan if uses else 0), (m, n, k)
        assert not uses or plan > 0
        asked, spared = asked + uses, spared + (plan > 0 and not uses)
    assert asked > 100 and spared > 100, (asked, spared)
    # (15.4 and 11.2 MB that nothing read)
    for m, n, k in ((478, 1152, 8736), (661, 1408, 8544)):
        assert cabi.lib().tmq_linear_workspace_bytes(m, n, k) > 11 * 10 ** 6 and cabi.lib().tmq_linear_scratch_bytes(m, n, k, 1) == 0
