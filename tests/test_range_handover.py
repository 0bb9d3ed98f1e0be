"""How the blocks of the range pass hand their pairs to the last one, read off the device code that the kernel's source
compiles to (no GPU): the order there is what the result rests on, and no run on a quiet chip would show it missing."""
import os
import re
import subprocess

import pytest
from torch_musa_amd import build


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    out = tmp_path_factory.mktemp("handover") / "quantize.s"
    subprocess.run([build._hipcc(), "-x", "hip", *build.DEVICE_FLAGS, "-I", os.path.join(build.ROOT, "include"),
                    "--offload-device-only", "-S", os.path.join(build.CSRC, "kernels", "quantize.hip"), "-o", str(out)],
                   check=True, capture_output=True)
    found = re.findall(r"^(_ZN3tmq\S*minmax_partial_kernel\S*):(.*?)^\.Lfunc_end", out.read_text(), re.S | re.M)
    assert len(found) == 2   # both kinds of load
    return [[line.split(";")[0].strip() for line in body.split("\n")] for _, body in found]


def test_pairs_are_out_before_the_count_and_read_behind_it(kernels):
    for code in kernels:
        at = {what: [i for i, line in enumerate(code) if re.match(what, line)]
              for what in ("global_atomic_swap_x2", "global_atomic_inc", r"buffer_inv sc1", r"s_waitcnt vmcnt\(0\)",
                           r"global_load_dwordx2 .*sc1", "buffer_wbl2", "s_barrier")}
        (swap,), (count,) = at["global_atomic_swap_x2"], at["global_atomic_inc"]
        (fence,), (load,) = at["buffer_inv sc1"], at[r"global_load_dwordx2 .*sc1"]
        # a block counts itself once its exchange has answered
        assert any(swap < i < count for i in at[r"s_waitcnt vmcnt\(0\)"])
        # the last block's counting wave acquires at agent scope once it has the count's answer, and all its
        # waves read the pairs behind a barrier that follows
        assert any(count < i < fence for i in at[r"s_waitcnt vmcnt\(0\)"])
        assert any(fence < i < load for i in at["s_barrier"])
        # and nothing writes an L2 back
        assert not at["buffer_wbl2"]
