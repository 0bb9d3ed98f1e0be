"""Reads near the end of a tensor: the offsets that the pointwise convolution kernel reads at, computed on the host
from the same function, on both sides of 2 GiB and 4 GiB."""
import ctypes as C
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE = """
#include "tail_read.h"
extern "C" void tail_read(int64_t o, int64_t bytes, int64_t* at, int* shift) {
  const tmq::TailRead r = tmq::tail_read16(o, bytes);
  *at = r.at;
  *shift = r.shift;
}
"""


@pytest.fixture(scope="module")
def tail_read(tmp_path_factory):
    d = tmp_path_factory.mktemp("tail_read")
    (d / "t.cpp").write_text(SOURCE)
    subprocess.run([os.environ.get("CXX", "g++"), "-std=c++17", "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__",
                    "-I/opt/rocm/include", "-I", os.path.join(ROOT, "torch_musa_amd", "csrc", "kernels"),
                    str(d / "t.cpp"), "-o", str(d / "t.so")], check=True)
    fn = C.CDLL(str(d / "t.so")).tail_read
    fn.argtypes = [C.c_int64, C.c_int64, C.POINTER(C.c_int64), C.POINTER(C.c_int)]

    def call(o, size):
        at, shift = C.c_int64(), C.c_int()
        fn(o, size, C.byref(at), C.byref(shift))
        return at.value, shift.value

    return call


@pytest.mark.parametrize("size", [16, 17, 100, 2**31 - 1, 2**31, 2**31 + 1, 2**31 + 16, 33 * 256 * 512 * 512,
                                  2**32 - 1, 2**32, 2**32 + 1, 2**32 + 2**31, 65 * 256 * 512 * 512, 2**40 + 3])
def test_reads_stay_in_the_tensor(tail_read, size):
    near = {d for b in (0, 2**31, 2**32, size - 2**31, size - 2**32, size) for d in range(b - 40, b + 40)}
    for o in sorted(o for o in near if 0 <= o < size):
        at, shift = tail_read(o, size)
        assert 0 <= at and at + 16 <= size, (o, size, at)
        assert 0 <= shift < 16 and at + shift == o, (o, size, at, shift)   # byte o is the value's first after the move
        assert shift == 0 or at == size - 16
