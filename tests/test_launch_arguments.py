"""A kernel's arguments reach it as its parameters say: one that a parameter is too narrow for does not compile."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE = """
#include "common.h"
void kernel(const float* x, int32_t n, uint32_t m, float f, int64_t k) {}
void launch(float* x, %s n, %s m, %s f) {
  tmq::enqueue(kernel, dim3(1), dim3(64), 0, nullptr, x, n, m, f, 7);
}
"""


@pytest.mark.parametrize("types,compiles", [
    (("int32_t", "uint32_t", "float"), True),
    (("uint8_t", "uint16_t", "float"), True),
    (("int64_t", "uint32_t", "float"), False),
    (("int32_t", "int32_t", "float"), False),
    (("int32_t", "uint32_t", "double"), False),
])
def test_no_narrowing(tmp_path, types, compiles):
    (tmp_path / "t.cpp").write_text(SOURCE % types)
    r = subprocess.run([os.environ.get("CXX", "g++"), "-std=c++17", "-fsyntax-only", "-Werror=narrowing",
                        "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I", os.path.join(ROOT, "include"),
                        "-I", os.path.join(ROOT, "torch_musa_amd", "csrc", "kernels"), str(tmp_path / "t.cpp")],
                       capture_output=True, text=True)
    assert (r.returncode == 0) == compiles, r.stderr
    if not compiles:
        assert "narrowing" in r.stderr, r.stderr
