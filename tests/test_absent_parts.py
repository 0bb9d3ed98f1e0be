"""Blocks that wait for blocks that are not on the chip: which missing part each of them reads, on the host.  Every turn a running
block reads one part, so the turns until nothing is missing are what the wait costs."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PROGRAM = r"""
#include "absent_parts.h"

#include <cstdio>
#include <random>
#include <vector>

using tmq::absent_part;

// Turns of `running` blocks that see each other's finds between two turns.
int turns(uint64_t (&absent)[4], const std::vector<int>& running) {
  for (int n = 0;; ++n) {
    uint64_t next[4] = {absent[0], absent[1], absent[2], absent[3]};
    bool any = false;
    for (const int block : running) {
      const int part = absent_part(absent, block);
      if (part < 0) continue;
      if (part > 255 || (absent[part / 64] >> (part % 64) & 1) == 0) { std::printf("part %d is not absent\n", part); return -1; }
      next[part / 64] &= ~(uint64_t{1} << (part % 64));
      any = true;
    }
    if (!any) return n;
    for (int j = 0; j < 4; ++j) absent[j] = next[j];
  }
}
int main() {
  std::mt19937 rng(3);
  for (int blocks = 1; blocks <= 256; blocks += blocks < 70 ? 1 : 31)
    for (int run = 1; run <= blocks; ++run)
      for (int scattered = 0; scattered < 2; ++scattered) {
        std::vector<int> running, order(blocks);
        uint64_t absent[4] = {0, 0, 0, 0};
        for (int i = 0; i < blocks; ++i) order[i] = i;
        if (scattered)
          for (int i = blocks - 1; i > 0; --i) std::swap(order[i], order[rng() % (i + 1)]);
        for (int i = 0; i < blocks; ++i) {
          if (i < run) running.push_back(order[i]);
          else absent[order[i] / 64] |= uint64_t{1} << (order[i] % 64);
        }
        const int missing = blocks - run, n = turns(absent, running);
        // the first of the grid run: one part each until all are there.  Any blocks: some pick the same one
        if (n < 0 || n > (scattered ? missing : (missing + run - 1) / run) || (missing > 0 && n < 1)) {
          std::printf("%d of %d blocks, scattered %d: %d turns\n", run, blocks, scattered, n);
          return 1;
        }
      }
  return 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    folder = tmp_path_factory.mktemp("absent")
    (folder / "main.cpp").write_text(PROGRAM)
    out = folder / "main"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wno-unknown-pragmas", "-I", os.path.join(ROOT, "torch_musa_amd", "csrc", "kernels"),
                    str(folder / "main.cpp"), "-o", str(out)], check=True, capture_output=True)
    return out


def test_running_blocks_take_different_parts(program):
    done = subprocess.run([str(program)], capture_output=True, text=True, timeout=120)
    assert done.returncode == 0, done.stdout
