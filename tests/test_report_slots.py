"""The host's report slots: which call may have one, shown on the host with calls that fail between two launches."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PROGRAM = r"""
#include "report_slots.h"

#include <cstdio>
#include <cstring>
#include <thread>

using tmq::ReportHold;
using tmq::ReportSlots;

#define CHECK(c) if (!(c)) { std::printf("line %d: %s\n", __LINE__, #c); return 1; }

int fails(bool drains) {   // the second launch of a chain fails while the first one's kernel runs
  ReportSlots slots(1);
  bool kernel_runs = false;
  {
    ReportHold a(slots);
    CHECK(a.slot() == 0);
    CHECK(a.queue([&] { kernel_runs = true; return TMQ_ERR_LAUNCH; },
                  [&] { if (drains) kernel_runs = false; return drains; }) == TMQ_ERR_LAUNCH);
  }
  ReportHold b(slots);
  CHECK(!(kernel_runs && b.slot() == 0));   // never while a kernel writes to it
  CHECK(b.slot() == (drains ? 0 : -1));     // -1, without a wait: it will not come back
  return 0;
}
int throws() {             // what raises between the call and its report leaves the slot with the device
  ReportSlots slots(2);
  int first = -1;
  try {
    ReportHold a(slots);
    first = a.slot();
    CHECK(a.queue([] { return TMQ_OK; }, [] { return true; }) == TMQ_OK);
    throw 1;
  } catch (int) {
  }
  ReportHold b(slots);
  CHECK(b.slot() == 1 - first);
  return 0;
}
int reports() {            // a call that has its report gives the slot back, with another ticket for the next
  ReportSlots slots(1);
  uint32_t first;
  {
    ReportHold a(slots);
    first = a.ticket();
    CHECK(a.queue([] { return TMQ_OK; }, [] { return false; }) == TMQ_OK);
    a.done();
  }
  ReportHold b(slots);
  CHECK(b.slot() == 0 && b.ticket() != first && b.ticket() != 0);
  return 0;
}
int waits() {              // a call without a slot waits for one
  ReportSlots slots(1);
  int got = -2;
  std::thread other;
  {
    ReportHold a(slots);
    other = std::thread([&] { ReportHold b(slots); got = b.slot(); });
  }
  other.join();
  CHECK(got == 0);
  return 0;
}

int main(int, char** argv) {
  if (!std::strcmp(argv[1], "drained")) return fails(true);
  if (!std::strcmp(argv[1], "lost")) return fails(false);
  if (!std::strcmp(argv[1], "throws")) return throws();
  if (!std::strcmp(argv[1], "reports")) return reports();
  return waits();
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    d = tmp_path_factory.mktemp("report_slots")
    (d / "t.cpp").write_text(PROGRAM)
    subprocess.run([os.environ.get("CXX", "g++"), "-std=c++17", "-O1", "-pthread", "-I", os.path.join(ROOT, "include"),
                    "-I", os.path.join(ROOT, "torch_musa_amd", "csrc", "aten"), str(d / "t.cpp"), "-o", str(d / "t")],
                   check=True)
    return str(d / "t")


@pytest.mark.parametrize("what", ["drained", "lost", "throws", "reports", "waits"])
def test_report_slots(program, what):
    got = subprocess.run([program, what], timeout=30, capture_output=True, text=True)
    assert got.returncode == 0, got.stdout
