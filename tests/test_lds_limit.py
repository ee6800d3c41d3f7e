"""A kernel's limit of dynamic LDS is raised on every device that it runs on: the helper against a runtime that counts (compiled for the
host), and no source with a flag of its own for all devices."""

import re
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "tokamak_amd" / "csrc"

PROGRAM = r"""
#include "lds_limit.h"
#include <cstdio>
static int device = 0, calls = 0, fails = 0;
extern "C" hipError_t hipGetDevice(int* d) { *d = device; return hipSuccess; }
extern "C" hipError_t hipGetLastError() { return hipSuccess; }
extern "C" hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int bytes) {
  ++calls;
  return fails || bytes != 1024 ? hipErrorInvalidValue : hipSuccess;
}
int main() {
  static tk::LdsLimits one, other;
  fails = 1;
  if (tk::raise_lds_limit(nullptr, 1024, one)) return 1;      // (and asks again)
  fails = 0;
  for (int pass = 0; pass < 3; ++pass)
    for (device = 0; device < 8; ++device)
      if (!tk::raise_lds_limit(nullptr, 1024, one)) return 2;
  device = 0;
  if (!tk::raise_lds_limit(nullptr, 1024, other)) return 3;
  device = 64;
  if (tk::raise_lds_limit(nullptr, 1024, one)) return 4;
  std::printf("%d\n", calls);
  return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None or not Path("/opt/rocm/include/hip").is_dir(), reason="no host compiler or no headers")
def test_the_limit_is_raised_once_a_device(tmp_path):
    (tmp_path / "limit.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", f"-I{CSRC}", "-I/opt/rocm/include", "limit.cpp", "-o", "limit"], cwd=tmp_path, check=True)
    out = subprocess.run([str(tmp_path / "limit")], check=True, capture_output=True, text=True).stdout
    assert int(out) == 1 + 8 + 1


def test_no_flag_holds_for_all_devices():
    assert not [s.name for s in sorted(CSRC.glob("*.hip")) if re.search(r"static bool raised(?!\[64\])", s.read_text())]
