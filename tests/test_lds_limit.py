"""csrc/lds_limit.h on the host: a kernel's LDS limit is raised once on every
device that launches it, also where another device came first or a first
request failed."""

import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
PROGRAM = r"""
#include <cstdio>
enum hipError_t { hipSuccess, hipErrorUnknown };
enum { hipFuncAttributeMaxDynamicSharedMemorySize };
static int device = 0, calls[4], fail = 0;
static hipError_t hipGetDevice(int* d) { *d = device; return hipSuccess; }
static hipError_t hipFuncSetAttribute(const void*, int, int bytes) {
  if (fail) return hipErrorUnknown;
  calls[device] += bytes;
  return hipSuccess;
}
#include "lds_limit.h"
int main() {
  std::atomic<unsigned long long> a{0}, b{0};
  const int order[] = {0, 0, 1, 0, 1, 3};
  for (int d : order) {
    device = d;
    lds_limit(nullptr, 1, a);
  }
  lds_limit(nullptr, 10, b);      // another kernel on device 3
  device = 2;
  fail = 1;
  lds_limit(nullptr, 1, a);       // refused: asked again later
  fail = 0;
  lds_limit(nullptr, 1, a);
  std::printf("%d %d %d %d\n", calls[0], calls[1], calls[2], calls[3]);
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")
def test_every_device_is_asked(tmp_path):
    src = tmp_path / "main.cpp"
    src.write_text(PROGRAM)
    exe = tmp_path / "main"
    subprocess.run(["g++", "-std=c++17", "-I", str(ROOT / "csrc"), str(src),
                    "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True)
    assert out.stdout.split() == ["1", "1", "1", "11"]


def test_launchers_use_it():
    """No launcher keeps a limit of its own that covers the first device only."""
    for path in sorted((ROOT / "csrc").glob("*.hip")):
        if path.stem.endswith("_hip"):
            continue
        text = path.read_text()
        assert "static bool once" not in text, path.name
