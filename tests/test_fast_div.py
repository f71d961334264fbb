"""fast_div / div_by (csrc/cra_internal.hpp) on the host: exact for every
divisor class and at the edges of its 32-bit range."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "cron-root-attention_amd", "csrc")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

CHECKER = r"""
#include "cra_internal.hpp"
#include <cstdio>
using namespace cra;
int main() {
  long bad = 0, cases = 0;
  for (uint32_t d = 1; d < 70000; d += d < 3000 ? 1 : 61) {
    const FastDiv f = fast_div(d);
    auto check = [&](uint32_t n) { ++cases; bad += div_by(n, f) != n / d; };
    for (uint32_t k = 0; k < 40; ++k) {
      const uint32_t m = k < 20 ? k * d : (0xffffffffu / d - (k - 20)) * d;
      check(m); check(m - 1); check(m + 1);
      check(k * 107374183u);
    }
    check(0x7fffffffu); check(0xffffffffu);
  }
  for (uint32_t d : {1u << 20, (1u << 30) + 1, 0x7fffffffu})
    for (uint32_t n : {0u, d - 1, d, d + 1, 0xffffffffu}) { ++cases; bad += div_by(n, fast_div(d)) != n / d; }
  printf("%ld %ld\n", cases, bad);
  return 0;
}
"""


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not available")
def test_division_by_a_constant(tmp_path):
    src, exe = tmp_path / "div.cpp", tmp_path / "div"
    src.write_text(CHECKER)
    subprocess.run([HIPCC, "-std=c++17", "-O1", "-I", CSRC, str(src), "-o", str(exe)], check=True,
                   capture_output=True, timeout=300)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True, timeout=120)
    cases, bad = map(int, out.stdout.split())
    assert cases > 500000 and bad == 0
