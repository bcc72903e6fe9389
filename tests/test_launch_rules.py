"""The rules that say how a backward is launched, on the CPU: a device that cannot be asked for its compute units."""
import os
import subprocess

import pytest

from jvp_flash_attention_amd import build

PROGRAM = """
#include <cstdio>
#include "split.hpp"
using namespace jvpfa;
template <int D> int all(long long b) {
  int one = 0;
  for (int f = 0; f < 32; ++f) {
    one += launch_both<D, BWD_PLAIN>(b, 2 * b, f & 1, f & 2, f & 4, false, f & 8, f & 16);
    one += launch_both<D, BWD_DUAL>(2 * b, b, f & 1, f & 2, f & 4, f & 8, false, f & 16);
    one += launch_both_f32(b, 3 * b, f & 1);
  }
  return one;
}
int main() {
  int one = 0;
  for (long long b : {1LL, 255LL, 300LL, 5000LL}) one += all<32>(b) + all<64>(b) + all<128>(b) + all<256>(b);
  std::printf("%d %d\\n", device_cus(), one);
}
"""


@pytest.mark.skipif(not os.path.exists(build.HIPCC), reason="no HIP compiler")
def test_device_that_cannot_be_asked(tmp_path):
    """Two launches, whatever the grid (and no division by the number of units)."""
    src, exe = tmp_path / "rules.hip", tmp_path / "rules"
    src.write_text(PROGRAM)
    subprocess.run([build.HIPCC, *build.FLAGS, "-I", build.CSRC, str(src), "-o", str(exe)], check=True, capture_output=True)
    run = subprocess.run([str(exe)], env={**os.environ, "HIP_VISIBLE_DEVICES": "-1"}, capture_output=True, text=True)
    assert run.returncode == 0, run.returncode
    assert run.stdout.split() == ["0", "0"]
