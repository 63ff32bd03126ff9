"""The divisions by constants of the SrLab2 non-linearity (zh_divide.h) equal
the division bit for bit: compiled for the host and compared over every
subnormal quotient, both zeros and a stride through the other floats."""
import os
import subprocess

from zosimos_amd import build

SOURCE = r"""
#include <stdint.h>
#include <stdio.h>
#include <string.h>
#include "zh_divide.h"
static float f(uint32_t u) { float x; memcpy(&x, &u, 4); return x; }
static uint32_t b(float x) { uint32_t u; memcpy(&u, &x, 4); return u; }
static volatile float kA = 2700.0f, kB = 24389.0f;
int main() {
  long bad = 0;
  uint32_t step = 1;
  for (uint64_t u = 0; u < 0x7f800000u; u += step) {
    step = u < 0x09000000u ? 1 : 251;  // below 2^-109 every float
    for (uint32_t s = 0; s < 2; ++s) {
      const float x = f((uint32_t)u | s << 31);
      if (b(zh::div_2700(x)) != b(x / kA) || b(zh::div_const(x, 24389.0f, 1.0f / 24389.0f)) != b(x / kB)) ++bad;
    }
  }
  printf("%ld\n", bad);
  return 0;
}
"""


def test_constant_divisions_round_as_the_division(tmp_path):
    # The compiler of the device code (others may move the sign of a zero
    # through a negated fma).
    cxx = os.path.join(os.path.dirname(build.hipcc()), "amdclang++")
    src, exe = tmp_path / "divide.cpp", tmp_path / "divide"
    src.write_text(SOURCE)
    subprocess.run([cxx, "-O2", "-march=native", "-ffp-contract=off", "-D__host__=", "-D__device__=",
                    "-D__forceinline__=inline", "-I", build.CSRC, str(src), "-o", str(exe)], check=True)
    assert subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout.strip() == "0"
