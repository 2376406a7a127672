"""The cast kernels' quotient (eltwise.hip, RowQuant): a product with the rounded reciprocal of the scale
and one correction step in two fused multiply-adds, instead of the division. The same steps in C on the
CPU, against the division, for every bf16 mantissa over every fp32 scale mantissa (2^30 pairs): a
quotient's rounding does not depend on the exponents as long as nothing under- or overflows."""
import ctypes
import shutil
import subprocess

import pytest

SOURCE = r"""
#include <stdint.h>
#include <string.h>
static float from_bits(uint32_t u) { float f; memcpy(&f, &u, 4); return f; }
// pairs (x, scale) with scale mantissas [begin, end) whose corrected quotient is not x / scale
int64_t mismatches(uint32_t begin, uint32_t end) {
  int64_t bad = 0;
  for (uint32_t f = 0; f < 128; ++f) {
    const float x = from_bits(0x3f800000u | f << 16);
    int32_t part = 0;
    for (uint32_t m = begin; m < end; ++m) {
      const float scale = from_bits(0x3f800000u | m), rcp = 1.0f / scale;
      const float q0 = x * rcp;
      const float q = __builtin_fmaf(-__builtin_fmaf(q0, scale, -x), rcp, q0);
      part += q != x / scale;
    }
    bad += part;
  }
  return bad;
}
"""


def test_corrected_quotient_is_the_division(tmp_path):
    if shutil.which("gcc") is None or " fma" not in open("/proc/cpuinfo").read():
        pytest.skip("needs gcc and a CPU with fused multiply-add")
    src, lib = tmp_path / "q.c", tmp_path / "q.so"
    src.write_text(SOURCE)
    subprocess.run(["gcc", "-O3", "-mavx2", "-mfma", "-ffp-contract=off", "-shared", "-fPIC", str(src), "-o", str(lib)],
                   check=True)
    fn = ctypes.CDLL(str(lib)).mismatches
    fn.restype, fn.argtypes = ctypes.c_int64, [ctypes.c_uint32, ctypes.c_uint32]
    assert fn(0, 1 << 23) == 0
