"""CPU check of the exact division of the brick cut (dda_math.h div_by): every divisor up to the longest axis of a ray,
dividends on both sides of a multiple over the whole range of quotients, the reciprocal one ulp off either way."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SRC = r"""
#include <cmath>
#include <cstdint>
#include <cstdio>
#include "dda_math.h"
int main() {
  long bad = 0, n_checked = 0;
  for (uint32_t n = 1; n <= 8192; ++n) {
    const float one = 1.0f / (float)n;
    const float invs[3] = {std::nextafterf(one, 0.0f), one, std::nextafterf(one, 2.0f)};
    for (uint32_t q = n % 13; q <= 16385; q += (q < 4 || q > 16380) ? 1 : 13)
      for (int k = -1; k <= 1; ++k) {
        if (q == 0 && k < 0) continue;
        const uint32_t X = q * n + k;
        for (float inv : invs) {
          uint32_t r = 0;
          const uint32_t got = vdbgpu::div_by(X, n, inv, r);
          bad += got != X / n || r != X % n;
          ++n_checked;
        }
      }
  }
  std::printf("%ld checked, %ld differ\n", n_checked, bad);
  return bad != 0;
}
"""


def test_div_by_is_exact(tmp_path):
    src = tmp_path / "div_by.cpp"
    src.write_text(SRC)
    exe = str(tmp_path / "div_by")
    subprocess.run(["g++", "-O2", "-std=c++17", "-I" + os.path.join(ROOT, "vdb_mapping_amd", "csrc"), str(src), "-o", exe],
                   check=True, timeout=300)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and " 0 differ" in r.stdout, r.stdout
