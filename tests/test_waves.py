"""Seeds per wavefront (mkfit_amd/csrc/mkf_waves.h), compiled and run on the host: they follow the device's compute units
and what a compute unit holds."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include "mkf_waves.h"
#include <cassert>
using namespace mkf_find;

int main() {
  for (int cus : {1, 32, 64, 256, 304})
    for (size_t n : {(size_t)0, (size_t)1, (size_t)63, (size_t)500, (size_t)30011, (size_t)500000, (size_t)25000000}) {
      const int lanes = lanes_per_wave(n, cus);
      assert(lanes >= 1 && lanes <= 64 && (lanes & (lanes - 1)) == 0);
      // half as many would be enough for a wavefront per SIMD, and these are not too many for it
      assert(lanes == 1 || n >= (size_t)lanes * 4 * cus);
      assert(lanes == 64 || n < (size_t)lanes * 2 * 4 * cus);
      for (int per_cu : {1, 4, 6, 8})
        for (int most : {8, 10}) {
          const int s = seeds_per_wave(n, most, cus, per_cu);
          assert(s >= 1 && s <= most);
          assert(s == most || (n + s - 1) / s <= (size_t)cus * per_cu);          // all on the device at once
          assert(s == 1 || (n + s - 2) / (s - 1) > (size_t)cus * per_cu);        // with one seed fewer they are not
        }
    }
  assert(lanes_per_wave(30011, 256) == 16 && lanes_per_wave(30011, 64) == 64);
  assert(seeds_per_wave(10000, 10, 256, 8) == 5 && seeds_per_wave(5003, 10, 256, 6) == 4);
  return 0;
}
"""


def test_seeds_per_wavefront(tmp_path):
    src, exe = tmp_path / "waves.cc", tmp_path / "waves"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I", os.path.join(ROOT, "mkfit_amd", "csrc"), "-o",
                    str(exe), str(src)], check=True)
    subprocess.run([str(exe)], check=True, timeout=60)
