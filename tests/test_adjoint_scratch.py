"""The policy of the gradient's scratch (mkfit_amd/csrc/mkf_adjoint_scratch.h), compiled and run on the host."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = r"""
#include "mkf_adjoint_scratch.h"
#include <cassert>
#include <climits>
#include <cstdlib>

struct Device {                        // counts what the policy asks of the device, and refuses large allocations
  size_t largest = SIZE_MAX;
  int drains = 0, allocs = 0, frees = 0;
  int ready(AdjointScratch& s, const AdjointSize& z) {
    return adjoint_ready(s, z, [&](void* p) { ++drains; if (p) { ++frees; std::free(p); } return true; },
                         [&](size_t b) -> void* { ++allocs; return b > largest ? nullptr : std::malloc(1); });
  }
};
AdjointSize size(size_t n, int asked) {
  AdjointSize z;
  z.n = n; z.layers = 25; z.word = 4; z.sum_bytes = 256; z.asked = asked;
  return z;
}

int main() {
  {  // a call that the scratch holds at the caller's spacing leaves it where it is, however much more it could use
    AdjointScratch s;
    Device d;
    assert(d.ready(s, size(20000, 5)) == 1 && s.bytes == size(20000, 5).bytes(1));
    void* const p = s.p;
    const size_t held = s.bytes;
    const AdjointSize b = size(30000, 5);
    assert(b.need() <= held && b.bytes(1) > held);
    const int every = d.ready(s, b);
    assert(every > 1 && every <= 5 && b.bytes(every) <= held);
    assert(s.p == p && s.bytes == held && d.drains == 1 && d.allocs == 1);
    assert(d.ready(s, size(20000, 5)) == 1 && s.p == p);
  }
  {  // a refused growth is not tried again by a call that fits what was given
    AdjointScratch s;
    Device d;
    const AdjointSize z = size(100000, 5);
    d.largest = z.need();
    assert(d.ready(s, z) == 5 && s.bytes == z.need() && d.allocs == 2);
    assert(d.ready(s, z) == 5 && d.allocs == 2 && d.drains == 1 && d.frees == 0);
    d.largest = 0;                     // nothing to be had: the scratch is empty, the next smaller call starts over
    assert(d.ready(s, size(200000, 5)) == 0 && !s.p && s.bytes == 0);
    d.largest = SIZE_MAX;
    assert(d.ready(s, size(100, 5)) == 1);
  }
  {  // the limit: nothing beyond the caller's spacing, or as many states as fit
    AdjointScratch s;
    Device d;
    const AdjointSize z = size(100000, 5);
    s.limit = 0;
    assert(d.ready(s, z) == 5 && s.bytes == z.need());
    AdjointScratch t;
    t.limit = z.bytes(1) - 1;
    assert(d.ready(t, z) == 2 && t.bytes == t.limit);
    AdjointSize w = z;                 // another type, which the rest of the limit serves too
    w.word = 8;
    assert(w.need() <= t.bytes && d.ready(t, w) == 3 && t.bytes == t.limit);
    AdjointScratch u;                  // a need above the limit, at a spacing far beyond the layers
    u.limit = 1;
    assert(d.ready(u, size(100000, INT_MAX)) == 25 && u.bytes == size(100000, 25).need());
    assert(size(100000, INT_MAX).spacing(1) == INT_MAX);
    assert(size(1000, INT_MAX).spacing(SIZE_MAX) == 1);
  }
  return 0;
}
"""


def test_scratch_policy(tmp_path):
    src, exe = tmp_path / "policy.cc", tmp_path / "policy"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I", os.path.join(ROOT, "mkfit_amd", "csrc"),
                    "-include", "cstdint", "-o", str(exe), str(src)], check=True)
    subprocess.run([str(exe)], check=True, timeout=60)
