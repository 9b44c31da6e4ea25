// mkf_adjoint_scratch.h -- which states the gradient of the fit keeps, and the scratch a context holds for them.
// Host code without HIP, so that the policy runs (and is tested) on the CPU.
#pragma once

#include <algorithm>
#include <cstddef>

// A call's scratch: the sums' partials (sum_bytes, 256-byte aligned), checkpoints of 27 values, gradient rows.
struct AdjointSize {
  size_t n = 0, layers = 0, word = 4, sum_bytes = 0;
  int asked = 1;                       // the caller's checkpoint_every

  size_t bytes(int every) const {
    return sum_bytes + ((layers + every - 1) / every * 27 + layers * 3) * n * word;
  }
  size_t need() const { return bytes(asked); }
  // The spacing a call uses: one, so that the reverse sweep recomputes no state, when the scratch for it stays within
  // `limit`; else the shortest that does, and the caller's at most.  The gradient does not depend on it.  Recomputing
  // the states of five-layer segments is two of the seven forward steps' worth of work per layer (100k tracks, 25
  // layers: 804 us at a spacing of 5, 496 us at 1), while a state's store and load are 216 bytes.
  int spacing(size_t limit) const {
    if (need() > limit) return asked;
    int every = 1;
    while (bytes(every) > limit) ++every;
    return every;
  }
};

struct AdjointScratch {
  void* p = nullptr;
  size_t bytes = 0;
  size_t limit = (size_t)512 << 20;    // what a growing call may take beyond the caller's spacing
};

// Readies the scratch for a call and returns the spacing to run it at, 0 when the memory is not to be had.  A scratch
// that holds the call at the caller's spacing is left where it is, whatever more the call could use: its address may
// stand in a captured graph, and another stream may be in the middle of a capture that a drain would break.  Only a
// call that it cannot hold replaces it: by what it would use with every state kept, or by all of `limit` where that is
// less, so that a later call of another type or size finds it too; or by what the call needs, if that is more or all
// there is.
// drain_free(p): waits for the device, frees p, true on success; alloc(bytes): NULL on failure.
template <class DrainFree, class Alloc>
int adjoint_ready(AdjointScratch& s, const AdjointSize& z, DrainFree&& drain_free, Alloc&& alloc) {
  if (z.need() <= s.bytes) return z.spacing(s.bytes);
  if (!drain_free(s.p)) return 0;
  s.p = nullptr;
  s.bytes = 0;
  size_t take = std::max(z.need(), std::min(z.bytes(1), s.limit));
  s.p = alloc(take);
  if (!s.p && take > z.need()) s.p = alloc(take = z.need());
  if (!s.p) return 0;
  s.bytes = take;
  return z.spacing(take);
}
