// mkf_find.hip -- best-hit track finding on gfx950.
//
//   LayerOfHits build   k_row_partition -> k_row_sort (hits by q row, then each row in LDS) -> k_row_tiles ->
//                       k_row_units (rows that do not fit there), or, with a layer of millions of hits,
//                       k_hit_keys -> stable LSD radix sort (hipCUB) -> k_loh_gather, k_loh_fill
//   SelectHitIndices    k_select (per-operation entry point)
//   FindTracksBestHit   k_find_best_hit: one lane per seed carries its track
//                       through every layer with the state in VGPRs; hit
//                       selection, the chi2 of each candidate and the update
//                       are fused, so per layer only the bin table, the
//                       (phi, q) of scanned hits and the 9 floats of each
//                       candidate are read.
//
// Event layout in HBM (one event, all layers back to back in visiting order):
//   sorted hits   [total][9]  hits of every layer in LayerOfHits order
//   phis, qs      [total]     phi and q (z on barrel, r on endcaps) per sorted hit
//   ranks         [total]     sorted position -> hit index within its layer
//   inv           [total]     event hit index -> sorted position
//   bins          [sum nq*256] int2 {first, end} per (layer, q bin, phi bin),
//                             positions relative to the layer's first hit
// Every layer's rows start at its hit offset, so a lane addresses a layer
// with one scalar base and no per-layer allocations.
//
// Sort key: layer << 21 | q bin << 11 | fine phi bin.  Within one layer this is
// the order of the reference's key fine_phi + (q_bin << 16)
// (HitStructures.cc:114-128) because the fine phi bin is at most 1024; the
// layer bits keep layers apart so one sort over the event serves all layers,
// and LSD radix sort is stable like the reference's radix sort of the keys.
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <cmath>
#include <vector>

#include "../../include/mkfit_amd.h"
#include "mkf_internal.h"
#include "mkf_track_math.h"
#include "mkf_find_common.h"

using namespace mkf;
using namespace mkf_detail;
using namespace mkf_find;

namespace {

// Per-load hit offsets into the layer table, passed by value in chunks of
// kOffChunk layers (stream-ordered, no host staging buffer to keep alive).
constexpr int kOffChunk = 256;
struct OffsetsArg {
  int first, count;
  int off[kOffChunk + 1];
  int tile[kOffChunk + 1];      // first tile of k_row_partition per layer
};

// What k_row_sort puts off: the entries of the unit table and the histograms taken so far.
struct PutOff {
  int units, hists;
};

__global__ void k_set_offsets(OffsetsArg o, LayerDev* __restrict__ L, int* __restrict__ tile_off,
                              PutOff* __restrict__ put) {
  const int l = threadIdx.x;
  if (o.first == 0 && l == 0) *put = PutOff{0, 0};
  if (l < o.count) {
    L[o.first + l].hit_off = o.off[l];
    L[o.first + l].n_hits = o.off[l + 1] - o.off[l];
    tile_off[o.first + l] = o.tile[l];
    if (l + 1 == o.count) tile_off[o.first + o.count] = o.tile[o.count];
  }
}

__global__ void k_fill_i32(int* __restrict__ p, long n, int v) {
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) p[i] = v;
}

// Hit::r of an endcap hit (Hit.h:64-80); the FMA is written out so that every kernel forms the same bits.
__device__ __forceinline__ float hit_r(float x, float y) { return sqrtf(__builtin_fmaf(x, x, y * y)); }

// Hit::phi and Hit::z (barrel) / Hit::r (endcap) of a hit (Hit.h:64-80).  Not
// inlined: the key kernel and the fill kernel run this one piece of machine
// code, so the phi and q stored with a sorted hit are bit for bit the values
// its sort key was formed from.
__device__ __noinline__ float2 hit_phi_q(float x, float y, float z, int is_barrel) {
  return make_float2(atan2_cr(y, x), is_barrel ? z : hit_r(x, y));
}

// Layer owning event hit i: the last one in [lo, hi] whose hit range starts at
// or before it.
__device__ __forceinline__ int layer_of_hit(int i, int lo, int hi, const LayerDev* __restrict__ L) {
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (L[mid].hit_off <= i) lo = mid; else hi = mid - 1;
  }
  return lo;
}

// The sort key of every hit.  The block's first and last hits are located
// over all layers once; every thread then searches only the layers between.
__global__ void __launch_bounds__(256)
k_hit_keys(int total, int n_layers, const float* __restrict__ hits, const LayerDev* __restrict__ L,
           uint32_t* __restrict__ keys, int* __restrict__ vals) {
  __shared__ int span[2];
  const int i0 = blockIdx.x * blockDim.x;
  if (threadIdx.x < 2) {
    const int e = threadIdx.x == 0 ? i0 : min(i0 + (int)blockDim.x, total) - 1;
    span[threadIdx.x] = layer_of_hit(e, 0, n_layers - 1, L);
  }
  __syncthreads();
  const int i = i0 + threadIdx.x;
  if (i >= total) return;
  const int lo = layer_of_hit(i, span[0], span[1], L);
  const LayerDev& d = L[lo];
  const float2 pq = hit_phi_q(hits[(size_t)i * 9 + 0], hits[(size_t)i * 9 + 1], hits[(size_t)i * 9 + 2], d.is_barrel);
  const int qb = q_bin_checked(d, pq.y);
  const int pf = phi_bin_fine(pq.x);
  keys[i] = ((uint32_t)lo << kLayerShift) | ((uint32_t)qb << kQShift) | (uint32_t)pf;
  vals[i] = i;
}

// Sorted copies (HitStructures.cc:130-183), 256 sorted positions per block: the
// block's 2304 hit floats are read in 9 rounds in which consecutive lanes read
// consecutive floats of each hit (one random 36-byte run per hit rather than
// three random vector loads per lane), staged in LDS and written out
// contiguously; then each thread forms its hit's phi and q through the key
// kernel's function.  In XCD-major block order each XCD gathers from its own
// few layers (3.65 -> 3.43 ms over 141.7M hits).
__global__ void __launch_bounds__(256)
k_loh_gather(int total, const uint32_t* __restrict__ keys_s, const int* __restrict__ vals_s,
             const LayerDev* __restrict__ L, const float* __restrict__ hits, float* __restrict__ shits,
             float* __restrict__ phis, float* __restrict__ qs) {
  __shared__ float sh[256 * 9];
  __shared__ int sj[256];
  const int t = threadIdx.x;
  const int i0 = xcd_major_block() * 256;
  const int n = min(256, total - i0);
  sj[t] = t < n ? vals_s[i0 + t] : 0;
  __syncthreads();
  for (int f = t; f < n * 9; f += 256) {
    const int h = f / 9;
    sh[f] = hits[(size_t)sj[h] * 9 + (f - h * 9)];
  }
  __syncthreads();
  for (int f = t; f < n * 9; f += 256) shits[(size_t)i0 * 9 + f] = sh[f];
  if (t < n) {
    const int i = i0 + t;
    const LayerDev& d = L[keys_s[i] >> kLayerShift];
    const float2 pq = hit_phi_q(sh[t * 9], sh[t * 9 + 1], sh[t * 9 + 2], d.is_barrel);
    phis[i] = pq.x;
    qs[i] = pq.y;
  }
}

// Ranks in the layer, the inverse map and bin ranges (HitStructures.cc:130-183).
// The fine phi bin 1024 (phi == +pi exactly) shares coarse bin 0 with the row's
// first bins but sorts last in the row; the reference's scan then overwrites
// that bin's range with the later run.  Pass 0 writes every other run, pass 1
// the 1024 runs, so the later run wins here as well.  (Writing the ranks and
// the inverse map from the gather kernel instead measured 0.35 ms slower over
// 141.7M hits.)  In XCD-major block order the scattered 4-byte inverse-map
// writes of a layer complete their lines in one L2 (1.7 -> 1.3 ms for pass 0
// over 141.7M hits).
__global__ void __launch_bounds__(256)
k_loh_fill(int total, int pass, const uint32_t* __restrict__ keys_s, const int* __restrict__ vals_s,
           const LayerDev* __restrict__ L, int* __restrict__ ranks, int* __restrict__ inv, int2* __restrict__ bins) {
  const int i = xcd_major_block() * blockDim.x + threadIdx.x;
  if (i >= total) return;
  const uint32_t key = keys_s[i];
  const LayerDev& d = L[key >> kLayerShift];
  const int local = i - d.hit_off;
  if (pass == 0) {
    const int j = vals_s[i];
    ranks[i] = j - d.hit_off;
    inv[j] = i;
  }
  const bool fine1024 = (key & 0x400u) != 0;
  if ((pass == 1) != fine1024) return;
  const uint32_t jq = key & ~3u;
  const bool first = i == 0 || (keys_s[i - 1] & ~3u) != jq;
  const bool last = i == total - 1 || (keys_s[i + 1] & ~3u) != jq;
  const int qb = (int)((key >> kQShift) & (kMaxQBins - 1));
  const int pb = (int)((key & 0x3ffu) >> 2);
  int2* row = bins + d.bin_off + qb * kNPhi;
  if (first) row[pb].x = local;
  if (last) row[pb].y = local + 1;
  if (pass == 1) return;
  // Empty bins 1..255 of a row hold {p, p}, p the position where their hits
  // would start, so bins b..b' (1 <= b <= b' <= 255) of a row span the sorted
  // positions [row[b].x, row[b'].y) and a window's run of them is read with
  // two loads.  Bin 0 is left out: the phi == +pi run may replace its range.
  const uint32_t rowkey = key >> kQShift;
  if (first && pb > 1 && (i == 0 || (keys_s[i - 1] >> kQShift) != rowkey))
    for (int b = 1; b < pb; ++b) row[b] = make_int2(local, local);
  if (last) {
    int nb = kNPhi;
    if (i + 1 < total) {
      const uint32_t nk = keys_s[i + 1];
      if ((nk >> kQShift) == rowkey && !(nk & 0x400u)) nb = (int)((nk & 0x3ffu) >> 2);
    }
    for (int b = max(pb + 1, 1); b < nb; ++b) row[b] = make_int2(local + 1, local + 1);
  }
}

// ---- LayerOfHits by q rows ---------------------------------------------------
// A layer's order is (q bin, fine phi bin, hit index), and its hits arrive in one
// run.  k_row_partition deals each tile of kTile hits of a layer into the layer's
// q rows in LDS and writes the tile's (phi, index) pairs row by row, with the
// tile's row starts; k_row_sort takes one row per block, collects its pairs from
// the layer's tiles, orders them in LDS by fine phi bin and index, and writes
// everything the finders read: the hits, phi, q, ranks, the inverse map and the
// row's bin ranges.  A hit moves 36 + 8 bytes in the first kernel and 8 + 36 + 52
// in the second, against 36 + 8, four radix passes of 16, 8 + 36 + 44 and 8 + 16
// for keys, sort, gather and fill.  Over 141.7M hits in 850 layers: 1.16 ms (5.4 TB/s) + 3.8 ms (23 GB moved, 15 of
// them read for 6: a gathered hit's 128-byte line is fetched for three or four rows, and a layer exceeds an XCD's
// L2) + 0.39 ms for the inverse map, against 10.6 ms.
constexpr int kTile = 3072;          // hits per tile; also the LDS capacity of k_row_sort, so one tile's part
constexpr int kRowCap = kTile;       // of a row always fits
constexpr int kPartBlock = 512, kRowBlock = 256;
constexpr int kUnitBlock = 512;
constexpr int kFineBins = 1025;      // fine phi bins 0..1024 (1024: phi == +pi)
// Hits of a fine bin ordered by comparing each with each; a row with a bin of more is put off (17 layers of 30k / 167k
// hits in bins of about 24 / 55 / 90 / 200, compared: 50 / 55 / 62 / 86 and 141 / 162 / 183 / 247 us, put off: 125 and 269).
constexpr int kBinMax = 256;
static_assert(kTile % kPartBlock == 0 && kRowCap % kRowBlock == 0 && kRowCap % kUnitBlock == 0 && kTile <= 4096,
              "tile size; a hit's place in its tile takes 12 bits");
// Hits of a row that one block orders, reading it once per run of bins that fits; a row of more is put off (17 layers of
// 167k hits, 4175 / 6958 / 11133 / 15308 a row, in runs: 174 / 216 / 282 / 473 us, put off: 334 / 296 / 267 / 269).
constexpr int kRowRuns = 3 * kRowCap;
// A load with a layer of more hits than this goes through the radix sort, because a put off row's units look into every
// tile of its layer (one layer, evenly filled / all in one q bin / radix sort: 0.5M hits 49 / 128 / 173 us, 1.05M 110 /
// 202 / 215, 2M 179 / 364 / 276).
constexpr size_t kRowLayerMax = (size_t)1 << 21;

// Beyond this many hits the sorted copies are stored past the caches: the 256 MB last-level cache no longer keeps
// them for the finder (best-hit step, stored past / through the caches: 562 / 516 us at 2.8M hits, 723 / 742 at
// 5.7M, 1517 / 1559 at 22.7M).
constexpr size_t kStreamHits = 4000000;

constexpr int kRowWeight = 100;      // a row's fixed cost in hits, for the XCDs' shares

struct RowPair {
  float phi;
  int idx;      // hit index in its layer
};

// A row that k_row_sort does not order -- of more than kRowRuns hits, or with a crowded fine bin -- is put off:
// k_row_tiles orders the row's part of each tile by fine bin and index and counts the row's bins (`hist`), and
// k_row_units writes the row, kRowCap positions per block.  What each block takes is found by searching the parts, so
// the work is linear in the row but for a few probes per unit and tile, in any distribution over q and phi (17 layers of
// 167k hits, us, with one block per row in runs, and now: one layer 80 % in two q bins 2854 / 188, all in two bins
// 6080 / 263; 400k hits in one bin 106004 / 115, in one fine bin 211980 / 82; radix sort 300, 304, 170, 152; evenly
// filled rows of 11133 / 27833 / 83500 hits, put off and radix sort: 267 / 267 / 263 and 304 / 297 / 298).
struct RowUnit {
  int row, start, n;      // the q row, its first position in the layer, its hits
  int first;              // the unit's first position in the row
  int hist;               // the row's histogram, or -1: the unit is the whole row
};
constexpr int kRowPutOff = -2;       // in row_hist: put off without a histogram; -1: not put off
// A histogram is kept in parts that tiles add to in turn, because additions to one cache line go one after the other.
constexpr int kHistParts = 4, kHistWords = kHistParts * (kFineBins + 1);

__device__ __forceinline__ int fine_bin_clamped(float phi) {
  return min(max(phi_bin_fine(phi), 0), kFineBins - 1);
}

// Exclusive prefix sum of v over the block's threads; *total gets the sum.  `part` holds a word per wavefront.
template <int BLOCK>
__device__ __forceinline__ int block_exclusive(int v, int* part, int* total) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int incl = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int u = __shfl_up(incl, o, 64);
    if (lane >= o) incl += u;
  }
  if (lane == 63) part[wave] = incl;
  __syncthreads();
  int before = 0, sum = 0;
#pragma unroll
  for (int w = 0; w < BLOCK / 64; ++w) {
    const int p = part[w];
    before += w < wave ? p : 0;
    sum += p;
  }
  __syncthreads();
  *total = sum;
  return before + incl - v;
}

// The layer holding a hit tile: the last of the layers whose first tile is at or before it, found by a
// wavefront in two steps of 64 lanes (of MKF_MAX_EOH_LAYERS = 64 * 32 layers).
__device__ __forceinline__ int layer_of_tile(int tile, int n_layers, const int* __restrict__ tile_off) {
  constexpr int kStep = MKF_MAX_EOH_LAYERS / 64;
  const int lane = threadIdx.x & 63;
  const int c = lane * kStep;
  const int coarse = __popcll(__ballot(c < n_layers && tile_off[min(c, n_layers)] <= tile)) - 1;
  const int l = coarse * kStep + lane;
  const int fine = __popcll(__ballot(lane < kStep && l < n_layers && tile_off[min(l, n_layers)] <= tile)) - 1;
  return coarse * kStep + fine;
}

__global__ void __launch_bounds__(kPartBlock)
k_row_partition(int n_layers, const int* __restrict__ tile_off, const LayerDev* __restrict__ L,
                const float* __restrict__ hits, RowPair* __restrict__ pairs, unsigned short* __restrict__ pre,
                int pre_stride) {
  __shared__ RowPair out[kTile];
  __shared__ int hist[kMaxQBins];
  __shared__ int part[kPartBlock / 64];
  __shared__ int s_layer;
  const int t = threadIdx.x, tile = blockIdx.x;
  if (t < 64) {
    const int l = layer_of_tile(tile, n_layers, tile_off);
    if (t == 0) s_layer = l;
  }
  for (int q = t; q < kMaxQBins; q += kPartBlock) hist[q] = 0;
  __syncthreads();
  const LayerDev& d = L[s_layer];
  const int first = (tile - tile_off[s_layer]) * kTile;       // in the layer
  const int n = min(kTile, d.n_hits - first);
  const float* __restrict__ src = hits + (size_t)(d.hit_off + first) * 9;
  constexpr int kPer = kTile / kPartBlock;
  float x[kPer], y[kPer], z[kPer];
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const int j = min(t + k * kPartBlock, n - 1);
    x[k] = src[(size_t)j * 9];
    y[k] = src[(size_t)j * 9 + 1];
    z[k] = src[(size_t)j * 9 + 2];
  }
  const bool barrel = d.is_barrel != 0;
  int qb[kPer], rank[kPer];
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    if (t + k * kPartBlock < n) {
      qb[k] = q_bin_checked(d, barrel ? z[k] : hit_r(x[k], y[k]));
      rank[k] = atomicAdd(&hist[qb[k]], 1);
    }
  }
  __syncthreads();
  // row starts within the tile
  static_assert(kMaxQBins == 2 * kPartBlock, "two rows per thread");
  const int h0 = hist[2 * t], h1 = hist[2 * t + 1];
  int total;
  const int e0 = block_exclusive<kPartBlock>(h0 + h1, part, &total);
  hist[2 * t] = e0;
  hist[2 * t + 1] = e0 + h0;
  unsigned short* __restrict__ row = pre + (size_t)tile * pre_stride;
  if (2 * t <= d.nq) row[2 * t] = (unsigned short)e0;
  if (2 * t + 1 <= d.nq) row[2 * t + 1] = (unsigned short)(e0 + h0);
  if (t == 0 && d.nq == kMaxQBins) row[kMaxQBins] = (unsigned short)n;
  __syncthreads();
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const int j = t + k * kPartBlock;
    if (j < n) out[hist[qb[k]] + rank[k]] = RowPair{atan2_cr(y[k], x[k]), first + j};
  }
  __syncthreads();
  RowPair* __restrict__ dst = pairs + d.hit_off + first;
  for (int j = t; j < n; j += kPartBlock) dst[j] = out[j];
}

// The rows each XCD takes, contiguous so that its L2 keeps the layers it gathers from, and of equal shares of the
// hits (equal numbers of rows gave the XCD of the outermost layers of one event twice the hits of the first: best-hit
// step 335 us, against 321 us with the rows dealt out singly and 310 us with equal shares; 50 events 7.21, 7.73 and
// 7.13 ms).
struct XcdRows {
  int first[9];
};

// cur (LDS): counts of the fine bins to their starts.
template <int BLOCK>
__device__ __forceinline__ void scan_bins(int* cur, int* part, int* crowded) {
  constexpr int kPer = (kFineBins + BLOCK) / BLOCK;
  int h[kPer], sum = 0;
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const int b = threadIdx.x * kPer + k;
    h[k] = b <= kFineBins ? cur[b] : 0;
    sum += h[k];
    if (crowded && h[k] > kBinMax) *crowded = 1;
  }
  int total;
  int e = block_exclusive<BLOCK>(sum, part, &total);
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const int b = threadIdx.x * kPer + k;
    if (b <= kFineBins) cur[b] = e;
    e += h[k];
  }
  __syncthreads();
}

template <bool NT>
__device__ __forceinline__ void put_out(float* p, float v) {
  if (NT) __builtin_nontemporal_store(v, p);
  else *p = v;
}

// The m hits listed in order in s_idx (LDS) to sorted positions g0..
template <int BLOCK, bool NT>
__device__ __forceinline__ void write_hits(const int* s_idx, int m, int g0, bool barrel, const float* __restrict__ lhits,
                                           float* __restrict__ shits, float* __restrict__ qs, int* __restrict__ ranks) {
  struct F3 { float a, b, c; };
  constexpr int kBatch = 6;
  for (int f0 = threadIdx.x; f0 < m * 3; f0 += BLOCK * kBatch) {
    F3 v[kBatch];
#pragma unroll
    for (int u = 0; u < kBatch; ++u) {
      const int f = min(f0 + u * BLOCK, m * 3 - 1), h = f / 3;
      __builtin_memcpy(&v[u], lhits + (size_t)s_idx[h] * 9 + (f - h * 3) * 3, 12);
    }
#pragma unroll
    for (int u = 0; u < kBatch; ++u) {
      const int f = f0 + u * BLOCK, h = f / 3;
      if (f < m * 3) {
        float* o = shits + (size_t)g0 * 9 + (size_t)f * 3;
        put_out<NT>(o, v[u].a);
        put_out<NT>(o + 1, v[u].b);
        put_out<NT>(o + 2, v[u].c);
        if (f == h * 3) put_out<NT>(qs + g0 + h, barrel ? v[u].c : hit_r(v[u].a, v[u].b));
      }
    }
  }
  for (int h = threadIdx.x; h < m; h += BLOCK) ranks[g0 + h] = s_idx[h];
}

// Range of coarse bin b of a row of n hits at position `start`, its places lo .. hi of the row, `regular` hits below
// phi = +pi (HitStructures.cc:146-171), as k_loh_fill's two passes leave it: an empty bin 1..255 of a row with hits
// below phi = +pi holds its insertion point, and the phi = +pi run takes over bin 0.
__device__ __forceinline__ int2 bin_range(int b, int lo, int hi, int regular, int start, int n) {
  int2 r = make_int2(start + lo, start + hi);
  if (regular == 0 || (b == 0 && hi == 0)) r = make_int2(0, 0);
  if (b == 0 && n > regular) r = make_int2(start + regular, start + n);
  return r;
}

// One q row per block; see above.  The pairs of a row come in any order within a
// tile's part, so the order inside a fine phi bin (one to three hits) is set by
// comparing indices.  A row that fits the LDS is read once; what it reads from
// memory is issued in batches, as the block waits on memory for most of its time.
// Rows beyond the LDS capacity (or of layers with more tiles than threads) go
// through it in runs of whole fine bins.
template <bool NT>
__global__ void __launch_bounds__(kRowBlock)
k_row_sort(XcdRows xr, const int* __restrict__ row_layer, const LayerDev* __restrict__ L, const int* __restrict__ tile_off,
           const unsigned short* __restrict__ pre, int pre_stride, const RowPair* __restrict__ pairs,
           const float* __restrict__ hits, float* __restrict__ shits, float* __restrict__ phis,
           float* __restrict__ qs, int* __restrict__ ranks, int* __restrict__ place, int2* __restrict__ bins,
           PutOff* __restrict__ put, int* __restrict__ row_hist, int* __restrict__ hist, RowUnit* __restrict__ units) {
  __shared__ int s_idx[kRowCap];
  __shared__ int cur[kFineBins + 1];     // fine bin starts, then (as cursors) the ends of the bins placed so far
  __shared__ int s_seg[kRowBlock];       // each tile's part: first place in the tile << 16 | length
  __shared__ int s_dst[kRowBlock];       // and the place of its first pair among the row's
  __shared__ int part[kRowBlock / 64];
  __shared__ int s_crowded, s_unit, s_hist, s_b1;
  const int t = threadIdx.x;
  const int row = xr.first[blockIdx.x % 8] + blockIdx.x / 8;
  if (row >= xr.first[blockIdx.x % 8 + 1]) return;
  const int layer = row_layer[row];
  const LayerDev& d = L[layer];
  const int q = row - d.bin_off / kNPhi;
  const int nt = (d.n_hits + kTile - 1) / kTile;
  const unsigned short* __restrict__ rp = pre + (size_t)tile_off[layer] * pre_stride + q;
  const RowPair* __restrict__ src = pairs + d.hit_off;
  int* __restrict__ lplace = place + d.hit_off;
  const float* __restrict__ lhits = hits + (size_t)d.hit_off * 9;
  for (int b = t; b <= kFineBins; b += kRowBlock) cur[b] = 0;
  if (t == 0) s_crowded = 0;
  int c = 0, before = 0;
  for (int i = t; i < nt; i += kRowBlock) {
    const int a = rp[(size_t)i * pre_stride], len = rp[(size_t)i * pre_stride + 1] - a;
    before += a;
    c += len;
    s_seg[t] = a << 16 | len;
  }
  int n, start;                          // hits of the row, its first position in the layer
  s_dst[t] = block_exclusive<kRowBlock>(c, part, &n);
  block_exclusive<kRowBlock>(before, part, &start);
  if (n == 0) {
    bins[d.bin_off + q * kNPhi + t] = make_int2(0, 0);
    if (t == 0) row_hist[row] = -1;
    return;
  }
  auto put_off = [&]() {
    const int m = (n + kRowCap - 1) / kRowCap;
    if (t == 0) {
      s_unit = atomicAdd(&put->units, m);
      s_hist = m > 1 ? atomicAdd(&put->hists, 1) : -1;
      row_hist[row] = m > 1 ? s_hist : kRowPutOff;
    }
    __syncthreads();
    for (int i = t; i < m; i += kRowBlock) units[s_unit + i] = RowUnit{row, start, n, i * kRowCap, s_hist};
    if (m > 1)
      for (int b = t; b < kHistWords; b += kRowBlock) hist[(size_t)s_hist * kHistWords + b] = 0;
  };
  if (n > kRowRuns) {
    put_off();
    return;
  }
  const int gbase = d.hit_off + start;
  if (n <= kRowCap && nt <= kRowBlock) {
    // the positions of the row's pairs, 32 lanes per tile's part
    constexpr int kGroups = kRowBlock / 32;
    for (int i = t >> 5; i < nt; i += kGroups) {
      const int seg = s_seg[i], len = seg & 0xffff, dst = s_dst[i], from = i * kTile + (seg >> 16);
      for (int j = t & 31; j < len; j += 32) s_idx[dst + j] = from + j;
    }
    __syncthreads();
    constexpr int kPer = kRowCap / kRowBlock;
    RowPair pr[kPer];
    int at[kPer];                          // fine bin << 16 | place in it; then the place in the row
#pragma unroll
    for (int k = 0; k < kPer; ++k)
      if (t + k * kRowBlock < n) pr[k] = src[s_idx[t + k * kRowBlock]];
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
      if (t + k * kRowBlock < n) {
        const int b = fine_bin_clamped(pr[k].phi);
        at[k] = b << 16 | atomicAdd(&cur[b], 1);
      }
    }
    __syncthreads();
    scan_bins<kRowBlock>(cur, part, &s_crowded);
    if (s_crowded) {
      put_off();
      return;
    }
    if (t == 0) row_hist[row] = -1;
    int at0[kPer];                         // the pairs' positions, kept to write their places there
#pragma unroll
    for (int k = 0; k < kPer; ++k) at0[k] = t + k * kRowBlock < n ? s_idx[t + k * kRowBlock] : 0;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kPer; ++k)
      if (t + k * kRowBlock < n) s_idx[cur[at[k] >> 16] + (at[k] & 0xffff)] = pr[k].idx;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
      if (t + k * kRowBlock < n) {
        const int lo = cur[at[k] >> 16], hi = cur[(at[k] >> 16) + 1];
        int p = lo;
        for (int i = lo; i < hi; ++i) p += s_idx[i] < pr[k].idx;
        at[k] = p;
        lplace[at0[k]] = gbase + p;
      }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kPer; ++k)
      if (t + k * kRowBlock < n) s_idx[at[k]] = pr[k].idx;
    __syncthreads();
    write_hits<kRowBlock, NT>(s_idx, n, gbase, d.is_barrel != 0, lhits, shits, qs, ranks);
    __syncthreads();
    float* s_phi = reinterpret_cast<float*>(s_idx);
#pragma unroll
    for (int k = 0; k < kPer; ++k)
      if (t + k * kRowBlock < n) s_phi[at[k]] = pr[k].phi;
    __syncthreads();
    for (int h = t; h < n; h += kRowBlock) put_out<NT>(phis + gbase + h, s_phi[h]);
    bins[d.bin_off + q * kNPhi + t] = bin_range(t, cur[4 * t], cur[4 * t + 4], cur[1024], start, n);
    return;
  }
  // every pair of the row, 16 lanes per tile's part: f(pair, its position)
  auto each_pair = [&](auto&& f) {
    for (int i = t >> 4; i < nt; i += kRowBlock / 16) {
      const int lo = rp[(size_t)i * pre_stride], hi = rp[(size_t)i * pre_stride + 1];
      for (int j = lo + (t & 15); j < hi; j += 16) f(src[i * kTile + j], i * kTile + j);
    }
  };
  each_pair([&](const RowPair& p, int) { atomicAdd(&cur[fine_bin_clamped(p.phi)], 1); });
  __syncthreads();
  scan_bins<kRowBlock>(cur, part, &s_crowded);
  if (s_crowded) {
    put_off();
    return;
  }
  if (t == 0) row_hist[row] = -1;
  // Puts each of the m entries (s_idx: the pairs' positions), whose equal-bin group lies at [x, y) = group(phi), at
  // its place by index, from row position `base` on; then s_idx holds hit indices.
  auto order = [&](int base, int m, auto&& group) {
    constexpr int kPer = kRowCap / kRowBlock;
    RowPair pr[kPer];
    int at[kPer], pos[kPer];
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
      if (t + k * kRowBlock < m) {
        at[k] = s_idx[t + k * kRowBlock];
        pr[k] = src[at[k]];
      }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kPer; ++k)
      if (t + k * kRowBlock < m) s_idx[t + k * kRowBlock] = pr[k].idx;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
      if (t + k * kRowBlock < m) {
        const int2 r = group(pr[k].phi);
        int p = r.x;
        for (int i = r.x; i < r.y; ++i) p += s_idx[i] < pr[k].idx;
        pos[k] = p;
        lplace[at[k]] = gbase + base + p;
        phis[gbase + base + p] = pr[k].phi;
      }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kPer; ++k)
      if (t + k * kRowBlock < m) s_idx[pos[k]] = pr[k].idx;
    __syncthreads();
  };
  for (int b0 = 0; b0 < kFineBins;) {
    const int base = cur[b0];
    // the longest run of bins from b0 that fits
    if (t == 0) s_b1 = b0;
    __syncthreads();
    for (int b = b0 + 1 + t; b <= kFineBins; b += kRowBlock)
      if (cur[b] - base <= kRowCap) atomicMax(&s_b1, b);
    __syncthreads();
    const int b1 = s_b1;                 // past b0: a bin holds at most kBinMax
    const int m = cur[b1] - base;        // cur[kFineBins] == n
    __syncthreads();
    each_pair([&](const RowPair& p, int at) {
      const int b = fine_bin_clamped(p.phi);
      if (b >= b0 && b < b1) s_idx[atomicAdd(&cur[b], 1) - base] = at;
    });
    __syncthreads();
    order(base, m, [&](float phi) {
      const int b = fine_bin_clamped(phi);
      return make_int2((b > b0 ? cur[b - 1] : base) - base, cur[b] - base);
    });
    write_hits<kRowBlock, NT>(s_idx, m, gbase + base, d.is_barrel != 0, lhits, shits, qs, ranks);
    b0 = b1;
    __syncthreads();
  }
  // the cursors stand at the bins' ends
  const int c0 = t > 0 ? cur[4 * t - 1] : 0, c1 = cur[4 * t + 3], regular = cur[1023];
  bins[d.bin_off + q * kNPhi + t] = bin_range(t, c0, c1, regular, start, n);
}

// Place of element i of an array being sorted in LDS: a word of padding after every eight, so that lanes' elements a
// power of two apart lie in different banks.
constexpr int kSortWords = 4096 + 4096 / 8;
__device__ __forceinline__ int padded(int i) { return i + (i >> 3); }

// Bitonic sort steps of strides s << (E - 1) .. s on the 2^E elements of a thread, in the direction of level k (the
// elements' complements ascend where the elements descend).  WHOLE: s is a multiple of eight.
template <int BLOCK, int E, bool WHOLE>
__device__ __forceinline__ void bitonic_trip(unsigned* v, int size, int k, int s) {
  constexpr int kN = 1 << E;
  for (int i = threadIdx.x; i < size / kN; i += BLOCK) {
    const int at = (i & ~(s - 1)) * kN + (i & (s - 1)), first = padded(at);
    const unsigned flip = (at & k) == 0 ? 0u : ~0u;
    auto element = [&](int e) -> unsigned& { return v[WHOLE ? first + e * (s + (s >> 3)) : padded(at + e * s)]; };
    unsigned x[kN];
#pragma unroll
    for (int e = 0; e < kN; ++e) x[e] = element(e) ^ flip;
#pragma unroll
    for (int j = kN / 2; j > 0; j /= 2) {
#pragma unroll
      for (int e = 0; e < kN; ++e) {
        if (e & j) continue;
        const unsigned lo = min(x[e], x[e + j]), hi = max(x[e], x[e + j]);
        x[e] = lo;
        x[e + j] = hi;
      }
    }
#pragma unroll
    for (int e = 0; e < kN; ++e) element(e) = x[e] ^ flip;
  }
  __syncthreads();
}

// Ascending sort of `size` padded elements in LDS, size a power of two: up to three strides per trip through the LDS,
// 32 trips and barriers for 4096 elements in place of the 78 of one stride each.
template <int BLOCK>
__device__ __forceinline__ void bitonic_sort(unsigned* v, int size) {
  for (int k = 2; k <= size; k *= 2) {
    for (int j = k / 2; j > 0;) {
      if (j >= 32) bitonic_trip<BLOCK, 3, true>(v, size, k, j / 4);
      else if (j >= 4) bitonic_trip<BLOCK, 3, false>(v, size, k, j / 4);
      else if (j == 2) bitonic_trip<BLOCK, 2, false>(v, size, k, 1);
      else bitonic_trip<BLOCK, 1, false>(v, size, k, 1);
      j = j >= 4 ? j / 8 : 0;
    }
  }
}
__device__ __forceinline__ int pow2_at_least(int n) { return n <= 1 ? 1 : 1 << (32 - __clz(n - 1)); }

// Per tile: the inverse map of its hits from their pairs' places, turned into hit order in LDS (scattering it from
// k_row_sort writes a 32-byte sector per 4-byte entry: 1.0 ms over 141.7M hits, against 0.1 ms there for the
// places and this kernel).  Then, where rows were put off, their parts in this tile are ordered by fine bin and index,
// in place, and their bins counted; k_row_units writes those hits' inverse map again.
__global__ void __launch_bounds__(kPartBlock) __attribute__((amdgpu_waves_per_eu(8)))
k_row_tiles(int n_layers, const int* __restrict__ tile_off, const LayerDev* __restrict__ L, RowPair* __restrict__ pairs,
            const int* __restrict__ place, int* __restrict__ inv, const unsigned short* __restrict__ pre, int pre_stride,
            const PutOff* __restrict__ put, const int* __restrict__ row_hist, int* __restrict__ hist) {
  __shared__ unsigned key[kSortWords];
  __shared__ unsigned short s_at[kTile];             // hit of the tile -> its pair's position
  __shared__ unsigned short s_row[kMaxQBins + 1];
  __shared__ int s_hist[kMaxQBins];
  __shared__ int s_lo, s_hi;
  int* out = reinterpret_cast<int*>(key);
  const int t = threadIdx.x, tile = blockIdx.x;
  const int l = layer_of_tile(tile, n_layers, tile_off);
  const LayerDev& d = L[l];
  const int first = (tile - tile_off[l]) * kTile;
  const int n = min(kTile, d.n_hits - first), g0 = d.hit_off + first;
  constexpr int kPer = kTile / kPartBlock;
  int idx[kPer], p[kPer];
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const int j = g0 + min(t + k * kPartBlock, n - 1);
    idx[k] = pairs[j].idx;
    p[k] = place[j];
  }
#pragma unroll
  for (int k = 0; k < kPer; ++k)
    if (t + k * kPartBlock < n) out[idx[k] - first] = p[k];
  __syncthreads();
  for (int j = t; j < n; j += kPartBlock) inv[g0 + j] = out[j];
  if (put->units == 0) return;
  for (int q = t; q <= d.nq; q += kPartBlock) {
    s_row[q] = pre[(size_t)tile * pre_stride + q];
    if (q < d.nq) s_hist[q] = row_hist[d.bin_off / kNPhi + q];
  }
  // Key: q bin (of half of them at a time), then fine bin and hit of a pair to order, or position of one that stays.
  constexpr int kQHalf = 512;
  static_assert(2 * kQHalf == kMaxQBins, "9 bits of a key hold half of the q bins");
  for (int q0 = 0; q0 < d.nq; q0 += kQHalf) {
    const int q1 = min(q0 + kQHalf, d.nq);
    __syncthreads();
    if (t == 0) {
      s_lo = n;
      s_hi = 0;
    }
    __syncthreads();
    // the span from the first put off row's part to the last's
    for (int q = q0 + t; q < q1; q += kPartBlock) {
      if (s_hist[q] != -1 && s_row[q + 1] > s_row[q]) {
        atomicMin(&s_lo, (int)s_row[q]);
        atomicMax(&s_hi, (int)s_row[q + 1]);
      }
    }
    __syncthreads();
    const int lo = s_lo, m = s_hi - lo;
    if (m <= 0) continue;
    const int size = pow2_at_least(m);
    RowPair* __restrict__ src = pairs + g0 + lo;
    RowPair pr[kPer];
#pragma unroll
    for (int k = 0; k < kPer; ++k) pr[k] = src[min(t + k * kPartBlock, m - 1)];
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
      const int j = t + k * kPartBlock;
      if (j >= m) continue;
      int a = q0;                                // the last row that starts at or before the position
#pragma unroll
      for (int step = kQHalf / 2; step > 0; step /= 2)
        if (a + step < q1 && s_row[a + step] <= lo + j) a += step;
      unsigned in = j;
      if (s_hist[a] != -1) {
        in = (unsigned)fine_bin_clamped(pr[k].phi) << 12 | (unsigned)(pr[k].idx - first);
        s_at[pr[k].idx - first] = (unsigned short)j;
      }
      key[padded(j)] = (unsigned)(a - q0) << 23 | in;
    }
    for (int j = m + t; j < size; j += kPartBlock) key[padded(j)] = ~0u;
    __syncthreads();
    bitonic_sort<kPartBlock>(key, size);
    int t1 = t;
    asm volatile("" : "+v"(t1));          // the addresses are formed anew, not kept in registers during the sort
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
      const int j = t1 + k * kPartBlock;
      if (j < m && s_hist[q0 + (int)(key[padded(j)] >> 23)] != -1) pr[k] = src[s_at[key[padded(j)] & 0xfff]];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
      const int j = t1 + k * kPartBlock;
      if (j >= m) continue;
      const unsigned v = key[padded(j)] >> 12;           // q bin and fine bin
      const int h = s_hist[q0 + (int)(v >> 11)];
      if (h == -1) continue;
      src[j] = pr[k];
      if (h < 0) continue;
      // a run of equal bins adds its length
      const bool first_of = j == 0 || key[padded(j - 1)] >> 12 != v, last_of = j + 1 == m || key[padded(j + 1)] >> 12 != v;
      const int add = (last_of ? j + 1 : 0) - (first_of ? j : 0);
      if (add) atomicAdd(&hist[(size_t)h * kHistWords + tile % kHistParts * (kFineBins + 1) + (int)(v & 0x7ff)], add);
    }
  }
}

// A put off row's positions first .. first + kRowCap.  Its tiles' parts are ordered by fine bin and index, and tiles
// follow each other by index, so the position of a part's first pair of a bin is the bin's start plus the bin's pairs
// in the tiles before: with those of the unit's first and last bin every tile's share of the unit is known.  Ordering
// the shares, tile by tile in the list, by bin and place in the list gives the row's order.  Each XCD takes a contiguous
// eighth of the units, so that units of a row, whose hits share lines, share an L2.
template <bool NT>
__global__ void __launch_bounds__(kUnitBlock)
k_row_units(const PutOff* __restrict__ put, const RowUnit* __restrict__ units, const int* __restrict__ hist,
            const int* __restrict__ row_layer, const LayerDev* __restrict__ L, const int* __restrict__ tile_off,
            const unsigned short* __restrict__ pre, int pre_stride, const RowPair* __restrict__ pairs,
            const float* __restrict__ hits, float* __restrict__ shits, float* __restrict__ phis, float* __restrict__ qs,
            int* __restrict__ ranks, int* __restrict__ inv, int2* __restrict__ bins) {
  __shared__ unsigned key[kSortWords];   // fine bin << 12 | place in the list; then the hits in order
  __shared__ int s_pos[kRowCap];         // the list: the pairs' positions
  __shared__ int cur[kFineBins + 1];     // the row's fine bin starts
  __shared__ int s_from[kUnitBlock], s_len[kUnitBlock], s_dst[kUnitBlock];
  __shared__ int part[kUnitBlock / 64];
  __shared__ int s_b0, s_b1;
  const int t = threadIdx.x, n_units = put->units;
  const int share = (n_units + 7) / 8, u1 = min(n_units, (int)(blockIdx.x % 8 + 1) * share);
  for (int u = blockIdx.x % 8 * share + blockIdx.x / 8; u < u1; u += gridDim.x / 8) {
    const RowUnit w = units[u];
    const int layer = row_layer[w.row];
    const LayerDev& d = L[layer];
    const int q = w.row - d.bin_off / kNPhi;
    const int nt = (d.n_hits + kTile - 1) / kTile;
    const unsigned short* __restrict__ rp = pre + (size_t)tile_off[layer] * pre_stride + q;
    const RowPair* __restrict__ src = pairs + d.hit_off;
    const int p0 = w.first, p1 = min(w.n, p0 + kRowCap), m = p1 - p0;
    const bool whole = w.hist < 0;
    __syncthreads();                     // the LDS of the unit before is read
    for (int b = t; b <= kFineBins; b += kUnitBlock) {
      int sum = 0;
      for (int c = 0; c < kHistParts && !whole; ++c) sum += hist[(size_t)w.hist * kHistWords + c * (kFineBins + 1) + b];
      cur[b] = sum;
    }
    __syncthreads();
    int b0 = 0, b1 = 0;
    if (!whole) {
      scan_bins<kUnitBlock>(cur, part, nullptr);
      for (int b = t; b < kFineBins; b += kUnitBlock) {
        if (cur[b] <= p0 && p0 < cur[b + 1]) s_b0 = b;
        if (cur[b] < p1 && p1 <= cur[b + 1]) s_b1 = b;
      }
      __syncthreads();
      b0 = s_b0;
      b1 = s_b1;
    }
    int done0 = 0, done1 = 0, listed = 0;        // pairs of bins b0 and b1 in the tiles before; pairs in the list
    for (int i0 = 0; i0 < nt; i0 += kUnitBlock) {
      const int i = i0 + t;
      int from = 0, to = 0;
      if (i < nt) {
        from = i * kTile + rp[(size_t)i * pre_stride];
        to = i * kTile + rp[(size_t)i * pre_stride + 1];
      }
      if (!whole) {
        // the part's first pair at or past bins b0, b0 + 1, b1, b1 + 1
        int at[4] = {from, from, from, from};
        for (int step = pow2_at_least(to - from + 1); step > 0; step >>= 1) {
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            const int b = k < 2 ? b0 + k : b1 + k - 2;
            if (at[k] + step <= to && fine_bin_clamped(src[at[k] + step - 1].phi) < b) at[k] += step;
          }
        }
        int all;
        const int g0 = cur[b0] + done0 + block_exclusive<kUnitBlock>(at[1] - at[0], part, &all);
        done0 += all;
        const int g1 = cur[b1] + done1 + block_exclusive<kUnitBlock>(at[3] - at[2], part, &all);
        done1 += all;
        from = at[0] + min(max(p0 - g0, 0), at[1] - at[0]);
        to = at[2] + min(max(p1 - g1, 0), at[3] - at[2]);
      }
      int all;
      const int dst = listed + block_exclusive<kUnitBlock>(to - from, part, &all);
      listed += all;
      s_from[t] = from;
      s_len[t] = to - from;
      s_dst[t] = dst;
      __syncthreads();
      for (int k = t >> 5; k < min(kUnitBlock, nt - i0); k += kUnitBlock / 32)
        for (int j = t & 31; j < s_len[k]; j += 32) s_pos[s_dst[k] + j] = s_from[k] + j;
      __syncthreads();
    }
    const int size = b0 == b1 && !whole ? 0 : pow2_at_least(m);
    constexpr int kPer = kRowCap / kUnitBlock;
    RowPair pr[kPer];
    if (size) {
#pragma unroll
      for (int k = 0; k < kPer; ++k) pr[k] = src[s_pos[min(t + k * kUnitBlock, m - 1)]];
    }
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
      const int j = t + k * kUnitBlock;
      if (j >= m) continue;
      const int b = size ? fine_bin_clamped(pr[k].phi) : 0;
      if (whole) atomicAdd(&cur[b], 1);
      key[padded(j)] = (unsigned)(b << 12 | j);
    }
    for (int j = m + t; j < size; j += kUnitBlock) key[padded(j)] = ~0u;
    __syncthreads();
    bitonic_sort<kUnitBlock>(key, size);
    const int g = d.hit_off + w.start + p0;
#pragma unroll
    for (int k = 0; k < kPer; ++k)
      if (t + k * kUnitBlock < m) pr[k] = src[s_pos[key[padded(t + k * kUnitBlock)] & 0xfff]];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
      const int j = t + k * kUnitBlock;
      if (j < m) {
        key[j] = pr[k].idx;
        put_out<NT>(phis + g + j, pr[k].phi);
        inv[d.hit_off + pr[k].idx] = g + j;
      }
    }
    if (whole) scan_bins<kUnitBlock>(cur, part, nullptr);
    __syncthreads();
    write_hits<kUnitBlock, NT>(reinterpret_cast<const int*>(key), m, g, d.is_barrel != 0, hits + (size_t)d.hit_off * 9,
                               shits, qs, ranks);
    if (p0 == 0 && t < kNPhi)
      bins[d.bin_off + q * kNPhi + t] = bin_range(t, cur[4 * t], cur[4 * t + 4], cur[1024], w.start, w.n);
  }
}

// Per-hit bytes (the iteration's hit mask, as 0 or 1, or the charge codes) in sorted order, one tile of sorted
// positions per block: out[i] = in[hit of sorted position i].  Gathered, because the bytes of a layer stay in L2 while
// its outputs are written whole (scattering them by the inverse map: 19 us for 2.8M hits, against 6 us).
template <bool MASK>
__global__ void __launch_bounds__(256)
k_bytes_sorted(int n_layers, const int* __restrict__ tile_off, const LayerDev* __restrict__ L,
               const int* __restrict__ ranks, const unsigned char* __restrict__ in, unsigned char* __restrict__ out) {
  const int tile = xcd_major_block();
  const int l = layer_of_tile(tile, n_layers, tile_off);
  const LayerDev& d = L[l];
  const int first = (tile - tile_off[l]) * kTile;
  const int n = min(kTile, d.n_hits - first), g0 = d.hit_off + first;
  constexpr int kPer = kTile / 256;
  int r[kPer];
#pragma unroll
  for (int k = 0; k < kPer; ++k) r[k] = ranks[g0 + min((int)threadIdx.x + k * 256, n - 1)];
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const int i = threadIdx.x + k * 256;
    const unsigned char v = in[d.hit_off + r[k]];
    if (i < n) out[g0 + i] = MASK ? (v ? 1 : 0) : v;
  }
}

// One wavefront per workgroup, `lanes` of its lanes with a window each, scanned by all of them (25 -> 14 us for 30k
// lanes, against one window per lane scanned by that lane).
__global__ void __launch_bounds__(64)
k_select(LayerDev d, int n, int lanes, const float* __restrict__ par, const float* __restrict__ err,
         const int2* __restrict__ bins, const float* __restrict__ phis, const float* __restrict__ qs,
         const unsigned char* __restrict__ mask, const int* __restrict__ ranks, int* __restrict__ xsize,
         int* __restrict__ xarr, int* __restrict__ wsr) {
  __shared__ ScanLds S;
  const int lane = threadIdx.x, t = blockIdx.x * lanes + lane;
  const bool valid = lane < lanes && t < n;
  Window w;
  w.wsr = MKF_WSR_OUTSIDE;
  if (valid) {
    float p[6], e[21];
#pragma unroll
    for (int k = 0; k < 6; ++k) p[k] = par[(size_t)k * n + t];
#pragma unroll
    for (int k = 0; k < 21; ++k) e[k] = err[(size_t)k * n + t];
    hit_window(d, p, e, w);
  }
  const bool search = valid && w.wsr != MKF_WSR_OUTSIDE;
  const int cnt = wave_scan(search, d, w, bins, phis, qs, mask, S);
  if (valid) {
    wsr[t] = w.wsr;
    xsize[t] = search ? cnt : -1;
  }
  // the lists, rows of `lanes` entries by all lanes
  for (int j = lane; j < lanes * kHitIdxMax; j += 64) {
    const int o = j % lanes, k = j / lanes, to = blockIdx.x * lanes + o;
    if (to < n) xarr[(size_t)k * n + to] = k < min(S.cnt[o], kHitIdxMax) ? ranks[S.list[o][k]] : -1;
  }
}

// ---- FindTracksBestHit -------------------------------------------------------

struct FindArgs {
  int n, n_layers, first_layer, eoh_layers, spw;
  const int* __restrict__ layer_base;
  float chi2_cut;
  int pflags, prop_to_hit, intra_pflags;
  float bfield;
  Material mat;
  float* __restrict__ par;
  float* __restrict__ err;
  int* __restrict__ chg;
  float* __restrict__ chi2;
  int* __restrict__ hot;
  int* __restrict__ n_found;
  const LayerDev* __restrict__ layers;
  const int2* __restrict__ bins;
  const float* __restrict__ phis;
  const float* __restrict__ qs;
  const unsigned char* __restrict__ mask;
  const float* __restrict__ shits;
  const int* __restrict__ ranks;
};

// The reference's block loop (MkBuilder.cc:1395-1478), one wavefront per workgroup
// and one lane per seed for everything but the hits.  A lane that stops keeps the
// state it had at that point, which is the state the reference outputs for it
// (OutputTrackAndHitIdx at stop time).  HitOnTrack bookkeeping as
// MkFinder::add_hit (MkFinder.h:312-354); with at most MKF_MAX_FIND_LAYERS layers
// a track never exceeds Config::nMaxTrkHits.
//
// The windows' hits are scanned by the whole wavefront (wave_scan) and their chi2
// evaluated as (seed, hit) pairs spread over its lanes, so a layer waits for a few
// batches of loads instead of one per hit of the fullest window.  A wavefront
// carries `spw` seeds: 64 when there are enough to fill the chip, fewer otherwise,
// since the lanes without a seed still share the scan and the pairs.  (One lane per seed scanning and evaluating its
// own hits: 241 us for 500 seeds, 2.35 ms for 500k; so 120 us, bound by 8.5 us of dependent work per layer, and
// 1.8 ms, bound by the gathers' L2 misses.)
struct BestHitLds {
  ScanLds scan;
  float c2[64][kHitIdxMax];
  int pre[64];
  unsigned char owner[64 * kHitIdxMax];
};
constexpr int kRowW = 29;    // words of a lane's staged state: par, err, charge << 1 | barrel; odd stride
static_assert(sizeof(ScanLds::desc) >= 64 * kRowW * sizeof(float), "the staged states fit the scan's work list");

__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2))) k_find_best_hit(FindArgs a) {
  __shared__ BestHitLds S;
  float* __restrict__ X = reinterpret_cast<float*>(S.scan.desc);   // free between two scans
  const size_t n = (size_t)a.n;
  const int lane = threadIdx.x;
  const int t = blockIdx.x * a.spw + lane;
  bool alive = lane < a.spw && t < a.n;
  const int base = (alive && a.layer_base) ? a.layer_base[t] : 0;   // first layer of the seed's event
  const bool valid = alive && base >= 0 && base <= a.eoh_layers - a.n_layers;
  alive = valid;
  const LayerDev* __restrict__ lays = a.layers + (valid ? base : 0);
  float par[6], err[21];
  int chg = 1;
  float chi2 = 0.f;
  int nfound = 0, ninside = 0, ntail = 0, stop = a.n_layers;
  if (valid) {
#pragma unroll
    for (int e = 0; e < 6; ++e) par[e] = a.par[e * n + t];
#pragma unroll
    for (int e = 0; e < 21; ++e) err[e] = a.err[e * n + t];
    chg = a.chg[t];
    chi2 = a.chi2[t];
    for (int l = 0; l < a.first_layer; ++l) nfound += a.hot[l * n + t] >= 0;
  }
  for (int layer = a.first_layer; layer < a.n_layers && __any(alive); ++layer) {
    const LayerDev& d = lays[layer];
    float pp[6], pe[21];
    Window w;
    w.wsr = MKF_WSR_OUTSIDE;
    if (alive) {
#pragma unroll
      for (int e = 0; e < 6; ++e) pp[e] = par[e];
#pragma unroll
      for (int e = 0; e < 21; ++e) pe[e] = err[e];
      if (d.is_barrel)
        propagate_to_r(pp, pe, chg, d.propagate_to, a.pflags, false, a.bfield, a.mat);
      else
        propagate_to_z(pp, pe, chg, d.propagate_to, a.pflags, false, a.bfield, a.mat);
      // Tracks that cannot reach a barrel layer stop here (MkBuilder.cc:1431-1455).
      if (d.is_barrel && pp[0] * pp[0] + pp[1] * pp[1] < d.rin * d.rin) {
        alive = false;
        stop = layer;
      } else {
        hit_window(d, pp, pe, w);
      }
    }
    const int nc = wave_scan(alive && w.wsr != MKF_WSR_OUTSIDE, d, w, a.bins, a.phis, a.qs, a.mask, S.scan);
    const int incl = wave_inclusive(nc);
    const int total = __shfl(incl, 63, 64);
    S.pre[lane] = incl - nc;
    if (nc) {
      float* xs = X + lane * kRowW;
      for (int k = 0; k < nc; ++k) S.owner[incl - nc + k] = (unsigned char)lane;
#pragma unroll
      for (int e = 0; e < 6; ++e) xs[e] = pp[e];
#pragma unroll
      for (int e = 0; e < 21; ++e) xs[6 + e] = pe[e];
      xs[27] = __int_as_float(chg);
      xs[28] = __int_as_float(d.is_barrel);
    }
    __syncthreads();
    for (int j = lane; j < total; j += 64) {
      const int o = S.owner[j], k = j - S.pre[o];
      const float* xs = X + o * kRowW;
      float hp[3], he[6];
      load_hit9(a.shits + (size_t)S.scan.list[o][k] * 9, hp, he);
      const bool barrel = __float_as_int(xs[28]) != 0;
      float q[6], qe[21];
#pragma unroll
      for (int e = 0; e < 6; ++e) q[e] = xs[e];
#pragma unroll
      for (int e = 0; e < 21; ++e) qe[e] = xs[6 + e];
      if (a.prop_to_hit) {                                    // kalmanPropagateAndComputeChi2
        const int c = __float_as_int(xs[27]);
        if (barrel)
          propagate_to_r(q, qe, c, hypot_ref(hp[0], hp[1]), a.intra_pflags, false, a.bfield, a.mat);
        else
          propagate_to_z(q, qe, c, hp[2], a.intra_pflags, false, a.bfield, a.mat);
      }
      S.c2[o][k] = fabsf(barrel ? kalman_barrel<true, false>(q, qe, hp, he) : kalman_endcap<true, false>(q, qe, hp, he));
    }
    __syncthreads();
    if (!alive) continue;
    float mp[3] = {pp[0], pp[1], pp[2]};
    float me[6] = {666.f, 0.f, 666.f, 0.f, 0.f, 666.f};       // fake hit (MkFinder.cc:776-800)
    int code = -9;
    if (w.wsr != MKF_WSR_OUTSIDE) {
      float min_c2 = dyn_chi2_cut(d, a.chi2_cut, pp[3], pp[5]);
      int best = -1;
      for (int k = 0; k < nc; ++k) {
        const float c2 = S.c2[lane][k];
        if (c2 < min_c2) {
          min_c2 = c2;
          best = k;
        }
      }
      if (best >= 0) {
        const int gi = S.scan.list[lane][best];
        load_hit9(a.shits + (size_t)gi * 9, mp, me);
        chi2 += min_c2;
        code = a.ranks[gi];
        ++nfound;
        ninside += ntail;
        ntail = 0;
      } else {
        code = w.wsr == MKF_WSR_EDGE ? -3 : (ninside + ntail ? -2 : -1);
        ntail += code == -1;
      }
    }
    a.hot[layer * n + t] = code;
    if (a.prop_to_hit) {                                      // kalmanPropagateAndUpdate
      if (d.is_barrel)
        propagate_to_r(pp, pe, chg, hypot_ref(mp[0], mp[1]), a.intra_pflags, false, a.bfield, a.mat);
      else
        propagate_to_z(pp, pe, chg, mp[2], a.intra_pflags, false, a.bfield, a.mat);
    }
    if (d.is_barrel)
      kalman_barrel<false, true>(pp, pe, mp, me);
    else
      kalman_endcap<false, true>(pp, pe, mp, me);
    if (pp[3] < 0.f) {                                        // KalmanUtilsMPlex.cc:497-504
      chg = -chg;
      pp[3] = -pp[3];
    }
#pragma unroll
    for (int e = 0; e < 6; ++e) par[e] = pp[e];
#pragma unroll
    for (int e = 0; e < 21; ++e) err[e] = pe[e];
    if (code == -2) {                                         // MkBuilder.cc:1465-1473
      alive = false;
      stop = layer + 1;
    }
  }
  if (!valid) return;
  for (int layer = max(stop, a.first_layer); layer < a.n_layers; ++layer) a.hot[layer * n + t] = -9;
#pragma unroll
  for (int e = 0; e < 6; ++e) a.par[e * n + t] = par[e];
#pragma unroll
  for (int e = 0; e < 21; ++e) a.err[e * n + t] = err[e];
  a.chg[t] = chg;
  a.chi2[t] = chi2;
  a.n_found[t] = nfound;
}

}  // namespace

// ============================================================================
// C ABI
// ============================================================================


namespace {

void free_hit_arrays(mkf_event_of_hits* h) {
  void* ps[] = {h->d_phis, h->d_qs, h->d_shits, h->d_ranks, h->d_inv, h->d_sort};
  for (void* p : ps)
    if (p) (void)hipFree(p);
  h->d_ranks = h->d_inv = nullptr;
  h->d_phis = h->d_qs = h->d_shits = nullptr;
  h->d_sort = nullptr;
  h->cap = 0;
}

size_t aligned(size_t bytes) { return (bytes + 255) / 256 * 256; }

// A load's scratch for up to `cap` hits, whichever way they are sorted and however they lie over the layers and rows.
struct RowScratch {
  size_t place, pre, put, row_hist, hist, units, bytes;       // offsets behind the pairs
};
RowScratch row_scratch(const mkf_event_of_hits* h, size_t cap) {
  const size_t n_rows = h->total_bins / kNPhi;
  RowScratch r;
  r.place = aligned(cap * sizeof(RowPair));
  r.pre = r.place + aligned(cap * 4);
  r.put = r.pre + aligned((cap / kTile + h->n_layers) * (size_t)(h->max_nq + 1) * sizeof(unsigned short));
  r.row_hist = r.put + aligned(sizeof(PutOff));
  r.hist = r.row_hist + aligned(n_rows * 4);
  r.units = r.hist + aligned(cap / (kRowCap + 1) * kHistWords * 4);     // rows of more than kRowCap hits
  r.bytes = r.units + (n_rows + cap / kRowCap) * sizeof(RowUnit);            // ceil(n / kRowCap) a row
  return r;
}
int radix_scratch(size_t cap, size_t* temp, size_t* bytes) {
  HIP_TRY(hipcub::DeviceRadixSort::SortPairs(nullptr, *temp, (uint32_t*)nullptr, (uint32_t*)nullptr, (int*)nullptr,
                                             (int*)nullptr, (int)cap, 0, 32, (hipStream_t) nullptr));
  *bytes = 4 * aligned(cap * 4) + *temp;
  return MKF_OK;
}

// Both ways' scratch is taken when the hits outgrow the arrays, so that no later load of as many hits allocates.
int grow(mkf_event_of_hits* h, size_t total, hipStream_t st) {
  if (total <= h->cap && h->cap) return MKF_OK;
  HIP_TRY(hipStreamSynchronize(st));
  HIP_TRY(hipDeviceSynchronize());
  h->loaded = false;              // until this load is through: a failed allocation leaves nothing to search
  free_hit_arrays(h);
  const size_t cap = std::max<size_t>(total, 1024);
  size_t temp = 0, bytes = 0;
  CHECK(radix_scratch(cap, &temp, &bytes));
  HIP_TRY(hipMalloc(&h->d_phis, (cap + kScanUnroll) * 4));   // the scans read whole kScanUnroll runs
  HIP_TRY(hipMalloc(&h->d_qs, (cap + kScanUnroll) * 4));
  HIP_TRY(hipMalloc(&h->d_ranks, cap * 4));
  HIP_TRY(hipMalloc(&h->d_inv, cap * 4));
  HIP_TRY(hipMalloc(&h->d_shits, cap * 9 * 4));
  HIP_TRY(hipMalloc(&h->d_sort, std::max(bytes, row_scratch(h, cap).bytes)));
  h->sort_temp = temp;
  h->cap = cap;
  return MKF_OK;
}


// Tiles of the loaded hits.
int hit_tiles(const mkf_event_of_hits* h) {
  int tiles = 0;
  for (const LayerDev& d : h->layers) tiles += (d.n_hits + kTile - 1) / kTile;
  return tiles;
}

int blocks_for(size_t n, int block) { return (int)std::max<size_t>(1, (n + block - 1) / block); }

}  // namespace

extern "C" {

int mkf_event_of_hits_create(mkf_context* c, int n_layers, const mkf_layer_desc* desc, mkf_event_of_hits** out) {
  CHECK(set_device(c));
  if (!out || !desc) return fail(MKF_ERR_INVALID_ARG, "NULL argument");
  *out = nullptr;
  if (n_layers <= 0 || n_layers > MKF_MAX_EOH_LAYERS)
    return fail(MKF_ERR_INVALID_ARG, "n_layers must be in [1, %d]", MKF_MAX_EOH_LAYERS);
  std::vector<LayerDev> L(n_layers);
  int bin_off = 0;
  for (int l = 0; l < n_layers; ++l) {
    const mkf_layer_desc& s = desc[l];
    LayerDev& d = L[l];
    std::memset(&d, 0, sizeof(d));
    if (!(s.q_bin != 0.f) || !(s.rout >= s.rin) || !(s.zmax >= s.zmin))
      return fail(MKF_ERR_INVALID_ARG, "layer %d: invalid limits or q_bin", l);
    if (!(s.min_dphi >= 0.f && s.min_dphi <= s.max_dphi && s.max_dphi <= kPI) ||
        !(s.min_dq >= 0.f && s.min_dq <= s.max_dq && std::isfinite(s.max_dq)))
      return fail(MKF_ERR_INVALID_ARG, "layer %d: selection limits need 0 <= min <= max (max_dphi <= pi)", l);
    d.is_barrel = s.is_barrel ? 1 : 0;
    d.rin = s.rin; d.rout = s.rout; d.zmin = s.zmin; d.zmax = s.zmax;
    d.propagate_to = s.propagate_to;
    if (d.is_barrel)
      setup_bins(s.zmin, s.zmax, s.q_bin, d.nq, d.qmin, d.fq);
    else
      setup_bins(s.rin, s.rout, s.q_bin, d.nq, d.qmin, d.fq);
    if (d.nq <= 0 || d.nq > kMaxQBins || !std::isfinite(d.fq))
      return fail(MKF_ERR_INVALID_ARG, "layer %d: %d q bins (1..%d allowed)", l, d.nq, kMaxQBins);
    d.min_dphi = s.min_dphi; d.max_dphi = s.max_dphi; d.min_dq = s.min_dq; d.max_dq = s.max_dq;
    d.c_dp_sf = s.c_dp_sf; d.c_dp_0 = s.c_dp_0; d.c_dp_1 = s.c_dp_1; d.c_dp_2 = s.c_dp_2;
    d.c_dq_sf = s.c_dq_sf; d.c_dq_0 = s.c_dq_0; d.c_dq_1 = s.c_dq_1; d.c_dq_2 = s.c_dq_2;
    d.c_c2_sf = s.c_c2_sf; d.c_c2_0 = s.c_c2_0; d.c_c2_1 = s.c_c2_1; d.c_c2_2 = s.c_c2_2;
    d.bin_off = bin_off;
    if ((long)bin_off + (long)d.nq * kNPhi > (1L << 30)) return fail(MKF_ERR_INVALID_ARG, "too many bins");
    bin_off += d.nq * kNPhi;
  }
  auto* h = new mkf_event_of_hits();
  h->ctx = c;
  h->device = c->device;
  h->n_layers = n_layers;
  h->layers = L;
  h->total_bins = bin_off;
  std::vector<int> row_layer(bin_off / kNPhi);              // layer of each q row
  for (int l = 0; l < n_layers; ++l) {
    std::fill_n(row_layer.begin() + L[l].bin_off / kNPhi, L[l].nq, l);
    h->max_nq = std::max(h->max_nq, L[l].nq);
  }
  hipError_t e = hipMalloc(&h->d_layers, sizeof(LayerDev) * n_layers);
  if (e == hipSuccess) e = hipMemcpy(h->d_layers, L.data(), sizeof(LayerDev) * n_layers, hipMemcpyHostToDevice);
  // first tile per layer (set by each load), then the rows' layers
  if (e == hipSuccess) e = hipMalloc(&h->d_tile_off, sizeof(int) * (n_layers + 1 + row_layer.size()));
  if (e == hipSuccess) {
    h->d_row_layer = h->d_tile_off + n_layers + 1;
    e = hipMemcpy(h->d_row_layer, row_layer.data(), sizeof(int) * row_layer.size(), hipMemcpyHostToDevice);
  }

  if (e == hipSuccess) e = hipMalloc(&h->d_bins, sizeof(int2) * (size_t)bin_off);
  if (e != hipSuccess) {
    int rc = fail(MKF_ERR_HIP, "event-of-hits setup: %s", hipGetErrorString(e));
    mkf_event_of_hits_destroy(h);
    return rc;
  }
  *out = h;
  return MKF_OK;
}

int mkf_event_of_hits_destroy(mkf_event_of_hits* h) {
  if (!h) return MKF_OK;
  (void)hipSetDevice(h->device);
  (void)hipDeviceSynchronize();
  free_hit_arrays(h);
  if (h->d_tile_off) (void)hipFree(h->d_tile_off);
  if (h->d_ce_nodes) (void)hipFree(h->d_ce_nodes);
  if (h->d_mask_s) (void)hipFree(h->d_mask_s);
  if (h->d_charge_s) (void)hipFree(h->d_charge_s);
  if (h->d_dead) (void)hipFree(h->d_dead);
  if (h->ce_done) (void)hipEventDestroy(h->ce_done);
  if (h->d_layers) (void)hipFree(h->d_layers);
  if (h->d_bins) (void)hipFree(h->d_bins);
  delete h;
  return MKF_OK;
}

int mkf_event_of_hits_load(mkf_event_of_hits* h, const int* hit_offset, const float* hits, void* stream) {
  if (!h) return fail(MKF_ERR_INVALID_ARG, "event of hits is NULL");
  CHECK(set_device(h->ctx));
  if (!hit_offset) return fail(MKF_ERR_INVALID_ARG, "hit_offset is NULL");
  const int L = h->n_layers;
  if (hit_offset[0] != 0) return fail(MKF_ERR_INVALID_ARG, "hit_offset[0] must be 0");
  for (int l = 0; l < L; ++l)
    if (hit_offset[l + 1] < hit_offset[l]) return fail(MKF_ERR_INVALID_ARG, "hit_offset decreases at layer %d", l);
  const size_t total = (size_t)hit_offset[L];
  // hit positions are int throughout (keys, ranks, bin ranges, the sort's item count)
  if (total >= ((size_t)1 << 31) - 1) return fail(MKF_ERR_INVALID_ARG, "too many hits in one event of hits");
  if (total) CHECK(check_dev(hits, total * 9 * 4, "hits"));
  hipStream_t st = (hipStream_t)stream;
  bool rows = true, put_off = false;            // put_off: a row may be (its layer holds more than kBinMax hits)
  int tiles = 0;
  for (int l = 0; l < L; ++l) {
    const size_t nl = (size_t)hit_offset[l + 1] - hit_offset[l];
    rows = rows && nl <= kRowLayerMax;
    put_off = put_off || nl > (size_t)kBinMax;
    tiles += (int)((nl + kTile - 1) / kTile);
  }
  const int pre_stride = h->max_nq + 1;
  CHECK(grow(h, total, st));
  h->has_mask = false;
  h->has_charge = false;
  for (int l = 0; l < L; ++l) {
    h->layers[l].hit_off = hit_offset[l];
    h->layers[l].n_hits = hit_offset[l + 1] - hit_offset[l];
  }
  const RowScratch lay = row_scratch(h, h->cap);
  char* scr = static_cast<char*>(h->d_sort);
  PutOff* put = reinterpret_cast<PutOff*>(scr + lay.put);
  for (int f = 0, tile = 0; f < L; f += kOffChunk) {
    OffsetsArg o;
    o.first = f;
    o.count = std::min(kOffChunk, L - f);
    for (int l = 0; l <= o.count; ++l) {
      o.off[l] = hit_offset[f + l];
      o.tile[l] = tile;
      if (l < o.count) tile += (h->layers[f + l].n_hits + kTile - 1) / kTile;
    }
    hipLaunchKernelGGL(k_set_offsets, dim3(1), dim3(kOffChunk), 0, st, o, h->d_layers, h->d_tile_off, put);
    HIP_TRY(hipGetLastError());
  }
  const int n_rows = h->total_bins / kNPhi;
  if (rows) {
    RowPair* pairs = reinterpret_cast<RowPair*>(scr);
    int* place = reinterpret_cast<int*>(scr + lay.place);
    unsigned short* pre = reinterpret_cast<unsigned short*>(scr + lay.pre);
    int* row_hist = reinterpret_cast<int*>(scr + lay.row_hist);
    int* hist = reinterpret_cast<int*>(scr + lay.hist);
    RowUnit* units = reinterpret_cast<RowUnit*>(scr + lay.units);
    if (tiles) {
      hipLaunchKernelGGL(k_row_partition, dim3(tiles), dim3(kPartBlock), 0, st, L, h->d_tile_off, h->d_layers, hits,
                         pairs, pre, pre_stride);
      HIP_TRY(hipGetLastError());
    }
    // a row weighs its layer's mean of hits and a constant for the block itself
    XcdRows xr;
    const double all = (double)total + (double)kRowWeight * n_rows;
    int x = 0, longest = 0;
    double w = 0.0;
    for (int l = 0; l < L; ++l) {
      const LayerDev& d = h->layers[l];
      const double each = (double)d.n_hits / d.nq + kRowWeight;
      for (; x < 8 && w + each * d.nq > all * x / 8; ++x)
        xr.first[x] = std::min(n_rows, d.bin_off / kNPhi + (int)std::max(0.0, std::ceil((all * x / 8 - w) / each)));
      w += each * d.nq;
    }
    for (; x <= 8; ++x) xr.first[x] = n_rows;
    xr.first[0] = 0;
    xr.first[8] = n_rows;
    for (int k = 0; k < 8; ++k) longest = std::max(longest, xr.first[k + 1] - xr.first[k]);
    hipLaunchKernelGGL((total > kStreamHits ? k_row_sort<true> : k_row_sort<false>), dim3(8 * longest), dim3(kRowBlock), 0,
                       st, xr, h->d_row_layer, h->d_layers, h->d_tile_off, pre, pre_stride, pairs, hits, h->d_shits,
                       h->d_phis, h->d_qs, h->d_ranks, place, h->d_bins, put, row_hist, hist, units);
    HIP_TRY(hipGetLastError());
    if (tiles) {
      hipLaunchKernelGGL(k_row_tiles, dim3(tiles), dim3(kPartBlock), 0, st, L, h->d_tile_off, h->d_layers, pairs, place,
                         h->d_inv, pre, pre_stride, put, row_hist, hist);
      HIP_TRY(hipGetLastError());
    }
    if (put_off) {
      // two blocks per CU (122 VGPRs), whole eights for the XCDs' shares
      const int grid = (std::min(2 * h->ctx->num_cus, n_rows + (int)(total / kRowCap)) + 7) / 8 * 8;
      hipLaunchKernelGGL((total > kStreamHits ? k_row_units<true> : k_row_units<false>), dim3(grid), dim3(kUnitBlock), 0,
                         st, put, units, hist, h->d_row_layer, h->d_layers, h->d_tile_off, pre, pre_stride, pairs, hits,
                         h->d_shits, h->d_phis, h->d_qs, h->d_ranks, h->d_inv, h->d_bins);
      HIP_TRY(hipGetLastError());
    }
    h->loaded = true;
    return MKF_OK;
  }
  hipLaunchKernelGGL(k_fill_i32, dim3(std::min(blocks_for((size_t)h->total_bins * 2, 256), 4096)), dim3(256), 0, st,
                     reinterpret_cast<int*>(h->d_bins), (long)h->total_bins * 2, 0);
  HIP_TRY(hipGetLastError());
  const int nt = (int)total;
  uint32_t* keys = reinterpret_cast<uint32_t*>(scr);
  uint32_t* keys_s = reinterpret_cast<uint32_t*>(scr + aligned(h->cap * 4));
  int* vals = reinterpret_cast<int*>(scr + 2 * aligned(h->cap * 4));
  int* vals_s = reinterpret_cast<int*>(scr + 3 * aligned(h->cap * 4));
  hipLaunchKernelGGL(k_hit_keys, dim3(blocks_for(total, 256)), dim3(256), 0, st, nt, L, hits, h->d_layers, keys, vals);
  HIP_TRY(hipGetLastError());
  size_t temp = h->sort_temp;
  HIP_TRY(hipcub::DeviceRadixSort::SortPairs(scr + 4 * aligned(h->cap * 4), temp, keys, keys_s, vals, vals_s, nt, 0, 32,
                                             st));
  hipLaunchKernelGGL(k_loh_gather, dim3(blocks_for(total, 256)), dim3(256), 0, st, nt, keys_s, vals_s, h->d_layers,
                     hits, h->d_shits, h->d_phis, h->d_qs);
  HIP_TRY(hipGetLastError());
  for (int pass = 0; pass < 2; ++pass) {
    hipLaunchKernelGGL(k_loh_fill, dim3(blocks_for(total, 256)), dim3(256), 0, st, nt, pass, keys_s, vals_s,
                       h->d_layers, h->d_ranks, h->d_inv, h->d_bins);
    HIP_TRY(hipGetLastError());
  }
  h->loaded = true;
  return MKF_OK;
}

int mkf_event_of_hits_set_hit_mask(mkf_event_of_hits* h, const unsigned char* mask, void* stream) {
  if (!h) return fail(MKF_ERR_INVALID_ARG, "event of hits is NULL");
  CHECK(set_device(h->ctx));
  if (!h->loaded) return fail(MKF_ERR_INVALID_ARG, "event of hits not loaded");
  if (!mask) {
    h->has_mask = false;
    return MKF_OK;
  }
  const LayerDev& last = h->layers[h->n_layers - 1];
  const size_t total = (size_t)last.hit_off + last.n_hits;
  hipStream_t st = (hipStream_t)stream;
  if (total) CHECK(check_dev(mask, total, "mask"));
  if (total > h->mask_cap) {
    HIP_TRY(hipStreamSynchronize(st));
    if (h->d_mask_s) HIP_TRY(hipFree(h->d_mask_s));
    h->has_mask = false;
    h->d_mask_s = nullptr;
    h->mask_cap = 0;
    HIP_TRY(hipMalloc(&h->d_mask_s, total));
    h->mask_cap = total;
  }
  if (total) {
    hipLaunchKernelGGL(k_bytes_sorted<true>, dim3(hit_tiles(h)), dim3(256), 0, st, h->n_layers, h->d_tile_off,
                       h->d_layers, h->d_ranks, mask, h->d_mask_s);
    HIP_TRY(hipGetLastError());
  }
  h->has_mask = true;
  return MKF_OK;
}

int mkf_event_of_hits_set_hit_charge(mkf_event_of_hits* h, const unsigned char* code, void* stream) {
  if (!h) return fail(MKF_ERR_INVALID_ARG, "event of hits is NULL");
  CHECK(set_device(h->ctx));
  if (!h->loaded) return fail(MKF_ERR_INVALID_ARG, "event of hits not loaded");
  if (!code) {
    h->has_charge = false;
    return MKF_OK;
  }
  const LayerDev& last = h->layers[h->n_layers - 1];
  const size_t total = (size_t)last.hit_off + last.n_hits;
  hipStream_t st = (hipStream_t)stream;
  if (total) CHECK(check_dev(code, total, "charge codes"));
  if (total > h->charge_cap) {
    HIP_TRY(hipStreamSynchronize(st));
    if (h->d_charge_s) HIP_TRY(hipFree(h->d_charge_s));
    h->has_charge = false;
    h->d_charge_s = nullptr;
    h->charge_cap = 0;
    HIP_TRY(hipMalloc(&h->d_charge_s, total));
    h->charge_cap = total;
  }
  if (total) {
    hipLaunchKernelGGL(k_bytes_sorted<false>, dim3(hit_tiles(h)), dim3(256), 0, st, h->n_layers, h->d_tile_off,
                       h->d_layers, h->d_ranks, code, h->d_charge_s);
    HIP_TRY(hipGetLastError());
  }
  h->has_charge = true;
  return MKF_OK;
}

int mkf_event_of_hits_set_dead_regions(mkf_event_of_hits* h, int n, const float* regions, void* stream) {
  if (!h) return fail(MKF_ERR_INVALID_ARG, "event of hits is NULL");
  CHECK(set_device(h->ctx));
  if (n < 0 || (n > 0 && !regions)) return fail(MKF_ERR_INVALID_ARG, "dead regions: bad count or NULL");
  if (n == 0) {
    h->has_dead = false;
    return MKF_OK;
  }
  // LayerOfHits::SuckInDeads (HitStructures.cc:186-212) per region's layer; a phi bin of 256 (phi2 = +pi)
  // stands for bin 0.
  std::vector<unsigned char> dead((size_t)h->total_bins, 0);
  for (int r = 0; r < n; ++r) {
    const float* g = regions + (size_t)r * 5;
    const int layer = (int)g[0];
    if (layer < 0 || layer >= h->n_layers || !(g[0] == (float)layer))
      return fail(MKF_ERR_INVALID_ARG, "dead region %d: layer %g is not a layer of the event of hits", r, g[0]);
    const LayerDev& d = h->layers[layer];
    const int q1 = q_bin_checked(d, g[3]), q2 = q_bin_checked(d, g[4]) + 1;
    const int p1 = phi_bin(g[1]), p2 = phi_bin(g[2]) + 1;
    if (p1 < -2 || p1 > kNPhi || p2 < -1 || p2 > kNPhi + 1)
      return fail(MKF_ERR_INVALID_ARG, "dead region %d: phi outside [-pi, pi]", r);
    unsigned char* row0 = dead.data() + d.bin_off;
    for (int q = q1; q < q2; ++q) {
      unsigned char* row = row0 + (size_t)q * kNPhi;
      if (p1 > p2) {
        for (int p = p1; p < kNPhi; ++p) row[p & 0xff] = 1;
        for (int p = 0; p < p2; ++p) row[p & 0xff] = 1;
      } else {
        for (int p = p1; p < p2; ++p) row[p & 0xff] = 1;
      }
    }
  }
  hipStream_t st = (hipStream_t)stream;
  if (!h->d_dead) HIP_TRY(hipMalloc(&h->d_dead, (size_t)h->total_bins));
  HIP_TRY(hipMemcpyAsync(h->d_dead, dead.data(), (size_t)h->total_bins, hipMemcpyHostToDevice, st));
  HIP_TRY(hipStreamSynchronize(st));
  h->has_dead = true;
  return MKF_OK;
}

int mkf_event_of_hits_layer(mkf_event_of_hits* h, int layer, int* n_hits, int* nq, const int** ranks,
                            const int** bins, const float** phis, const float** qs) {
  if (!h) return fail(MKF_ERR_INVALID_ARG, "event of hits is NULL");
  if (!h->loaded) return fail(MKF_ERR_INVALID_ARG, "event of hits not loaded");
  if (layer < 0 || layer >= h->n_layers) return fail(MKF_ERR_INVALID_ARG, "layer %d out of range", layer);
  const LayerDev& d = h->layers[layer];
  if (n_hits) *n_hits = d.n_hits;
  if (nq) *nq = d.nq;
  if (ranks) *ranks = h->d_ranks ? h->d_ranks + d.hit_off : nullptr;
  if (bins) *bins = reinterpret_cast<const int*>(h->d_bins + d.bin_off);
  if (phis) *phis = h->d_phis ? h->d_phis + d.hit_off : nullptr;
  if (qs) *qs = h->d_qs ? h->d_qs + d.hit_off : nullptr;
  return MKF_OK;
}

int mkf_select_hit_indices(mkf_event_of_hits* h, int layer, int n, const float* par, const float* err, int* xsize,
                           int* xarr, int* wsr, void* stream) {
  if (!h) return fail(MKF_ERR_INVALID_ARG, "event of hits is NULL");
  CHECK(set_device(h->ctx));
  if (!h->loaded) return fail(MKF_ERR_INVALID_ARG, "event of hits not loaded");
  if (layer < 0 || layer >= h->n_layers) return fail(MKF_ERR_INVALID_ARG, "layer %d out of range", layer);
  if (n < 0) return fail(MKF_ERR_INVALID_ARG, "n < 0");
  if (n == 0) return MKF_OK;
  const size_t N = n;
  CHECK(check_dev(par, 6 * N * 4, "par"));
  CHECK(check_dev(err, 21 * N * 4, "err"));
  CHECK(check_dev(xsize, N * 4, "xsize"));
  CHECK(check_dev(xarr, kHitIdxMax * N * 4, "xarr"));
  CHECK(check_dev(wsr, N * 4, "wsr"));
  const int lanes = lanes_per_wave(N, h->ctx->num_cus);
  hipLaunchKernelGGL(k_select, dim3(blocks_for(N, lanes)), dim3(64), 0, (hipStream_t)stream, h->layers[layer], n, lanes,
                     par, err, h->d_bins, h->d_phis, h->d_qs, h->mask(), h->d_ranks, xsize, xarr, wsr);
  HIP_TRY(hipGetLastError());
  return MKF_OK;
}

int mkf_find_tracks_best_hit(mkf_context* c, mkf_event_of_hits* h, const mkf_find_batch* b, void* stream) {
  CHECK(set_device(c));
  if (!h || !b) return fail(MKF_ERR_INVALID_ARG, "NULL argument");
  if (h->ctx != c) return fail(MKF_ERR_INVALID_ARG, "event of hits belongs to another context");
  if (!h->loaded) return fail(MKF_ERR_INVALID_ARG, "event of hits not loaded");
  if (b->n_tracks < 0) return fail(MKF_ERR_INVALID_ARG, "n_tracks < 0");
  const int LE = b->n_layers ? b->n_layers : h->n_layers;   // layers per event
  if (LE < 1 || LE > h->n_layers || LE > MKF_MAX_FIND_LAYERS)
    return fail(MKF_ERR_INVALID_ARG, "n_layers %d outside [1, min(%d, %d)]", LE, h->n_layers, MKF_MAX_FIND_LAYERS);
  if (b->first_layer < 0 || b->first_layer > LE)
    return fail(MKF_ERR_INVALID_ARG, "first_layer %d outside [0, %d]", b->first_layer, LE);
  if (((b->pflags | (b->prop_to_hit ? b->intra_pflags : 0)) & MKF_PF_APPLY_MATERIAL) && !c->d_rl)
    return fail(MKF_ERR_INVALID_ARG, "material requested but the context has no material grid");
  if (b->n_tracks == 0) return MKF_OK;
  const size_t N = b->n_tracks;
  if (21 * N * 4 >= ((size_t)1 << 31) || (size_t)LE * N >= ((size_t)1 << 31))
    return fail(MKF_ERR_INVALID_ARG, "batch too large");
  CHECK(check_dev(b->par, 6 * N * 4, "par"));
  CHECK(check_dev(b->err, 21 * N * 4, "err"));
  CHECK(check_dev(b->chg, N * 4, "chg"));
  CHECK(check_dev(b->chi2, N * 4, "chi2"));
  CHECK(check_dev(b->hot_idx, (size_t)LE * N * 4, "hot_idx"));
  CHECK(check_dev(b->n_found, N * 4, "n_found"));
  if (b->layer_base) CHECK(check_dev(b->layer_base, N * 4, "layer_base"));
  else if (LE != h->n_layers)
    return fail(MKF_ERR_INVALID_ARG, "n_layers %d below the event of hits' %d needs layer_base", LE, h->n_layers);
  FindArgs a;
  a.n = b->n_tracks;
  a.n_layers = LE;
  a.eoh_layers = h->n_layers;
  a.layer_base = b->layer_base;
  a.first_layer = b->first_layer;
  a.chi2_cut = b->chi2_cut;
  a.pflags = b->pflags;
  a.prop_to_hit = b->prop_to_hit;
  a.intra_pflags = b->intra_pflags;
  a.bfield = c->bfield;
  a.mat = mat_of(c);
  a.par = b->par; a.err = b->err; a.chg = b->chg; a.chi2 = b->chi2;
  a.hot = b->hot_idx; a.n_found = b->n_found;
  a.layers = h->d_layers;
  a.bins = h->d_bins;
  a.phis = h->d_phis; a.qs = h->d_qs; a.shits = h->d_shits; a.ranks = h->d_ranks;
  a.mask = h->mask();
  a.spw = lanes_per_wave(N, h->ctx->num_cus);
  hipLaunchKernelGGL(k_find_best_hit, dim3(blocks_for(N, a.spw)), dim3(64), 0, (hipStream_t)stream, a);
  HIP_TRY(hipGetLastError());
  return MKF_OK;
}

}  // extern "C"
