// mkf_ce.hip -- clone-engine track finding on gfx950.
//
// One 64-lane workgroup carries up to 8 or 10 seeds through every layer: lane
// g*KS + c holds candidate c of seed g (KS = 8 slots per seed, or 6 when at most
// 6 candidates are kept) with its state in VGPRs.
// Per layer:
//   (a) lanes propagate their candidate to the layer, select hits and compute
//       each hit's chi2 (after propagating to the hit, as the reference does
//       with finding_requires_propagation_to_hit_pos); accepted hits and the
//       invalid-hit entry go to LDS as IdxChi2List records;
//   (b) the seed's lanes rank its records (each lane offers its best remaining
//       one, max_cands times: a stable top-K by score in the reference's
//       generation order) and one of them lays out the seed's next candidate
//       list -- records interleaved with held-back extras, the best short
//       candidate set aside (CandCloner::ProcessSeedRange);
//   (c) every lane builds its new candidate from its parent's state (exchanged
//       through LDS), appends the HitOnTrack node and, for a real hit, applies
//       the Kalman update after propagating to the hit (UpdateWithLastHit).
// Hit lists live in a per-seed append-only node store in HBM, like the
// reference's CombCandidate::m_hots: cloning a candidate copies one index.
// After the last layer MergeCandsAndBestShortOne orders the candidates, and
// each lane walks its node chain to write the per-layer hit indices.
//
// The same kernel with STD runs standard combinatorial finding
// (MkBuilder::FindTracksStandard, MkFinder::FindCandidates, MkFinder.cc:902-1109):
// a new candidate carries its parent's state at the layer -- updated with its
// hit after propagating to it with the intra-layer flags -- and is scored with
// its own updated pT; held-back, new and invalid-hit candidates are ranked
// together, the best max_cands without a -2 hit are kept and the first -2 one
// in that order competes for the best short candidate (MkBuilder.cc:1760-1828).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <vector>

#include "../../include/mkfit_amd.h"
#include "mkf_find_common.h"
#include "mkf_internal.h"
#include "mkf_track_math.h"

using namespace mkf;
using namespace mkf_detail;
using namespace mkf_find;

namespace {

constexpr int kSMax = 8;              // candidate slots per seed, at most
constexpr int kLanes = 64;            // one wavefront per workgroup
constexpr int kW = 37;                // LDS words per exchanged candidate (36 used, odd stride)
// Words of a lane's X row during (a), beside the propagated state in words 0-27:
// chi2 cut, exclusive prefix of the window hit counts, layer hit offset,
// barrel flag of the lane's layer and, in words 32-35, sin / cos of the
// propagated phi and theta.  Word 36, which put / get leave alone, holds
// the score of the lane's invalid-hit record from (a) to the new candidates (c).
constexpr int kXCut = 28, kXPre = 29, kXOff = 30, kXBar = 31, kXTrig = 32, kXScore = 36;
constexpr int kMaxLayerHits = (1 << 28) - 1;   // most hits of a layer: a limit of the entry points, not of the kernel
constexpr int kBsW = 40;              // words per seed of the best short candidate store (36 used)

// Ranking key of an entry: its score, then the earlier place in the reference's
// generation order.  Held back (standard finding): place = slot; a record: kSMax + hit_cnt * kSMax
// + slot; an invalid-hit entry: after every record.  0: no entry.  Scores are finite; adding 0 makes
// -0 equal to +0.
constexpr int kGenRec = kSMax, kGenFake = kSMax + kHitIdxMax * kSMax, kGenEnd = kGenFake + kSMax;
__device__ __forceinline__ uint64_t rank_key(float score, int gen) {
  const unsigned b = __float_as_uint(score + 0.f);
  const unsigned o = b ^ ((b >> 31) ? 0xffffffffu : 0x80000000u);
  return (uint64_t)o << 32 | (unsigned)(kGenEnd - gen);
}
__device__ __forceinline__ float key_score(uint64_t key) {
  const unsigned o = (unsigned)(key >> 32);
  return __uint_as_float(o ^ ((o >> 31) ? 0x80000000u : 0xffffffffu));
}
__device__ __forceinline__ int key_gen(uint64_t key) { return kGenEnd - (int)(unsigned)key; }

// The greatest key of the lane's seed group (lanes lane0 .. lane0 + KS - 1): after the steps 1, 2 and KS - 4, taken
// around the group, a lane has seen all of its KS <= 8 keys.
template <int KS>
__device__ __forceinline__ uint64_t group_max(uint64_t key, int lane0, int c) {
  static_assert(KS > 4 && KS <= 8, "three steps cover the group");
#pragma unroll
  for (int o : {1, 2, KS - 4}) {
    const uint64_t k = __shfl(key, lane0 + (c + o >= KS ? c + o - KS : c + o), 64);
    key = k > key ? k : key;
  }
  return key;
}

struct Cand {
  float par[6], err[21];
  int chg;
  float chi2, score;
  int nfound, nmissing, ninside, ntail;
  int last;       // node index of the last HitOnTrack (CombCandidate::m_hots position)
  int last_hit;   // hit index stored in that node
};

__device__ __forceinline__ void add_hit_counts(Cand& c, int idx, float chi2) {   // TrackCand::addHitIdx
  if (idx >= 0 || idx == -9) {
    ++c.nfound;
    c.chi2 += chi2;
    c.ninside += c.ntail;
    c.ntail = 0;
  } else {
    ++c.nmissing;
    if (idx == -1) ++c.ntail;
  }
  c.last_hit = idx;
}

__device__ __forceinline__ float cand_score(const Cand& c) {                       // getScoreCand
  const float chi2 = c.chi2 < 0 ? 0.f : c.chi2;
  return score_calc(c.nfound, 0, 0, c.ninside, chi2, fabsf(1.f / c.par[3]), false);
}

__device__ __forceinline__ void put(float* X, const Cand& c) {
#pragma unroll
  for (int e = 0; e < 6; ++e) X[e] = c.par[e];
#pragma unroll
  for (int e = 0; e < 21; ++e) X[6 + e] = c.err[e];
  X[27] = __int_as_float(c.chg);
  X[28] = c.chi2;
  X[29] = c.score;
  X[30] = __int_as_float(c.nfound);
  X[31] = __int_as_float(c.nmissing);
  X[32] = __int_as_float(c.ninside);
  X[33] = __int_as_float(c.ntail);
  X[34] = __int_as_float(c.last);
  X[35] = __int_as_float(c.last_hit);
}
// The words of `put` after the state: charge, chi2, score, counters, nodes.
__device__ __forceinline__ void put_counts(float* X, const Cand& c) {
  X[27] = __int_as_float(c.chg);
  X[28] = c.chi2;
  X[29] = c.score;
  X[30] = __int_as_float(c.nfound);
  X[31] = __int_as_float(c.nmissing);
  X[32] = __int_as_float(c.ninside);
  X[33] = __int_as_float(c.ntail);
  X[34] = __int_as_float(c.last);
  X[35] = __int_as_float(c.last_hit);
}
__device__ __forceinline__ void get(const float* X, Cand& c) {
#pragma unroll
  for (int e = 0; e < 6; ++e) c.par[e] = X[e];
#pragma unroll
  for (int e = 0; e < 21; ++e) c.err[e] = X[6 + e];
  c.chg = __float_as_int(X[27]);
  c.chi2 = X[28];
  c.score = X[29];
  c.nfound = __float_as_int(X[30]);
  c.nmissing = __float_as_int(X[31]);
  c.ninside = __float_as_int(X[32]);
  c.ntail = __float_as_int(X[33]);
  c.last = __float_as_int(X[34]);
  c.last_hit = __float_as_int(X[35]);
}

struct CeArgs {
  int n, n_layers, first_layer, eoh_layers, spw;
  const int* __restrict__ layer_base;
  int max_cands, max_holes, max_consec, prop_to_hit, intra_pflags, inter_pflags;
  float chi2_cut, bfield;
  Material mat;
  const float* __restrict__ seed_par;
  const float* __restrict__ seed_err;
  const int* __restrict__ seed_chg;
  const int* __restrict__ seed_hits;
  int* __restrict__ n_cands;
  float* __restrict__ par;
  float* __restrict__ err;
  int* __restrict__ chg;
  float* __restrict__ chi2;
  float* __restrict__ bs;         // per seed kBsW words: the best short candidate
  float* __restrict__ score;
  int* __restrict__ n_found;
  int* __restrict__ hot;
  int4* __restrict__ nodes;   // [n][node_cap] {hit index, layer, prev node, 0}
  int node_cap;
  const LayerDev* __restrict__ layers;
  const int2* __restrict__ bins;
  const float* __restrict__ phis;
  const float* __restrict__ qs;
  const unsigned char* __restrict__ mask;
  const unsigned char* __restrict__ charge;   // per sorted hit: strip charge code, or NULL (every hit passes)
  const unsigned char* __restrict__ dead;     // dead-module bins per (layer, q bin, phi bin), or NULL
  const float* __restrict__ shits;
  const int* __restrict__ ranks;
};

// Appends a node to seed `s`'s store; returns its index, or -1 when the store
// is full (never for the store size the host allocates: 3 nodes per candidate
// slot and layer plus the seed hits).
__device__ __forceinline__ int append_node(const CeArgs& a, int s, int* cnt, int hit, int layer, int prev) {
  const int k = atomicAdd(cnt, 1);
  if (k >= a.node_cap) return -1;
  a.nodes[(size_t)s * a.node_cap + k] = make_int4(hit, layer, prev, 0);
  return k;
}

__device__ __forceinline__ void propagate(bool barrel, float (&p)[6], float (&e)[21], int chg, float target,
                                          int pflags, const CeArgs& a, const float* trig = nullptr) {
  if (barrel)
    propagate_to_r(p, e, chg, target, pflags, false, a.bfield, a.mat, trig);
  else
    propagate_to_z(p, e, chg, target, pflags, false, a.bfield, a.mat, trig);
}

// KS candidate slots per seed (max_cands <= KS): KS = 6 packs up to 10 seeds into
// the wavefront's 64 lanes (4 idle), KS = 8 up to 8; a.spw of them are used.  Lanes past the last
// seed group take no part.  STD: standard finding (see the top).
// WAVES: waves per SIMD the registers are allotted for.  Left to itself the compiler spends all 512
// registers of a lane on one wave; two measured 21.0 against 29.7 ms for the standard form and 15.3
// against 28.1 ms for the clone engine (50 events).  mkf_autotune_find picks KS and WAVES by timing.
template <int KS, bool STD, int WAVES>
__global__ void __launch_bounds__(kLanes) __attribute__((amdgpu_waves_per_eu(WAVES))) k_find_clone_engine(CeArgs a) {
  constexpr int kS = KS;
  constexpr int kG = kLanes / KS;             // seeds per workgroup
  constexpr int kGA = kG + 1;                 // seed rows in LDS: one more for the idle lanes
  // 19.9 KB (kS = 6) / 20.4 KB (kS = 8): eight workgroups per CU, as many as
  // the VGPRs allow.
  __shared__ float X[kLanes * kW];          // candidate state exchange (and the kX* words in (a))
  __shared__ int Gh[kLanes][kHitIdxMax];    // each lane's window hits (positions in the layer), in scan order
  __shared__ float Gc[kLanes][kHitIdxMax];  // their chi2 if accepted, else -1
  __shared__ float Es[kLanes][kS];          // (a2) the pairs' owners; (b) row g*kS + r: the seed's r-th ranked entry
  __shared__ float Gp[STD ? kLanes : 1][kHitIdxMax];   // STD: pT of each accepted hit's updated state
  __shared__ signed char fcode[kLanes];     // invalid-hit record's hit code, 0 = none
  __shared__ unsigned char xkind[kLanes];   // 1 = held back unchanged, 2 = stopped replica
  __shared__ int D[kGA][kS];                // next candidates: kind | parent slot << 2 | rank << 5 | hit_cnt << 8
  __shared__ float s_bsc[kGA];              // score of the best short candidate (the candidate: a.bs)
  __shared__ int s_nnodes[kGA];
  __shared__ unsigned char s_bs[kGA], s_state[kGA], s_ncand[kGA], s_any[kGA], s_nnew[kGA], s_merge[kGA];
  __shared__ unsigned char s_nout[kGA];

  const int lane = threadIdx.x;
  const int g = lane / kS, c = lane % kS;
  const int seed = blockIdx.x * a.spw + g;
  const bool gin = g < a.spw && seed < a.n;
  const int base = (gin && a.layer_base) ? a.layer_base[seed] : 0;   // first layer of the seed's event
  const bool gvalid = gin && base >= 0 && base <= a.eoh_layers - a.n_layers;
  const LayerDev* __restrict__ lays = a.layers + (gvalid ? base : 0);
  const size_t N = (size_t)a.n;
  const int K = a.max_cands;

  Cand st = {};
  if (c == 0) {
    s_state[g] = 0;
    s_ncand[g] = gvalid ? 1 : 0;
    s_nnodes[g] = 0;
    s_bs[g] = 0;
    s_bsc[g] = kScoreWorst;
  }
  __syncthreads();
  if (gvalid && c == 0) {                                    // CombCandidate::ImportSeed
#pragma unroll
    for (int e = 0; e < 6; ++e) st.par[e] = a.seed_par[e * N + seed];
#pragma unroll
    for (int e = 0; e < 21; ++e) st.err[e] = a.seed_err[e * N + seed];
    st.chg = a.seed_chg[seed];
    st.chi2 = 0.f;
    st.nfound = st.nmissing = st.ninside = st.ntail = 0;
    st.last = -1;
    st.last_hit = -1;
    for (int l = 0; l < a.first_layer; ++l) {
      const int h = a.seed_hits[l * N + seed];
      const int k = append_node(a, seed, &s_nnodes[g], h, l, st.last);
      if (k >= 0) st.last = k;
      add_hit_counts(st, h, 0.f);
    }
    st.score = cand_score(st);
  }

  for (int layer = a.first_layer; layer < a.n_layers; ++layer) {
    const LayerDev& d = lays[layer];
    const bool barrel = d.is_barrel != 0;
    // ---- (a) find_tracks_unroll_candidates
    if (c == 0 && gvalid) {
      if (s_state[g] == 0 && layer - 1 == a.first_layer - 1) s_state[g] = 1;
      s_any[g] = 0;
    }
    fcode[lane] = 0;
    xkind[lane] = 0;
    __syncthreads();
    const bool finding = gvalid && s_state[g] == 1;
    const bool valid = finding && c < s_ncand[g];
    bool active = valid && st.last_hit != -2;
    if (active && fabsf(1.f / st.par[3]) < 1.2f) {          // near the apex of a low-pT helix
      const float dphi = fabsf(atan2_cr(st.par[1], st.par[0]) - st.par[4]);
      if (st.par[0] * st.par[0] + st.par[1] * st.par[1] > 625.f && dphi > 1.371f && dphi < 4.512f) {
        const int k = append_node(a, seed, &s_nnodes[g], -2, layer, st.last);
        if (k >= 0) st.last = k;
        add_hit_counts(st, -2, 0.f);
        active = false;
      }
    }
    if (active) s_any[g] = 1;
    __syncthreads();
    if (c == 0) s_merge[g] = finding && s_any[g];
    if (c == 0 && finding && !s_any[g]) s_state[g] = 2;
    // FindCandidatesCloneEngine (MkFinder.cc:1114-1284) in three phases, so the
    // costly part -- the propagation to each window hit and its chi2 -- runs
    // on a compacted list of (lane, hit) pairs with every lane of the
    // wavefront busy, however unevenly the hits fall into the lanes' windows:
    //   (a1) each lane propagates to the layer, builds its window and lists
    //        the window's hits (at most 16, in scan order);
    //   (a2) a wavefront prefix sum of the list lengths numbers all pairs, and
    //        lane i evaluates pairs i, i + 64, ... for their owners;
    //   (a3) each lane turns its accepted hits into records, in scan order.
    int nh = 0;
    float pt_l = 0.f;
    bool search = false, gap = false;
    if (active) {
      float pp[6], pe[21];
#pragma unroll
      for (int e = 0; e < 6; ++e) pp[e] = st.par[e];
#pragma unroll
      for (int e = 0; e < 21; ++e) pe[e] = st.err[e];
      propagate(barrel, pp, pe, st.chg, d.propagate_to, a.inter_pflags, a);
      Window w;
      hit_window(d, pp, pe, w);
      // find_tracks_handle_missed_layers (MkBuilder.cc:1568-1630)
      if (barrel && hypot_ref(pp[0], pp[1]) < d.rin) {
        const int k = append_node(a, seed, &s_nnodes[g], -2, layer, st.last);
        if (k >= 0) st.last = k;
        add_hit_counts(st, -2, 0.f);
        xkind[lane] = 2;
      } else if (w.wsr == MKF_WSR_OUTSIDE) {
        xkind[lane] = 1;
      } else {
        search = true;
        pt_l = fabsf(1.0f / pp[3]);
        nh = scan_window(d, w, a.bins, a.phis, a.qs, a.mask, [&](int gi) { Gh[lane][nh++] = gi - d.hit_off; });
        float* xs = &X[lane * kW];                       // words 0-35 are free until the end of (a)
#pragma unroll
        for (int e = 0; e < 6; ++e) xs[e] = pp[e];
#pragma unroll
        for (int e = 0; e < 21; ++e) xs[6 + e] = pe[e];
        xs[27] = __int_as_float(st.chg);
        xs[kXCut] = dyn_chi2_cut(d, a.chi2_cut, pp[3], pp[5]);
        xs[kXOff] = __int_as_float(d.hit_off);
        xs[kXBar] = __int_as_float(barrel ? 1 : 0);
        if (a.prop_to_hit) {                             // sin, cos of phi and theta for every pair's propagation
          sincosf(pp[4], &xs[kXTrig], &xs[kXTrig + 1]);
          sincosf(pp[5], &xs[kXTrig + 2], &xs[kXTrig + 3]);
        }
        int fake = (st.ninside + st.ntail < a.max_holes && st.ntail < a.max_consec) ? -1 : -2;
        if (w.wsr == MKF_WSR_EDGE) fake = -3;
        else if (a.dead) {          // XWsrResult::m_in_gap: a dead bin of the central q row in the window (MkFinder.cc:451-462)
          const unsigned char* __restrict__ row = a.dead + d.bin_off + q_bin_checked(d, w.q) * kNPhi;
          for (int pi = w.pb1; pi < w.pb2 && !gap; ++pi) gap = row[pi & 0xff] != 0;
        }
        const int nt = fake == -1 ? st.ntail + 1 : st.ntail;
        fcode[lane] = fake;
        X[lane * kW + kXScore] = score_calc(st.nfound, nt, 0, st.ninside, st.chi2 < 0 ? 0.f : st.chi2, pt_l, true);
      }
    }
    // (a2) inclusive prefix sum of nh over the wavefront (the workgroup is one wavefront)
    int incl = nh;
#pragma unroll
    for (int o = 1; o < kLanes; o <<= 1) {
      const int v = __shfl_up(incl, o, kLanes);
      if (lane >= o) incl += v;
    }
    X[lane * kW + kXPre] = __int_as_float(incl - nh);
    const int total = __shfl(incl, kLanes - 1, kLanes);
    // Each pair's owner lane, one byte per pair (at most kLanes * kHitIdxMax), in the score
    // rows, which (a3) fills only after this phase.
    unsigned char* owner = reinterpret_cast<unsigned char*>(&Es[0][0]);
    static_assert(sizeof(Es) >= kLanes * kHitIdxMax, "owner table fits the score rows");
    for (int k = 0; k < nh; ++k) owner[incl - nh + k] = (unsigned char)lane;
    __syncthreads();
    for (int j = lane; j < total; j += kLanes) {
      const int lo = owner[j];
      const float* xs = &X[lo * kW];
      const int o = lo, k = j - __float_as_int(xs[kXPre]);
      // The owner's layer: in a batch of events, lanes of other seeds hold other events' layers.
      const bool ob = __float_as_int(xs[kXBar]) != 0;
      float mp[3], me[6];
      load_hit9(a.shits + (size_t)(__float_as_int(xs[kXOff]) + Gh[o][k]) * 9, mp, me);
      float q[6], qe[21], pe[21];
#pragma unroll
      for (int e = 0; e < 6; ++e) q[e] = xs[e];
#pragma unroll
      for (int e = 0; e < 21; ++e) qe[e] = pe[e] = xs[6 + e];
      if (a.prop_to_hit)
        propagate(ob, q, qe, __float_as_int(xs[27]), ob ? hypot_ref(mp[0], mp[1]) : mp[2], a.intra_pflags, a,
                  &xs[kXTrig]);
      const float c2 = fabsf(ob ? kalman_barrel<true, false>(q, qe, mp, me)
                                : kalman_endcap<true, false>(q, qe, mp, me));
      const int gi = __float_as_int(xs[kXOff]) + Gh[o][k];
      const bool acc = c2 < xs[kXCut] && strip_q_compatible(ob, pe, q, mp, me) &&
                       (!a.charge || pass_strip_charge(ob, a.charge[gi], q, me));
      Gc[o][k] = acc ? c2 : -1.f;
      if (STD && acc) {
        // getScoreCand of the new candidate takes the pT of its updated state (m_update_param_foo)
        if (ob)
          kalman_barrel<false, true>(q, qe, mp, me);
        else
          kalman_endcap<false, true>(q, qe, mp, me);
        Gp[o][k] = fabsf(1.0f / q[3]);
      }
    }
    __syncthreads();
    // (a3) the lane's best K records, sorted by score, in scan order among equals: the seed's top K never takes
    // a record that K records of its own lane beat
    float rs[kS];
    int rh[kS], ne = 0;
    if (search) {
      int nacc = 0;
      for (int hc = 0; hc < nh; ++hc) {
        const float c2 = Gc[lane][hc];
        if (!(c2 >= 0.f)) continue;
        ++nacc;
        const float tot = st.chi2 + c2;
        const float sc = score_calc(st.nfound + 1, 0, 0, st.ninside + st.ntail, tot < 0 ? 0.f : tot,
                                    STD ? Gp[lane][hc] : pt_l, true);
        int pos = 0;                                    // kept records with score >= sc
#pragma unroll
        for (int q = 0; q < kS; ++q) pos += (q < ne && !(rs[q] < sc)) ? 1 : 0;
        if (pos >= K) continue;
#pragma unroll
        for (int q = kS - 1; q > 0; --q) {
          rs[q] = q > pos ? rs[q - 1] : rs[q];
          rh[q] = q > pos ? rh[q - 1] : rh[q];
        }
#pragma unroll
        for (int q = 0; q < kS; ++q) {
          rs[q] = q == pos ? sc : rs[q];
          rh[q] = q == pos ? hc : rh[q];
        }
        if (ne < K) ++ne;
      }
      if (gap && nacc == 0) {      // dead module, no hit taken: -7, which is no hole (MkFinder.cc:1092-1096, 1263-1267)
        fcode[lane] = -7;
        X[lane * kW + kXScore] = score_calc(st.nfound, st.ntail, 0, st.ninside, st.chi2 < 0 ? 0.f : st.chi2, pt_l, true);
      }
    }
    // STD: a searching lane's new candidates start from its state at the layer, which (a1) left in words
    // 0-26; the others (held back, stopped, idle) keep their own.
    if (STD && search)
      put_counts(&X[lane * kW], st);
    else
      put(&X[lane * kW], st);
    __syncthreads();
    // ---- (b) CandCloner::ProcessSeedRange.  Each lane's entries are its records, its invalid-hit record and (STD,
    // where find_tracks_handle_missed_layers runs before FindCandidates) itself when held back; K times the group
    // takes the best of the lanes' best remaining ones.  (One lane per seed merging all records took 28k of a
    // wavefront's 104k cycles per layer, this and the layout below 10k: 15.7 -> 13.4 ms for 500k seeds.)
    {
      const int l0 = g * kS;
      const int fc = fcode[lane];
      uint64_t fake = 0;                             // the lane's one entry beside its records
      if (fc && !(STD && fc == -2)) fake = rank_key(X[lane * kW + kXScore], kGenFake + c);
      if (STD && xkind[lane] == 1) fake = rank_key(X[lane * kW + 29], c);
      const int rounds = g < kG ? K : 0;
      for (int r = 0; r < K; ++r) {
        const uint64_t rec = ne > 0 ? rank_key(rs[0], kGenRec + rh[0] * kSMax + c) : 0;
        const uint64_t own = rec > fake ? rec : fake;
        const uint64_t best = group_max<kS>(own, l0, c);
        if (r < rounds && c == 0) {                  // the r-th ranked entry; word 1: 0 when there is none
          Es[l0 + r][0] = best ? key_score(best) : 0.f;
          Es[l0 + r][1] = __int_as_float(best ? key_gen(best) + 1 : 0);
        }
        if (own && own == best) {
          if (rec > fake) {
#pragma unroll
            for (int q = 0; q + 1 < kS; ++q) {
              rs[q] = rs[q + 1];
              rh[q] = rh[q + 1];
            }
            --ne;
          } else {
            fake = 0;
          }
        }
      }
      if (STD) {
        // the first entry with a -2 hit in ranked order: a stopped replica or a -2 invalid-hit entry
        uint64_t shrt = 0;
        if (xkind[lane] == 2) shrt = rank_key(X[lane * kW + 29], c);
        else if (fc == -2) shrt = rank_key(X[lane * kW + kXScore], kGenFake + c);
        shrt = group_max<kS>(shrt, l0, c);
        if (c == 0 && g < kG) {
          Es[l0][2] = shrt ? key_score(shrt) : 0.f;
          Es[l0][3] = __int_as_float(shrt ? key_gen(shrt) + 1 : 0);
        }
      }
    }
    __syncthreads();
    // One lane per seed lays out the next candidates.
    if (c == 0 && s_merge[g]) {
      const int l0 = g * kS;
      float tsc[kS];
      int tg[kS];                                    // generation places of the ranked entries, -1 past the last
      int nt = 0;
#pragma unroll
      for (int q = 0; q < kS; ++q) {
        const bool in = q < K;
        tsc[q] = in ? Es[l0 + q][0] : 0.f;
        tg[q] = in ? __float_as_int(Es[l0 + q][1]) - 1 : -1;
        nt += tg[q] >= 0 ? 1 : 0;
      }
      // D's word of the ranked entry q
      auto entry = [&](int gen, int q) {
        if (gen < kGenRec) return 1 | gen << 2;
        if (gen < kGenFake) return 2 | (gen & (kSMax - 1)) << 2 | q << 5 | (gen - kGenRec) / kSMax << 8;
        return 3 | (gen & (kSMax - 1)) << 2;
      };
      static_assert((kGenRec & (kSMax - 1)) == 0 && (kGenFake & (kSMax - 1)) == 0, "the slot is gen's low bits");
      if (STD) {
        // MkBuilder.cc:1776-1828: the kept entries in ranked order become the next candidates; the first -2
        // entry is met if it ranks before the K-th of them
        int np = 0;
#pragma unroll
        for (int q = 0; q < kS; ++q)
          if (tg[q] >= 0) D[g][np++] = entry(tg[q], q);
        const float bsc = Es[l0][2];
        const int bgen = __float_as_int(Es[l0][3]) - 1;
        if (bgen >= 0) {
          bool met = nt < K;
          if (!met) {
            const float sK = Es[l0 + K - 1][0];
            const int gK = __float_as_int(Es[l0 + K - 1][1]) - 1;
            met = bsc > sK || (bsc == sK && bgen < gK);
          }
          if (met && bsc > s_bsc[g]) {                   // best short candidate
            Cand b;
            get(&X[(l0 + (bgen & (kSMax - 1))) * kW], b);
            if (bgen >= kGenFake) {                      // an invalid-hit entry; a stopped replica has its -2
              const int k = append_node(a, seed, &s_nnodes[g], -2, layer, b.last);
              if (k >= 0) b.last = k;
              add_hit_counts(b, -2, 0.f);
            }
            b.score = bsc;
            put(a.bs + (size_t)seed * kBsW, b);
            s_bsc[g] = bsc;
            s_bs[g] = 1;
          }
        }
        if (nt == 0 && bgen < 0)                         // no entry at all: the candidates stay
          for (int i = 0; i < s_ncand[g]; ++i) D[g][np++] = 1 | i << 2;
        s_nnew[g] = np;
      } else {
      int np = 0;
      unsigned xm = 0;                                // held-back slots, lowest first
      for (int s = 0; s < kS; ++s)
        if (xkind[g * kS + s]) xm |= 1u << s;
      if (nt == 0) {
        for (; xm; xm &= xm - 1) {
          D[g][np] = 1 | (__ffs(xm) - 1) << 2;
          ++np;
        }
      } else {
        bool full = false;
#pragma unroll
        for (int q = 0; q < kS; ++q) {
          if (tg[q] < 0 || full) continue;
          const float sc = tsc[q];
          const int slot = tg[q] & (kSMax - 1);
          if (tg[q] >= kGenFake && fcode[l0 + slot] == -2) {   // a short candidate
            if (sc > s_bsc[g]) {                      // best short candidate
              Cand b;
              get(&X[(l0 + slot) * kW], b);
              const int k = append_node(a, seed, &s_nnodes[g], -2, layer, b.last);
              if (k >= 0) b.last = k;
              add_hit_counts(b, -2, 0.f);
              b.score = sc;
              put(a.bs + (size_t)seed * kBsW, b);
              s_bsc[g] = b.score;
              s_bs[g] = 1;
            }
            continue;
          }
          while (xm && X[(l0 + __ffs(xm) - 1) * kW + 29] > sc && np < K) {
            D[g][np] = 1 | (__ffs(xm) - 1) << 2;
            ++np;
            xm &= xm - 1;
          }
          if (np >= K) {
            full = true;
            continue;
          }
          D[g][np] = entry(tg[q], q);
          ++np;
        }
        for (; xm && np < K; xm &= xm - 1) {
          D[g][np] = 1 | (__ffs(xm) - 1) << 2;
          ++np;
        }
      }
      s_nnew[g] = np;
      }
    }
    __syncthreads();
    // ---- (c) new candidates; UpdateWithLastHit for those that took a hit
    if (s_merge[g] && gvalid) {
      if (c < s_nnew[g]) {
        const int dd = D[g][c];
        const int kind = dd & 3, l = g * kS + ((dd >> 2) & 7), rank = (dd >> 5) & 7, hc = dd >> 8;
        get(&X[l * kW], st);
        if (kind != 1) {
          // kind 2: the slot lane's window hit hc; kind 3: its invalid-hit record
          const int val = kind == 2 ? d.hit_off + Gh[l][hc] : fcode[l];
          const int hit = kind == 2 ? a.ranks[val] : val;
          const int k = append_node(a, seed, &s_nnodes[g], hit, layer, st.last);
          if (k >= 0) st.last = k;
          add_hit_counts(st, hit, kind == 2 ? Gc[l][hc] : 0.f);
          st.score = kind == 2 ? Es[g * kS + rank][0] : X[l * kW + kXScore];
          if (kind == 2) {
            float mp[3], me[6];
            load_hit9(a.shits + (size_t)val * 9, mp, me);
            if (a.prop_to_hit)
              propagate(barrel, st.par, st.err, st.chg, barrel ? hypot_ref(mp[0], mp[1]) : mp[2],
                        STD ? a.intra_pflags : a.inter_pflags, a);
            if (barrel)
              kalman_barrel<false, true>(st.par, st.err, mp, me);
            else
              kalman_endcap<false, true>(st.par, st.err, mp, me);
            if (st.par[3] < 0.f) {
              st.chg = -st.chg;
              st.par[3] = -st.par[3];
            }
          }
        }
      }
    }
    __syncthreads();
    if (c == 0 && s_merge[g]) s_ncand[g] = s_nnew[g];
  }

  // ---- MergeCandsAndBestShortOne(update_score, sort) and output
  __syncthreads();
  const bool valid = gvalid && c < s_ncand[g];
  if (valid) st.score = cand_score(st);
  put(&X[lane * kW], st);
  __syncthreads();
  int (*O)[kS + 1] = reinterpret_cast<int (*)[kS + 1]>(&Gh[0][0]);   // final order (kS = best short); Gh is free
  static_assert(kGA * (kS + 1) <= kLanes * kHitIdxMax, "the final order must fit in Gh");
  if (c == 0 && gvalid) {
    const int nc = s_ncand[g];
    int ord[kS + 1];
    int m = 0;
    for (int i = 0; i < nc; ++i) {                            // stable insertion sort by score
      const float sc = X[(g * kS + i) * kW + 29];
      int pos = m;
      while (pos > 0 && X[(g * kS + ord[pos - 1]) * kW + 29] < sc) {
        ord[pos] = ord[pos - 1];
        --pos;
      }
      ord[pos] = i;
      ++m;
    }
    if (s_bs[g]) {
      // The best short candidate's score is recomputed only alongside the
      // candidates' (HitStructures.cc:515-521); alone it keeps its finding score.
      Cand b;
      get(a.bs + (size_t)seed * kBsW, b);
      if (m > 0) b.score = cand_score(b);
      put(a.bs + (size_t)seed * kBsW, b);
      if (m > 0) {
        if (b.score > X[(g * kS + ord[m - 1]) * kW + 29]) {
          int ci = 0;
          while (X[(g * kS + ord[ci]) * kW + 29] > b.score) ++ci;
          if (m >= K) --m;
          for (int j = m; j > ci; --j) ord[j] = ord[j - 1];
          ord[ci] = kS;
          ++m;
        }
      } else {
        ord[m++] = kS;
      }
    }
    for (int i = 0; i < m; ++i) O[g][i] = ord[i];
    s_nout[g] = m;
    a.n_cands[seed] = m;
  } else if (c == 0 && gin) {      // layer_base outside the event of hits: no candidates
    s_nout[g] = 0;
    a.n_cands[seed] = 0;
  }
  __syncthreads();
  if (!gin || c >= K) return;
  const int L = a.n_layers;
  int* hot = a.hot + ((size_t)c * L) * N + seed;
  for (int l = 0; l < L; ++l) hot[(size_t)l * N] = -9;
  if (c >= s_nout[g]) {
    a.score[c * N + seed] = kScoreWorst;
    a.n_found[c * N + seed] = 0;
    return;
  }
  Cand o;
  get(O[g][c] == kS ? a.bs + (size_t)seed * kBsW : &X[(g * kS + O[g][c]) * kW], o);
#pragma unroll
  for (int e = 0; e < 6; ++e) a.par[((size_t)c * 6 + e) * N + seed] = o.par[e];
#pragma unroll
  for (int e = 0; e < 21; ++e) a.err[((size_t)c * 21 + e) * N + seed] = o.err[e];
  a.chg[c * N + seed] = o.chg;
  a.chi2[c * N + seed] = o.chi2;
  a.score[c * N + seed] = o.score;
  a.n_found[c * N + seed] = o.nfound;
  const int4* nodes = a.nodes + (size_t)seed * a.node_cap;
  for (int k = o.last, steps = 0; k >= 0 && steps < a.node_cap; k = nodes[k].z, ++steps) {
    const int4 nd = nodes[k];
    if (nd.y >= 0 && nd.y < L && hot[(size_t)nd.y * N] == -9) hot[(size_t)nd.y * N] = nd.x;
  }
}

}  // namespace

namespace {

int find_combinatorial(mkf_context* c, mkf_event_of_hits* h, const mkf_ce_batch* b, void* stream, bool standard) {
  CHECK(set_device(c));
  if (!h || !b) return fail(MKF_ERR_INVALID_ARG, "NULL argument");
  if (h->ctx != c) return fail(MKF_ERR_INVALID_ARG, "event of hits belongs to another context");
  if (!h->loaded) return fail(MKF_ERR_INVALID_ARG, "event of hits not loaded");
  if (b->n_seeds < 0) return fail(MKF_ERR_INVALID_ARG, "n_seeds < 0");
  for (const LayerDev& ld : h->layers)
    if (ld.n_hits > kMaxLayerHits)
      return fail(MKF_ERR_INVALID_ARG, "a layer holds %d hits, above %d", ld.n_hits, kMaxLayerHits);
  const int LE = b->n_layers ? b->n_layers : h->n_layers;   // layers per event
  if (LE < 1 || LE > h->n_layers || LE > MKF_MAX_FIND_LAYERS)
    return fail(MKF_ERR_INVALID_ARG, "n_layers %d outside [1, min(%d, %d)]", LE, h->n_layers, MKF_MAX_FIND_LAYERS);
  if (b->first_layer < 1 || b->first_layer > LE)
    return fail(MKF_ERR_INVALID_ARG, "first_layer %d outside [1, %d]", b->first_layer, LE);
  if (!b->layer_base && LE != h->n_layers)
    return fail(MKF_ERR_INVALID_ARG, "n_layers %d below the event of hits' %d needs layer_base", LE, h->n_layers);
  if (b->max_cands < 1 || b->max_cands > MKF_CE_MAX_CANDS)
    return fail(MKF_ERR_INVALID_ARG, "max_cands must be in [1, %d]", MKF_CE_MAX_CANDS);
  if (((b->pflags | b->intra_pflags) & MKF_PF_APPLY_MATERIAL) && !c->d_rl)
    return fail(MKF_ERR_INVALID_ARG, "material requested but the context has no material grid");
  if (b->n_seeds == 0) return MKF_OK;
  const size_t N = b->n_seeds, K = b->max_cands, L = LE;
  if (K * 21 * N * 4 >= ((size_t)1 << 31) || K * L * N >= ((size_t)1 << 31))
    return fail(MKF_ERR_INVALID_ARG, "batch too large");
  CHECK(check_dev(b->seed_par, 6 * N * 4, "seed_par"));
  CHECK(check_dev(b->seed_err, 21 * N * 4, "seed_err"));
  CHECK(check_dev(b->seed_chg, N * 4, "seed_chg"));
  CHECK(check_dev(b->seed_hits, (size_t)b->first_layer * N * 4, "seed_hits"));
  CHECK(check_dev(b->n_cands, N * 4, "n_cands"));
  CHECK(check_dev(b->par, K * 6 * N * 4, "par"));
  CHECK(check_dev(b->err, K * 21 * N * 4, "err"));
  CHECK(check_dev(b->chg, K * N * 4, "chg"));
  CHECK(check_dev(b->chi2, K * N * 4, "chi2"));
  CHECK(check_dev(b->score, K * N * 4, "score"));
  CHECK(check_dev(b->n_found, K * N * 4, "n_found"));
  CHECK(check_dev(b->hot_idx, K * L * N * 4, "hot_idx"));
  if (b->layer_base) CHECK(check_dev(b->layer_base, N * 4, "layer_base"));
  const int node_cap = b->first_layer + 3 * kSMax * (LE - b->first_layer) + kSMax;
  const size_t need = ((size_t)node_cap + kBsW / 4) * N;    // nodes, then the best short candidates
  hipStream_t st = (hipStream_t)stream;
  std::lock_guard<std::mutex> lk(h->ce_mu);
  CHECK(scratch_acquire(h->ce_done, st));
  if (need > h->ce_node_cap) {
    HIP_TRY(hipStreamSynchronize(st));
    if (h->d_ce_nodes) HIP_TRY(hipFree(h->d_ce_nodes));
    h->d_ce_nodes = nullptr;
    h->ce_node_cap = 0;
    HIP_TRY(hipMalloc(&h->d_ce_nodes, need * sizeof(int4)));
    h->ce_node_cap = need;
  }
  CeArgs a;
  a.n = b->n_seeds;
  a.n_layers = LE;
  a.eoh_layers = h->n_layers;
  a.layer_base = b->layer_base;
  a.first_layer = b->first_layer;
  a.max_cands = b->max_cands;
  a.max_holes = b->max_holes;
  a.max_consec = b->max_consec_holes;
  a.prop_to_hit = b->prop_to_hit;
  a.intra_pflags = b->intra_pflags;
  a.inter_pflags = b->pflags;
  a.chi2_cut = b->chi2_cut;
  a.bfield = c->bfield;
  a.mat = mat_of(c);
  a.seed_par = b->seed_par; a.seed_err = b->seed_err; a.seed_chg = b->seed_chg; a.seed_hits = b->seed_hits;
  a.n_cands = b->n_cands; a.par = b->par; a.err = b->err; a.chg = b->chg; a.chi2 = b->chi2; a.score = b->score;
  a.n_found = b->n_found; a.hot = b->hot_idx;
  a.nodes = reinterpret_cast<int4*>(h->d_ce_nodes);
  a.node_cap = node_cap;
  a.bs = reinterpret_cast<float*>(a.nodes + (size_t)node_cap * N);
  a.layers = h->d_layers; a.bins = h->d_bins; a.phis = h->d_phis; a.qs = h->d_qs; a.shits = h->d_shits;
  a.mask = h->mask();
  a.charge = h->charge();
  a.dead = h->dead();
  a.ranks = h->d_ranks;
  const mkf_find_shape sh = c->find_shape[standard ? 1 : 0];
  const int slots = sh.slots ? sh.slots : (b->max_cands <= 6 ? 6 : 8);
  if (slots < b->max_cands) return fail(MKF_ERR_INVALID_ARG, "find shape: %d slots < max_cands %d", slots, b->max_cands);
  using Kernel = void (*)(CeArgs);
  static const Kernel kernels[8] = {
      k_find_clone_engine<6, false, 2>, k_find_clone_engine<6, false, 1>, k_find_clone_engine<6, true, 2>,
      k_find_clone_engine<6, true, 1>,  k_find_clone_engine<8, false, 2>, k_find_clone_engine<8, false, 1>,
      k_find_clone_engine<8, true, 2>,  k_find_clone_engine<8, true, 1>};
  const int sel = (slots == 8 ? 4 : 0) | (standard ? 2 : 0) | (sh.waves_per_simd == 1 ? 1 : 0);
  // Wavefronts a CU holds, by the registers and LDS the variant was compiled to (8 and, standard, 6; 4 of <8, false, 1>).
  int per_cu = c->ce_per_cu[sel].load(std::memory_order_relaxed);
  if (!per_cu) {
    HIP_TRY(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernels[sel], kLanes, 0));
    per_cu = std::max(1, per_cu);
    c->ce_per_cu[sel].store(per_cu, std::memory_order_relaxed);
  }
  a.spw = seeds_per_wave(N, kLanes / slots, c->num_cus, per_cu);
  const int grid = (int)((N + a.spw - 1) / a.spw);
  hipLaunchKernelGGL(kernels[sel], dim3(grid), dim3(kLanes), 0, st, a);
  HIP_TRY(hipGetLastError());
  return scratch_release(h->ce_done, st);
}

}  // namespace

extern "C" int mkf_find_tracks_clone_engine(mkf_context* c, mkf_event_of_hits* h, const mkf_ce_batch* b,
                                            void* stream) {
  return find_combinatorial(c, h, b, stream, false);
}

extern "C" int mkf_find_tracks_standard(mkf_context* c, mkf_event_of_hits* h, const mkf_ce_batch* b, void* stream) {
  return find_combinatorial(c, h, b, stream, true);
}

extern "C" int mkf_set_find_shape(mkf_context* c, int standard, const mkf_find_shape* shape) {
  if (!c || !shape) return fail(MKF_ERR_INVALID_ARG, "NULL argument");
  if (shape->slots != 0 && shape->slots != 6 && shape->slots != 8)
    return fail(MKF_ERR_INVALID_ARG, "find shape: slots must be 0, 6 or 8");
  if (shape->waves_per_simd != 1 && shape->waves_per_simd != 2)
    return fail(MKF_ERR_INVALID_ARG, "find shape: waves_per_simd must be 1 or 2");
  std::lock_guard<std::mutex> lk(c->mu);
  c->find_shape[standard ? 1 : 0] = *shape;
  return MKF_OK;
}

extern "C" int mkf_get_find_shape(mkf_context* c, int standard, mkf_find_shape* shape) {
  if (!c || !shape) return fail(MKF_ERR_INVALID_ARG, "NULL argument");
  std::lock_guard<std::mutex> lk(c->mu);
  *shape = c->find_shape[standard ? 1 : 0];
  return MKF_OK;
}

// Every shape valid for the batch's max_cands, timed on the batch: one warm-up launch of each, then reps
// timed launches; the fastest stays in the context.  Results do not depend on the shape.
extern "C" int mkf_autotune_find(mkf_context* c, mkf_event_of_hits* h, const mkf_ce_batch* b, int standard, int reps,
                                 mkf_find_shape* best, float* best_ms, void* stream) {
  if (!c || !b) return fail(MKF_ERR_INVALID_ARG, "NULL argument");
  if (reps < 1 || reps > 100) return fail(MKF_ERR_INVALID_ARG, "reps must be in [1, 100]");
  CHECK(set_device(c));
  hipStream_t st = (hipStream_t)stream;
  std::vector<mkf_find_shape> cand;
  for (int slots : {6, 8})
    if (slots >= b->max_cands)
      for (int w : {2, 1}) cand.push_back(mkf_find_shape{slots, w});
  hipEvent_t e0, e1;
  HIP_TRY(hipEventCreate(&e0));
  HIP_TRY(hipEventCreate(&e1));
  const mkf_find_shape keep = c->find_shape[standard ? 1 : 0];
  float best_t = 1e30f;
  mkf_find_shape best_s = keep;
  int rc = MKF_OK;
  for (const mkf_find_shape& s : cand) {
    c->find_shape[standard ? 1 : 0] = s;
    rc = find_combinatorial(c, h, b, stream, standard != 0);                  // warm-up
    if (rc != MKF_OK) break;
    if (hipEventRecord(e0, st) != hipSuccess) { rc = fail(MKF_ERR_HIP, "hipEventRecord"); break; }
    for (int r = 0; r < reps && rc == MKF_OK; ++r) rc = find_combinatorial(c, h, b, stream, standard != 0);
    if (rc != MKF_OK) break;
    float ms = 0.f;
    if (hipEventRecord(e1, st) != hipSuccess || hipEventSynchronize(e1) != hipSuccess ||
        hipEventElapsedTime(&ms, e0, e1) != hipSuccess) {
      rc = fail(MKF_ERR_HIP, "timing the find shapes");
      break;
    }
    ms /= reps;
    if (ms < best_t) {
      best_t = ms;
      best_s = s;
    }
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  c->find_shape[standard ? 1 : 0] = rc == MKF_OK ? best_s : keep;
  if (rc != MKF_OK) return rc;
  if (best) *best = best_s;
  if (best_ms) *best_ms = best_t;
  return MKF_OK;
}
