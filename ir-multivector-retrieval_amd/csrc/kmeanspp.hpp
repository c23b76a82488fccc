// kmeanspp.hpp — k-means++ seeding of every subspace at once
// (src/tac/kmeans.zig:106-136, src/util/rng.zig:22-82).  Included once, by
// tac_gpu.hip, after pq_kernels.hpp.
//
// Per subspace m the reference draws with std.Random.DefaultPrng seeded with
// seed +% m (src/index/pq.zig:323):
//   c0 = row intRangeLessThan(0, n); w_i = l2sq(x_i, c0)
//   for c = 1 .. K-1:  idx = weightedSample(w); c_c = row idx;
//                      w_i = min(w_i, l2sq(x_i, c_c))   (strict <)
// weightedSample folds the weights sequentially in f64 (total, then the
// running cum), draws u = float(f64) * total and returns the first i with
// u < cum_i (last positive index if none).
//
// The GPU sums the weights in parallel, in any order.  For non-negative
// terms every rounded sum (the reference's sequential fold or ours) lies
// within i * 2^-53 * P_i of the exact prefix P_i, so the two differ by at
// most band_i = 2.1 (i + 1) 2^-53 P_i.  When the draw clears the bands of the
// candidate index on both sides the reference's pick is determined;
// otherwise the subspace falls back to the exact sequential fold on one wave.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "cand_rules.hpp"
#include "kpp_rules.hpp"

namespace tacgpu {

struct KppState {
  uint64_t s[4];
  double r;          // draw of the current round
  uint32_t chosen;   // row picked in the current round
  uint32_t fallback; // 1: the parallel decision was inconclusive this round
  int32_t err;       // 0 or a tac_status (NonFinite / AllZero)
  uint32_t pad;
};

constexpr uint32_t kKppBlock = 4096;  // rows of a kpp_round_kernel block
// Work-items of a kpp_round_kernel block, 8 rows each.
constexpr uint32_t kKppThreads = 512;

// A subspace's seeding state between launches, in two copies: launch l reads
// copy l & 1 and block 0 of the subspace writes the other.
struct KppSeed {
  uint64_t s[4];       // PRNG
  double r;            // the last draw
  uint32_t chosen;     // the row of codeword `next`, when it is known (pending 2, next 0)
  uint32_t next;       // codewords written
  uint32_t pending;    // 1: the draw of codeword `next` was inconclusive and waits for
                       // kpp_exact_kernel; 2: that kernel has set `chosen`
  int32_t err;         // 0 or a tac_status (NonFinite / AllZero)
  uint32_t patch_run;  // the run whose weights are in the patch instead of w, or kKppNone
  uint32_t patch_sel;  // which half of the patch
  uint32_t bsel;       // which half of bsum holds the last round's sums
  uint32_t pad;
};
constexpr uint32_t kKppNone = 0xFFFFFFFFu;

constexpr uint32_t kKppRun = 512;  // rows of a wave, whose weights have a sum of their own
constexpr uint32_t kKppRuns = kKppBlock / kKppRun;

// Inclusive f64 sum over the wave's lanes (DPP row shifts and broadcasts): the
// same instructions in the same order for the same values in every block.
__device__ __forceinline__ double wave_inclusive_sum_f64(double v) {
  auto step = [&](uint64_t moved) { v += __longlong_as_double((long long)moved); };
  step(dpp_u64<0x111, 0xF>((uint64_t)__double_as_longlong(v)));
  step(dpp_u64<0x112, 0xF>((uint64_t)__double_as_longlong(v)));
  step(dpp_u64<0x114, 0xF>((uint64_t)__double_as_longlong(v)));
  step(dpp_u64<0x118, 0xF>((uint64_t)__double_as_longlong(v)));
  step(dpp_u64<0x142, 0xA>((uint64_t)__double_as_longlong(v)));
  step(dpp_u64<0x143, 0xC>((uint64_t)__double_as_longlong(v)));
  return v;
}
__device__ __forceinline__ double readlane_f64(double v, uint32_t l) {
  return __longlong_as_double((long long)readlane_u64((uint64_t)__double_as_longlong(v), l));
}
// The lane below's value (0 in lane 0): exclusive sums from inclusive ones.
// Inclusive minus own would carry a rounding error of the own value's size,
// which the bands of kpp_decides, relative to the prefix, do not cover.
__device__ __forceinline__ double wave_below_f64(double v) {
  return __longlong_as_double((long long)dpp_u64<0x138, 0xF>((uint64_t)__double_as_longlong(v)));
}

// What the draw of a round found.
struct KppDraw {
  uint32_t row;  // kKppNone: left open
  uint32_t run;  // the run of kKppRun rows that it read
  int32_t err;
  double r;
};

// Runs up to which every block draws for itself (kpp_round_kernel): a lane
// then holds its share of the sums in registers.
constexpr uint32_t kKppLaneRuns = 8;
constexpr uint32_t kKppFusedRuns = kKppLaneRuns * kWave;

// The draw from the weights' sums per run and the weights, by one wave; lane l
// owns the runs from l * per on (per = ceil(n_runs / 64)).  FUSED: n_runs is
// at most kKppFusedRuns; else `share` is the lane's total.  The bands of
// kpp_decides hold for sums in any order, formed by additions only.
template <bool FUSED>
__device__ __forceinline__ KppDraw kpp_draw_wave(const double* __restrict__ sums, uint32_t n_runs,
                                                 double share, const float* wm,
                                                 const float* patch, uint32_t patch_run,
                                                 uint64_t n, uint64_t* prng, bool leave_open) {
  const uint32_t lane = threadIdx.x % kWave;
  KppDraw out{kKppNone, kKppNone, 0, 0.0};
  const uint32_t per = (n_runs + kWave - 1) / kWave;
  const uint32_t q0 = lane * per, q1 = q0 + per < n_runs ? q0 + per : n_runs;
  double mine[kKppLaneRuns];
  if constexpr (FUSED) {
#pragma unroll
    for (uint32_t j = 0; j < kKppLaneRuns; ++j) mine[j] = q0 + j < q1 ? sums[q0 + j] : 0.0;
    share = 0.0;
#pragma unroll
    for (uint32_t j = 0; j < kKppLaneRuns; ++j) share += mine[j];
  }
  const double incl = wave_inclusive_sum_f64(share);
  const double tot = readlane_f64(incl, kWave - 1);
  if (!(tot > 0.0)) {
    out.err = 10;  // AllZero
    return out;
  }
  out.r = kpp_float64(prng);
  const double u = out.r * tot;
  const uint64_t over = __ballot(q0 < n_runs && u < incl);
  if (leave_open || !over) return out;  // u at or beyond the total: the tail rule decides
  const uint32_t fl = (uint32_t)__builtin_ctzll(over);
  // the run within that lane's share (its last when rounding leaves none)
  const uint32_t f0 = fl * per, f1 = f0 + per < n_runs ? f0 + per : n_runs;
  double before = fl ? readlane_f64(incl, fl - 1) : 0.0;
  uint32_t run = f0;
  if constexpr (FUSED) {
#pragma unroll
    for (uint32_t j = 0; j + 1 < kKppLaneRuns; ++j) {
      const double next = before + readlane_f64(mine[j], fl);
      const bool on = run == f0 + j && run + 1 < f1 && !(u < next);
      before = on ? next : before;
      run += on ? 1u : 0u;
    }
  } else {
    for (uint32_t base = f0;; base += kWave) {
      const double x = base + lane < f1 ? sums[base + lane] : 0.0;
      const double within = wave_inclusive_sum_f64(x);
      const double end = before + within;
      const uint32_t last = f1 - 1 - base < kWave ? f1 - 1 - base : kWave - 1;
      const uint64_t in = __ballot(base + lane < f1 && u < end);
      if (in || base + kWave >= f1) {
        const uint32_t at = in ? (uint32_t)__builtin_ctzll(in) : last;
        run = base + at;
        before = before + (at ? readlane_f64(within, at - 1) : 0.0);
        break;
      }
      before = readlane_f64(end, kWave - 1);
    }
  }
  out.run = run;
  const uint64_t lo = (uint64_t)run * kKppRun;
  const float* dw = run == patch_run ? patch : wm + lo;
  constexpr uint32_t kPer = kKppRun / kWave;
  double v[kPer], sum = 0.0;
#pragma unroll
  for (uint32_t q = 0; q < kPer; ++q) {
    const uint32_t o = lane * kPer + q;
    v[q] = lo + o < n ? (double)dw[o] : 0.0;
  }
#pragma unroll
  for (uint32_t q = 0; q < kPer; ++q) sum += v[q];
  double p = before + wave_below_f64(wave_inclusive_sum_f64(sum)), prev = p, at = p;
  uint32_t k = kKppNone;
#pragma unroll
  for (uint32_t q = 0; q < kPer; ++q) {
    const double b = p;
    p += v[q];
    if (k == kKppNone && lo + lane * kPer + q < n && u < p) {
      k = q;
      prev = b;
      at = p;
    }
  }
  const uint64_t hit = __ballot(k != kKppNone);
  if (!hit) return out;
  const uint32_t owner = (uint32_t)__builtin_ctzll(hit);
  const uint64_t i = lo + lane * kPer + k;
  const bool ok = lane == owner && kpp_decides(out.r, tot, n, i, prev, at);
  if (__ballot(ok)) out.row = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)i, (int)owner);
  return out;
}

// One seeding round of every subspace in one launch: the draw of codeword c
// from the weights that round c - 1 left, then round c's update: codeword c,
// w = min(w, l2sq(x, c_new)) (the first round assigns) and the weights' f64
// sums per run of kKppRun rows.
//
// The first wave of every block makes its subspace's draw itself, from the
// same inputs in the same order, so all of them agree on it without a launch
// in between: total and run from the runs' sums, then the row from the run's
// weights and the bands (kpp_decides).  A draw the bands leave open is marked
// pending: no block updates, later rounds pass the subspace by, and the host
// runs kpp_exact_kernel and the missing rounds.  The sums are double-buffered
// (bsel).  The weights are updated in place, except those of the drawn run,
// which the other blocks are reading: its wave writes them to one half of a
// per-subspace patch, where the next round finds them, and a run that leaves
// the patch goes back to w.  A non-finite weight stamps `bad` with its round,
// so that a stamp made while a round runs does not reach that round's draw.
//
// src[m][i] is the seed whose distance is w_i (w_i = l2sq(x_i, c_src)
// exactly: it is the minimum so far).  A seed c_new can lower w_i only if
// l2sq(x_i, c_new) < w_i, and by the candidate rule (cand_rules.hpp) it
// cannot when a rounded-down bound of ||c_src - c_new||^2 exceeds
// cand_radius(w_i): such weights are kept without reading the vector.
//
// Bound by latency: five dependent round trips (state, run sums, the run's
// weights, the drawn row, the rows it may lower).  As three launches (update,
// draw, exact fallback) a round of 117,645 rows x 16 subspaces took 22 us
// with its gaps beside the other 16's; this kernel takes 10.
//
// Without FUSED (more runs than kKppFusedRuns) kpp_draw_kernel has made the
// draw, and no run is being read by others.
template <int D, bool FUSED>
__global__ __launch_bounds__(kKppThreads) void kpp_round_kernel(
    const float* __restrict__ xs, float* __restrict__ w, uint16_t* __restrict__ src,
    double* __restrict__ bsum, uint64_t bstride, float* __restrict__ patch,
    uint32_t* __restrict__ bad, const KppSeed* __restrict__ st_in, KppSeed* __restrict__ st_out,
    float* __restrict__ cb, uint64_t n, uint32_t K, uint32_t NB, uint32_t exact_every) {
  constexpr int DP = Pad<D>::value;
  constexpr float g = cand_gamma(D);
  constexpr uint32_t kPer = kKppRun / kWave;
  __shared__ float lo_tab[1024];  // bound of ||c_j - c_new||^2 per earlier seed j
  __shared__ KppDraw s_draw;
  const uint32_t m = blockIdx.y, b = blockIdx.x, t = threadIdx.x;
  const KppSeed& S = st_in[m];
  const bool writer = b == 0 && t == 0;
  const uint32_t c = S.next, pending = S.pending;
  if (S.err || c == K || pending == 1) {
    if (writer) st_out[m] = S;
    return;
  }
  const uint32_t bsel = S.bsel, patch_sel = FUSED ? S.patch_sel : 0u;
  uint64_t prng[4];  // of the first wave
  double r = 0.0;
  const uint32_t run = b * kKppRuns + t / kWave;           // this wave's rows
  const uint64_t lo = (uint64_t)run * kKppRun + t % kWave;  // row j of the thread: lo + 64 j
  float* wm = w + (uint64_t)m * n;
  uint16_t* sm = src + (uint64_t)m * n;
  const float* xm = xs + (uint64_t)m * n * DP;
  float* cm = cb + (uint64_t)m * K * D;
  float* pm = patch + (uint64_t)m * 2 * kKppRun;
  const uint32_t n_runs = NB * kKppRuns;
  const bool own_patch = FUSED && S.patch_run == run;
  // The wave's own weights and sources, in flight under the draw.
  float wv[kPer];
  uint32_t sv[kPer];
#pragma unroll
  for (uint32_t j = 0; j < kPer; ++j) {
    const uint64_t i = lo + j * kWave;
    wv[j] = 0.0f;
    sv[j] = 0;
    if (c > 0 && i < n) {
      wv[j] = own_patch ? pm[patch_sel * kKppRun + j * kWave + t % kWave] : wm[i];
      sv[j] = sm[i];
    }
  }
  uint32_t chosen = S.chosen, drawn = kKppNone;
  if (FUSED && c > 0 && pending == 0) {
    if (t < kWave) {
#pragma unroll
      for (int q = 0; q < 4; ++q) prng[q] = S.s[q];
      const bool non_finite = bad[m] < c;  // rng.zig:62
      KppDraw d = kpp_draw_wave<true>(bsum + bsel * bstride + (uint64_t)m * n_runs, n_runs, 0.0,
                                      wm, pm + patch_sel * kKppRun, S.patch_run, n, prng,
                                      exact_every && (c + m) % exact_every == 0);
      if (non_finite) d.err = 9;  // NonFinite, before AllZero
      if (t == 0) s_draw = d;
    }
    __syncthreads();
    if (s_draw.err) {
      if (writer) {
        st_out[m] = S;
        st_out[m].err = s_draw.err;
      }
      return;
    }
    chosen = s_draw.row;
    drawn = s_draw.run;
    r = s_draw.r;
    if (chosen == kKppNone) {
      // kpp_exact_kernel reads the weights from w alone
      if (own_patch)
#pragma unroll
        for (uint32_t j = 0; j < kPer; ++j)
          if (lo + j * kWave < n) wm[lo + j * kWave] = wv[j];
      if (writer) {
        KppSeed& o = st_out[m];
        o = S;
        o.pending = 1;
        o.patch_run = kKppNone;
        o.r = r;
#pragma unroll
        for (int q = 0; q < 4; ++q) o.s[q] = prng[q];
      }
      return;
    }
  }
  float cv[D];
  load_padded<D>(xm + (uint64_t)chosen * DP, cv);
  if (b == 0 && t < (uint32_t)D) cm[(uint64_t)c * D + t] = xm[(uint64_t)chosen * DP + t];
  for (uint32_t j = t; j < c; j += kKppThreads) {
    float cj[D];
#pragma unroll
    for (int k = 0; k < D; ++k) cj[k] = cm[(uint64_t)j * D + k];
    lo_tab[j] = cand_lower_bound(exact_l2sq<D>(cj, cv), g);
  }
  __syncthreads();
  bool need[kPer];
#pragma unroll
  for (uint32_t j = 0; j < kPer; ++j)
    need[j] = lo + j * kWave < n && (c == 0 || !cand_cannot_beat(lo_tab[sv[j]], wv[j], g));
  float xv[kPer][D];
#pragma unroll
  for (uint32_t j = 0; j < kPer; ++j)
    if (need[j]) load_padded<D>(xm + (lo + j * kWave) * DP, xv[j]);
  const bool to_patch = FUSED && run == drawn;
  const uint32_t sel = patch_sel ^ 1u;
  double acc = 0.0;
  bool invalid = false;
#pragma unroll
  for (uint32_t j = 0; j < kPer; ++j) {
    const uint64_t i = lo + j * kWave;
    if (i >= n) continue;
    float wi = wv[j];
    bool changed = false;
    if (need[j]) {
      const float d = exact_l2sq<D>(xv[j], cv);
      if (c == 0 || d < wi) {  // kmeans.zig:134: replace on strict <
        wi = d;
        sm[i] = (uint16_t)c;
        changed = true;
      }
    }
    if (to_patch)
      pm[sel * kKppRun + j * kWave + t % kWave] = wi;
    else if (changed || own_patch)
      wm[i] = wi;  // unchanged weights are not rewritten
    invalid |= !(wi >= 0.0f && wi <= 3.402823466e38f);  // rng.zig:62 NonFinite
    acc += (double)wi;
  }
  if (invalid) atomicMin(&bad[m], c);
  acc = wave_inclusive_sum_f64(acc);
  if (t % kWave == kWave - 1) bsum[(bsel ^ 1u) * bstride + (uint64_t)m * n_runs + run] = acc;
  if (writer) {
    KppSeed& o = st_out[m];
    o = S;
    o.next = c + 1;
    o.pending = 0;
    o.bsel = bsel ^ 1u;
    if (FUSED) {
      o.patch_run = drawn;
      o.patch_sel = sel;
      if (c > 0 && pending == 0) {
        o.r = r;
#pragma unroll
        for (int q = 0; q < 4; ++q) o.s[q] = prng[q];
      }
    }
  }
}

// Exact weightedSample (rng.zig:60-81) for subspaces whose parallel decision
// was inconclusive, one block per such subspace.  The reference folds the
// f64 weights sequentially twice (the total, then the running cum up to the
// first u < cum).  Here the first fold is evaluated exactly in chunks of
// kFoldChunk weights (fold_rules.hpp with an f64 accumulator): all waves
// form the chunk descriptors, then wave 0 applies them in order, recording
// the exact running value before every chunk.  Because the weights are
// non-negative the running value never decreases, so the first u < cum lies
// in the first chunk whose end value exceeds u; wave 0 finds that chunk and
// folds only it term by term from its exact start.
// pre, chunks: [M][nc] scratch (nc = ceil(n / kFoldChunk)).
constexpr uint32_t kKppFallbackThreads = 1024;

// The body, for one weight vector wm[0 .. n) and its state S, run by a whole
// block of kKppFallbackThreads threads (the caller has checked that S needs
// it).  pm, cm: nc = ceil(n / kFoldChunk) entries of scratch.
__device__ __forceinline__ void kpp_fallback_block(const float* __restrict__ wm, uint64_t n, KppState& S,
                                          double* __restrict__ pm, FoldChunk* __restrict__ cm,
                                          uint32_t nc) {
  constexpr uint32_t kWaves = kKppFallbackThreads / kWave;
  __shared__ double wsum[kWaves];
  __shared__ double carry;
  __shared__ __attribute__((aligned(16))) float buf[kFoldChunk];
  const uint32_t lane = threadIdx.x % kWave, wv = threadIdx.x / kWave;
  // Chunk sums and descriptors, each wave kFallbackBatch chunks at a time
  // (all their loads in flight together).
  constexpr uint32_t kFallbackBatch = 4;
  for (uint32_t j0 = wv * kFallbackBatch; j0 < nc; j0 += kWaves * kFallbackBatch) {
    double cs[kFallbackBatch];
    fold_chunk_sums_wave<kFallbackBatch>(wm, n, j0, nc, cs);
    if (lane == 0)
#pragma unroll
      for (uint32_t b = 0; b < kFallbackBatch; ++b)
        if (j0 + b < nc) pm[j0 + b] = cs[b];
  }
  __syncthreads();
  block_prefix_f64<kKppFallbackThreads>(pm, nc, wsum, &carry);
  for (uint32_t j0 = wv * kFallbackBatch; j0 < nc; j0 += kWaves * kFallbackBatch) {
    double pre[kFallbackBatch];
#pragma unroll
    for (uint32_t b = 0; b < kFallbackBatch; ++b) pre[b] = j0 + b < nc ? pm[j0 + b] : 0.0;
    fold_quantize_chunks_wave<double, kFallbackBatch>(wm, n, j0, nc, pre, cm + j0);
  }
  __syncthreads();
  if (wv != 0) return;
  // Wave 0 only from here: pm[j] becomes the exact value before chunk j.
  const double total = fold_apply_wave<double>(wm, n, cm, nc, buf, pm);
  __threadfence_block();
  const double u = S.r * total;
  uint32_t jf = 0xFFFFFFFFu;
  for (uint32_t j0 = 0; j0 < nc && jf == 0xFFFFFFFFu; j0 += kWave) {
    const uint32_t j = j0 + lane;
    const bool hit = j < nc && u < (j + 1 < nc ? pm[j + 1] : total);
    const uint64_t ballot = __ballot(hit);
    if (ballot) jf = j0 + (uint32_t)__ffsll((long long)ballot) - 1;
  }
  uint64_t found = ~0ull;
  if (jf != 0xFFFFFFFFu) {
    const uint64_t lo = (uint64_t)jf * kFoldChunk;
    const uint32_t len = fold_chunk_len(n, jf);
    wave_lds_sync();
    for (uint32_t t = lane; t < len; t += kWave) buf[t] = wm[lo + t];
    wave_lds_sync();
    double cum = pm[jf];
    for (uint32_t t = 0; t < len; ++t) {
      cum += (double)buf[t];
      if (u < cum) {
        found = lo + t;
        break;
      }
    }
  } else {
    // rng.zig:79-81: no u < cum: the last positive weight (index 0 if none)
    found = 0;
    for (uint64_t b = n; b > 0;) {
      const uint64_t lo = b > kWave ? b - kWave : 0;
      const uint64_t i = lo + lane;
      const uint64_t ballot = __ballot(i < b && wm[i] != 0.0f);
      if (ballot) {
        found = lo + 63 - (uint64_t)__clzll((long long)ballot);
        break;
      }
      b = lo;
    }
  }
  if (lane == 0) {
    S.chosen = (uint32_t)found;
    S.fallback = 0;
  }
}

// The draw of codeword `next` of every subspace, one block each, for rows past
// kKppFusedRuns runs (262,144 rows): there the blocks' own draws cost more
// than a launch (1,521,797 rows x 16 subspaces, drop-in train: 55 ms with
// them, 42 with this kernel), and open draws are not rare (about n^2 2e-16
// each, 2-3 of 4,080 there), so the block makes the exact draw at once.  Sets
// `chosen` and pending 2.
__global__ __launch_bounds__(kKppFallbackThreads) void kpp_draw_kernel(
    const float* __restrict__ w, const double* __restrict__ bsum, uint64_t bstride,
    const uint32_t* __restrict__ bad, KppSeed* __restrict__ st, uint64_t n, uint32_t K,
    uint32_t n_runs, uint32_t exact_every, double* __restrict__ pre,
    FoldChunk* __restrict__ chunks, uint32_t nc) {
  constexpr uint32_t kPerShare = kKppFallbackThreads / kWave;  // lanes to a share of the runs
  __shared__ double shares[kWave];
  __shared__ KppState S;  // the exact draw works on this copy
  __shared__ uint32_t s_open;
  const uint32_t m = blockIdx.x, t = threadIdx.x;
  const KppSeed& in = st[m];
  if (in.err || in.next == K || in.next == 0) return;
  const double* sums = bsum + in.bsel * bstride + (uint64_t)m * n_runs;
  const uint32_t per = (n_runs + kWave - 1) / kWave, l = t / kPerShare;
  const uint32_t q1 = (l + 1) * per < n_runs ? (l + 1) * per : n_runs;
  double sum = 0.0;
#pragma unroll 4
  for (uint32_t q = l * per + t % kPerShare; q < q1; q += kPerShare) sum += sums[q];
  for (uint32_t off = 1; off < kPerShare; off <<= 1) sum += __shfl_xor(sum, (int)off, kWave);
  if (t % kPerShare == 0) shares[l] = sum;
  __syncthreads();
  if (t < kWave) {
    uint64_t prng[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) prng[q] = in.s[q];
    const bool non_finite = bad[m] < in.next;  // rng.zig:62
    const KppDraw d = kpp_draw_wave<false>(sums, n_runs, shares[t], w + (uint64_t)m * n, nullptr,
                                           kKppNone, n, prng,
                                           exact_every && (in.next + m) % exact_every == 0);
    if (t == 0) {
      KppSeed& o = st[m];
      const int32_t err = non_finite ? 9 : d.err;  // NonFinite before AllZero
#pragma unroll
      for (int q = 0; q < 4; ++q) o.s[q] = prng[q];
      o.r = d.r;
      o.chosen = d.row;
      o.err = err;
      o.pending = 2;
      S.r = d.r;
      s_open = !err && d.row == kKppNone;
    }
  }
  __syncthreads();
  if (!s_open) return;
  kpp_fallback_block(w + (uint64_t)m * n, n, S, pre + (uint64_t)m * nc,
                     chunks + (uint64_t)m * nc, nc);
  if (t == 0) st[m].chosen = S.chosen;  // of wave 0, whose first lane set it
}

// The exact draw of every pending subspace, one block each: sets `chosen` for
// the rounds that follow.
__global__ __launch_bounds__(kKppFallbackThreads) void kpp_exact_kernel(
    const float* __restrict__ w, KppSeed* __restrict__ st, uint64_t n, double* __restrict__ pre,
    FoldChunk* __restrict__ chunks, uint32_t nc) {
  __shared__ KppState S;  // the draw works on this copy; thread 0 writes it back
  const uint32_t m = blockIdx.x;
  if (st[m].err || st[m].pending != 1) return;
  if (threadIdx.x == 0) S.r = st[m].r;
  __syncthreads();
  kpp_fallback_block(w + (uint64_t)m * n, n, S, pre + (uint64_t)m * nc,
                     chunks + (uint64_t)m * nc, nc);
  if (threadIdx.x == 0) {  // of wave 0, whose first lane set S.chosen
    st[m].chosen = S.chosen;
    st[m].pending = 2;
  }
}

// Seeds every subspace's stream with seed +% m and draws the first row.
__global__ void kpp_init_kernel(KppSeed* __restrict__ st, uint32_t* __restrict__ bad,
                                uint64_t seed, uint64_t n, uint32_t M) {
  const uint32_t m = blockIdx.x * blockDim.x + threadIdx.x;
  if (m >= M) return;
  KppSeed S{};
  uint64_t sm = seed + m;
  for (int q = 0; q < 4; ++q) S.s[q] = kpp_splitmix(&sm);
  S.chosen = (uint32_t)kpp_uint_less_than(S.s, n);
  S.patch_run = kKppNone;
  st[m] = S;
  bad[m] = kKppNone;
}

}  // namespace tacgpu
