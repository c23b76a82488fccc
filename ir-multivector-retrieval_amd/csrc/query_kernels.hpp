// query_kernels.hpp — gfx950 kernels of the query side that consumes PQ
// codes: the per-query distance table (src/index/pq.zig:92-123) and refine's
// exact MaxSim over candidate documents (src/retrieval/refine.zig:83-145).
// Included once, by tac_gpu.hip.  Compiled with -ffp-contract=off: every
// multiply and add is rounded separately, in the reference's order.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "pq_kernels.hpp"

namespace tacgpu {

// vec.dot (src/util/vec.zig:37-103): dims 2 and 4 are left folds from 0,
// dims 64 and 128 accumulate in 4 lanes chunk after chunk and reduce
// ((a0 + a1) + a2) + a3, other dims take the generic path at the device's
// lane count (generic_vec: lanes, lane-order reduce, tail).
// `a` and `b` may live in LDS or global memory.
__device__ inline float ref_dot(const float* a, const float* b, uint32_t d) {
  if (d == 2) return a[0] * b[0] + a[1] * b[1];
  if (d == 4) {
    float s = 0.0f;
    for (int i = 0; i < 4; ++i) s = s + a[i] * b[i];
    return s;
  }
  if (d == 64 || d == 128) {
    float acc0 = 0.0f, acc1 = 0.0f, acc2 = 0.0f, acc3 = 0.0f;
    for (uint32_t c = 0; c < d; c += 4) {
      acc0 = acc0 + a[c] * b[c];
      acc1 = acc1 + a[c + 1] * b[c + 1];
      acc2 = acc2 + a[c + 2] * b[c + 2];
      acc3 = acc3 + a[c + 3] * b[c + 3];
    }
    return ((acc0 + acc1) + acc2) + acc3;
  }
  return generic_vec<true>(a, b, d);
}

// PQ.buildDistanceTable: table[((mm * K) + c) * n_q + i] =
// dot(query_i[mm * D .. +D], codebook[mm][c]); one thread per entry, so
// consecutive threads write consecutive i.
__global__ __launch_bounds__(256) void distance_table_kernel(
    const float* __restrict__ q, const float* __restrict__ cb, float* __restrict__ table,
    uint32_t n_q, uint32_t dim, uint32_t M, uint32_t K, uint32_t D) {
  const uint64_t g = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const uint64_t total = (uint64_t)M * K * n_q;
  if (g >= total) return;
  const uint32_t i = (uint32_t)(g % n_q);
  const uint64_t mc = g / n_q;
  const uint32_t mm = (uint32_t)(mc / K);
  table[g] = ref_dot(q + (uint64_t)i * dim + (uint64_t)mm * D, cb + mc * D, D);
}

// Refine status codes of a candidate (tac_status values).
constexpr uint32_t kRefineOk = 0;
constexpr uint32_t kRefineDocOutOfRange = 18;
constexpr uint32_t kRefineLayoutCorrupt = 19;

struct RefineIndex {
  const float* centroids;            // [kappa][dim]
  const uint64_t* doc_index;         // [n_docs + 1]
  const uint8_t* payload;            // per-doc layouts
  const uint64_t* doc_token_offsets; // [n_docs + 1]
  const float* norms;                // [n_tokens]
  uint64_t n_docs, n_tokens, payload_len;
  uint32_t dim, kappa, M, K;
};

__device__ __forceinline__ uint32_t load_u32_le(const uint8_t* p) {
  return (uint32_t)p[0] | (uint32_t)p[1] << 8 | (uint32_t)p[2] << 16 | (uint32_t)p[3] << 24;
}

// A team of one block of W waves, or with WAVES of one of its waves, per
// candidate document (the host chooses by the documents' mean length),
// grid-stride over candidates.  A wave covers QP = n_q rounded up to a power of
// two (at most 64) query tokens and S = 64 / QP slots; lane (s, i) takes query
// token i0 + i against R document tokens of slot s at a time, for every token k
//   cent  = dot(q_i, centroid[c_k])            (centroid rows staged in LDS)
//   res   = sum over m of table[m][code_km][i]  (in m order, from 0)
//   score = cent + norm_k * res
// and keeps the first k of its running maximum (strict >, from -inf).  The
// slots and waves of a query token then merge (larger value; on equal values
// the earlier k, which keeps the sign of a zero maximum the reference would
// keep), and the team's wave 0 folds best_0 + best_1 + ... in i order (0 for an empty
// document).  Layout checks follow refine.zig:51-65,107-114; a failing
// candidate scores 0, `first_bad` keeps the lowest one with its status
// (candidate << 32 | status) and `any_bad`, a word of pinned host memory,
// tells the host to look (no copy is needed after a clean call).
//
// Bound by latency on few candidates (a chain of doc id, layout, ids, rows,
// table) and by the table gathers and the LDS reads of the dots on many.
// One wave per document with a tile of S tokens left 50-1,000 waves on 1,024
// SIMDs, each walking its document through some 25 dependent round trips:
// 314 us at 32 query tokens x 1,000 documents of 1-100 tokens (m16), 220 us
// at 8 x 50 (m32).  Here a tile's ids, codes and rows are in flight at once,
// a query row read from LDS serves R tokens, and 16 R table entries are in
// flight while the dots run: 31 us and 8 us.  Four tokens a lane spill
// registers (73 against 51 us a call at 32 x 1,000).
constexpr uint32_t kRefineTileFloats = 8192;  // most row floats, and codes, of a tile
constexpr uint32_t kRefineWaveFloats = 1536;  // of a tile that one wave works on

__host__ __device__ inline uint32_t refine_qp(uint32_t n_q) {
  uint32_t qp = 1;
  while (qp < n_q && qp < 64) qp <<= 1;
  return qp;
}

// Row stride in LDS: 16-byte aligned and staggered over the banks for the
// vector reads of dims 64 and 128, odd for the scalar reads of the others.
__host__ __device__ inline uint32_t refine_stride(uint32_t dim, bool fast) {
  return fast ? dim + 4 : dim + 1;
}

// Tokens of a tile: at most `floats` row floats and as many codes, or one.
inline uint32_t refine_tile(uint32_t dim, uint32_t M, uint32_t floats, uint32_t most) {
  const uint32_t w = dim > M ? dim : M, t = floats / w;
  return t > most ? most : (t ? t : 1u);
}

// Dynamic LDS floats of the queries, and of a team of `waves` waves: its tile's
// centroid rows, per wave 64 best values and their token indices, and the
// tile's codes as u16, in rows of whole 16 bytes.
__host__ __device__ inline uint32_t refine_query_floats(uint32_t n_q, uint32_t ld) {
  return (n_q * ld + 3) / 4 * 4;
}
__host__ __device__ inline uint32_t refine_team_floats(uint32_t ld, uint32_t waves, uint32_t M,
                                                       uint32_t tile) {
  return (tile * ld + 3) / 4 * 4 + waves * 128 +
         (M <= kRefineTileFloats ? tile * ((M + 7) / 8 * 4) : 0u);
}

// dot(q_i, centroid row) of R rows in LDS; FAST is vec.dot's 4-lane form.
template <int R, bool FAST>
__device__ __forceinline__ void refine_dots(const float* qrow, const float* const (&row)[R],
                                            uint32_t dim, float (&cent)[R]) {
  if constexpr (FAST) {
    float acc[R][4];
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[r][j] = 0.0f;
#pragma unroll 4
    for (uint32_t c = 0; c < dim; c += 4) {
      const float4 a = *reinterpret_cast<const float4*>(qrow + c);
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const float4 v = *reinterpret_cast<const float4*>(row[r] + c);
        acc[r][0] = acc[r][0] + a.x * v.x;
        acc[r][1] = acc[r][1] + a.y * v.y;
        acc[r][2] = acc[r][2] + a.z * v.z;
        acc[r][3] = acc[r][3] + a.w * v.w;
      }
    }
#pragma unroll
    for (int r = 0; r < R; ++r) cent[r] = ((acc[r][0] + acc[r][1]) + acc[r][2]) + acc[r][3];
  } else {
    cent[0] = ref_dot(qrow, row[0], dim);
  }
}

// Scores of R tokens for query token i.  `codes[r]` is the token's row of
// codes in LDS, a multiple of 8 (zero past M).  The table entries of up to
// U subspaces are in flight while the dots run.
template <int R, bool FAST>
__device__ __forceinline__ void refine_scores(const uint16_t* const (&codes)[R],
                                              const float* table, uint32_t M, uint32_t step,
                                              uint32_t n_q, uint32_t i, const float* qrow,
                                              const float* const (&row)[R], uint32_t dim,
                                              const float (&norm)[R], float (&score)[R]) {
  constexpr uint32_t U = 16;
  float res[R], cent[R];
#pragma unroll
  for (int r = 0; r < R; ++r) res[r] = 0.0f;
  for (uint32_t m0 = 0; m0 < M; m0 += U) {
    float v[R][U];
#pragma unroll
    for (uint32_t g = 0; g < U; g += 8) {
      if (m0 + g >= M) break;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const uint4 w = *reinterpret_cast<const uint4*>(codes[r] + m0 + g);
        const uint32_t pair[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
        for (uint32_t u = 0; u < 8; ++u) {
          const uint32_t mm = m0 + g + u < M ? m0 + g + u : M - 1;
          const uint32_t code = u % 2 ? pair[u / 2] >> 16 : pair[u / 2] & 0xFFFFu;
          // at most 65,536 codes x 8,192 query tokens: the byte offset fits
          // 32 bits, beside a scalar base
          const uint32_t off = (code * n_q + i) * (uint32_t)sizeof(float);
          v[r][g + u] = *reinterpret_cast<const float*>(
              reinterpret_cast<const char*>(table + (size_t)mm * step) + off);
        }
      }
    }
    if (m0 == 0) refine_dots<R, FAST>(qrow, row, dim, cent);
#pragma unroll
    for (uint32_t g = 0; g < U; g += 8) {
      if (m0 + g >= M) break;
#pragma unroll
      for (uint32_t u = 0; u < 8; ++u)
        if (m0 + g + u < M)
#pragma unroll
          for (int r = 0; r < R; ++r) res[r] = res[r] + v[r][g + u];
    }
  }
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const float scaled = norm[r] * res[r];
    score[r] = cent[r] + scaled;
  }
}

// The same with the codes read from the payload one by one, for rows of codes
// past the LDS tile (M above kRefineTileFloats); a code past K raises `bad`.
template <bool FAST>
__device__ __forceinline__ float refine_score_raw(const uint8_t* codes, uint32_t cb,
                                               const float* table, uint32_t M, uint32_t K,
                                               uint32_t n_q, uint32_t i, const float* qrow,
                                               const float* row, uint32_t dim, float norm,
                                               bool& bad) {
  const float* const rows[1] = {row};
  float cent[1], res = 0.0f;
  refine_dots<1, FAST>(qrow, rows, dim, cent);
  for (uint32_t mm = 0; mm < M; ++mm) {
    const uint8_t* p = codes + (uint64_t)mm * cb;
    const uint32_t code = cb == 1 ? p[0] : (uint32_t)p[0] | (uint32_t)p[1] << 8;
    bad = bad || code >= K;
    res = res + table[((uint64_t)mm * K + (code < K ? code : 0u)) * n_q + i];
  }
  const float scaled = norm * res;
  return cent[0] + scaled;
}

// Keeps the larger value, and on equal values the earlier token.
__device__ __forceinline__ void refine_keep(float& b, uint32_t& bk, float o, uint32_t ok) {
  if (o > b || (o == b && ok < bk)) {
    b = o;
    bk = ok;
  }
}

// FAST: dims 64 and 128 (vec.dot's 4-lane form), with 16-byte aligned
// centroid and query arrays; else R is 1 and ref_dot serves any dim.  WAVES: a
// candidate to each wave instead of each block, with the queries shared.
template <int R, bool FAST, bool WAVES>
__global__ __launch_bounds__(512, 4) void refine_kernel(
    RefineIndex ix, const float* __restrict__ q, uint32_t n_q, const float* __restrict__ table,
    const uint32_t* __restrict__ doc_ids, uint32_t n_cand, uint32_t TT, float* __restrict__ scores,
    unsigned long long* __restrict__ first_bad, uint32_t* __restrict__ any_bad) {
  static_assert(FAST || R == 1, "the generic dot takes one token at a time");
  extern __shared__ __attribute__((aligned(16))) float lds[];
  const uint32_t lane = threadIdx.x % 64;
  // The team: W waves, this one its wave w, this thread its thread tid of nt.
  const uint32_t teams = WAVES ? blockDim.x / 64 : 1, team = WAVES ? threadIdx.x / 64 : 0;
  const uint32_t W = WAVES ? 1 : blockDim.x / 64, w = WAVES ? 0 : threadIdx.x / 64;
  const uint32_t tid = WAVES ? lane : threadIdx.x, nt = WAVES ? 64 : blockDim.x;
  const uint32_t ld = refine_stride(ix.dim, FAST);
  const uint32_t QP = refine_qp(n_q), S = 64 / QP;
  const uint32_t slot = lane / QP, qi = lane % QP;
  float* qs = lds;  // [n_q][ld]
  float* rows = lds + refine_query_floats(n_q, ld) +
                team * refine_team_floats(ld, W, ix.M, TT);         // [TT][ld]
  float* bestv = rows + (TT * ld + 3) / 4 * 4;                      // [W][64]
  uint32_t* bestk = reinterpret_cast<uint32_t*>(bestv + 64 * W);    // [W][64]
  uint16_t* scodes = reinterpret_cast<uint16_t*>(bestk + 64 * W);   // [TT][lc]
  const bool long_codes = ix.M > kRefineTileFloats;
  const uint32_t lc = (ix.M + 7) / 8 * 8;
  if constexpr (FAST) {
    const uint32_t d4 = ix.dim / 4;
    const float4* q4 = reinterpret_cast<const float4*>(q);
    for (uint32_t f = threadIdx.x; f < n_q * d4; f += blockDim.x)
      *reinterpret_cast<float4*>(qs + (f / d4) * ld + f % d4 * 4) = q4[f];
  } else {
    for (uint32_t f = threadIdx.x; f < n_q * ix.dim; f += blockDim.x)
      qs[(f / ix.dim) * ld + f % ix.dim] = q[f];
  }
  if constexpr (WAVES) __syncthreads();  // the teams' only common point
  const uint32_t cb = ix.K <= 256 ? 1u : 2u, step = ix.K * n_q;
  for (uint32_t cand = blockIdx.x * teams + team; cand < n_cand; cand += gridDim.x * teams) {
    const uint64_t doc = doc_ids[cand];
    uint32_t st = kRefineOk;
    uint32_t n_d = 0;
    uint64_t lo = 0, t_lo = 0;
    if (doc >= ix.n_docs) {
      st = kRefineDocOutOfRange;
    } else {
      lo = ix.doc_index[doc];
      const uint64_t hi = ix.doc_index[doc + 1];
      t_lo = ix.doc_token_offsets[doc];
      const uint64_t t_hi = ix.doc_token_offsets[doc + 1];
      if (hi < lo || hi > ix.payload_len || hi - lo < 4) {
        st = kRefineLayoutCorrupt;
      } else {
        // A sound layout holds t_hi - t_lo tokens: its size is checked by
        // that count, so that the loads of its ids need not wait for the
        // layout's own count, checked beside them (bad_count).
        const uint64_t n_t = t_hi - t_lo;
        if (t_hi < t_lo || n_t > 0xFFFFFFFFull || t_hi > ix.n_tokens ||
            __umul64hi(n_t, 4ull + (uint64_t)ix.M * cb) != 0 ||
            hi - lo - 4 < n_t * (4ull + (uint64_t)ix.M * cb))
          st = kRefineLayoutCorrupt;
        else
          n_d = (uint32_t)n_t;
      }
    }
    const uint8_t* lay = ix.payload + lo;
    const uint8_t* ids = lay + 4;
    const uint8_t* codes0 = lay + 4 + 4ull * n_d;
    const bool id_words = ((uintptr_t)lay & 3) == 0;
    const bool words = cb == 1 && ix.M % 8 == 0 && ((uintptr_t)codes0 & 3) == 0;
    const bool bad_count = st == kRefineOk && load_u32_le(lay) != n_d;
    if (n_d == 0 && bad_count) st = kRefineLayoutCorrupt;
    float total = 0.0f;
    for (uint32_t i0 = 0; st == kRefineOk && i0 < n_q; i0 += QP) {
      const uint32_t i = i0 + qi;
      const uint32_t ic = i < n_q ? i : n_q - 1;
      float b = -__builtin_inff();
      uint32_t bk = 0xFFFFFFFFu;
      bool bad = bad_count;
      for (uint32_t k0 = 0; k0 < n_d; k0 += TT) {
        const uint32_t cnt = n_d - k0 < TT ? n_d - k0 : TT;
        // the tile's codes, as u16
        if (long_codes) {
        } else if (words) {
          const uint32_t* src = reinterpret_cast<const uint32_t*>(codes0 + (uint64_t)k0 * ix.M);
          for (uint32_t f = tid; f < cnt * ix.M / 4; f += nt) {
            const uint32_t v = src[f];
            const uint32_t c0 = v & 0xFFu, c1 = (v >> 8) & 0xFFu, c2 = (v >> 16) & 0xFFu,
                           c3 = v >> 24;
            bad = bad || c0 >= ix.K || c1 >= ix.K || c2 >= ix.K || c3 >= ix.K;
            *reinterpret_cast<uint2*>(scodes + 4 * f) = make_uint2(c0 | c1 << 16, c2 | c3 << 16);
          }
        } else {
          const uint8_t* src = codes0 + (uint64_t)k0 * ix.M * cb;
          for (uint32_t f = tid; f < cnt * lc; f += nt) {
            const uint32_t mm = f % lc;
            const uint8_t* p = src + ((uint64_t)(f / lc) * ix.M + mm) * cb;
            uint32_t c = 0;
            if (mm < ix.M) c = cb == 1 ? p[0] : (uint32_t)p[0] | (uint32_t)p[1] << 8;
            bad = bad || c >= ix.K;
            scodes[f] = (uint16_t)c;
          }
        }
        // centroid rows of tokens k0 .. k0 + cnt - 1
        const uint32_t units = FAST ? ix.dim / 4 : ix.dim;
        for (uint32_t f = tid; f < cnt * units; f += nt) {
          const uint32_t s = f / units, d = f % units;
          const uint8_t* idp = ids + 4ull * (k0 + s);
          const uint32_t cid =
              id_words ? *reinterpret_cast<const uint32_t*>(idp) : load_u32_le(idp);
          if (cid >= ix.kappa) {
            bad = true;
          } else if constexpr (FAST) {
            *reinterpret_cast<float4*>(rows + s * ld + 4 * d) =
                reinterpret_cast<const float4*>(ix.centroids)[(uint64_t)cid * units + d];
          } else {
            rows[s * ld + d] = ix.centroids[(uint64_t)cid * ix.dim + d];
          }
        }
        if constexpr (WAVES) wave_lds_sync();
        // also: the rows (and the queries) are staged
        if (WAVES ? __any(bad) : __syncthreads_or(bad)) {
          st = kRefineLayoutCorrupt;
          break;
        }
        for (uint32_t base = w * S * R; base < cnt; base += W * S * R) {
          uint32_t t[R];
          float norm[R], score[R];
          const float* row[R];
          const uint16_t* codes[R];
#pragma unroll
          for (int r = 0; r < R; ++r) {
            t[r] = base + r * S + slot;
            const uint32_t tc = t[r] < cnt ? t[r] : cnt - 1;  // a lane past the end repeats one
            norm[r] = ix.norms[t_lo + k0 + tc];
            row[r] = rows + tc * ld;
            codes[r] = scodes + tc * lc;
          }
          if (long_codes) {
            for (int r = 0; r < R; ++r) {
              const uint32_t tc = t[r] < cnt ? t[r] : cnt - 1;
              score[r] = refine_score_raw<FAST>(
                  codes0 + (uint64_t)(k0 + tc) * ix.M * cb, cb, table, ix.M, ix.K, n_q, ic,
                  qs + ic * ld, rows + tc * ld, ix.dim, norm[r], bad);
            }
          } else
            refine_scores<R, FAST>(codes, table, ix.M, step, n_q, ic, qs + ic * ld, row, ix.dim,
                                 norm, score);
#pragma unroll
          for (int r = 0; r < R; ++r)
            if (t[r] < cnt && i < n_q && score[r] > b) {
              b = score[r];
              bk = k0 + t[r];
            }
        }
        if constexpr (WAVES) wave_lds_sync();
        // also: the rows may be overwritten
        if (WAVES ? __any(bad) : __syncthreads_or(bad)) {
          st = kRefineLayoutCorrupt;
          break;
        }
      }
      if (st != kRefineOk || n_d == 0) break;
      for (uint32_t off = QP; off < 64; off <<= 1) {
        const float o = __shfl_xor(b, off, 64);
        const uint32_t ok = __shfl_xor(bk, off, 64);
        refine_keep(b, bk, o, ok);
      }
      if constexpr (!WAVES) {
        bestv[threadIdx.x] = b;
        bestk[threadIdx.x] = bk;
        __syncthreads();
      }
      if (w == 0) {
        for (uint32_t ww = 1; ww < W; ++ww)
          refine_keep(b, bk, bestv[ww * 64 + lane], bestk[ww * 64 + lane]);
        const uint32_t cnt = n_q - i0 < QP ? n_q - i0 : QP;
        for (uint32_t j = 0; j < cnt; ++j)
          total = total + __uint_as_float(
                              (uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(b), (int)j));
      }
      if constexpr (!WAVES) __syncthreads();  // wave 0 has read the best values
    }
    if (tid == 0) {
      scores[cand] = st == kRefineOk ? total : 0.0f;
      if (st != kRefineOk) {
        atomicMin(first_bad, (unsigned long long)cand << 32 | st);
        __hip_atomic_store(any_bad, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      }
    }
  }
}

}  // namespace tacgpu
