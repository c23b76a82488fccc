// storage_kernels.hpp — gfx950 kernels of the storage.build stages around the
// PQ build: per-token residuals and norms.  Included once, by tac_gpu.hip.
//
// Arithmetic contract: compiled with -ffp-contract=off, so every subtract,
// multiply and add is rounded separately as in Zig's strict float mode;
// sqrtf and 1.0f / x are the correctly rounded IEEE operations (HIP's
// default for single precision).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "pq_kernels.hpp"

namespace tacgpu {

constexpr int kResBlock = 256;  // threads per residual block
constexpr uint32_t kBadRow = 0xFFFFFFFFu;

// Rows per residual block: one folding thread per row and an LDS tile of
// rows x (dim + 1) floats within 64 KB.
__host__ __device__ inline uint32_t residual_rows(uint32_t dim) {
  uint32_t r = 16000u / (dim + 1u);
  return r > 64u ? 64u : (r == 0u ? 1u : r);
}

// storage.zig:255-278 (residualsAndNormsChunk) over rows [row0, row0 + R):
//   1. all threads load the rows and their centroids in VW-float units,
//      coalesced, and park diff = v - c in an LDS tile [R][dim + 1];
//   2. thread r folds row r: sum = 0; sum = sum + diff_d * diff_d for d
//      ascending; norm = sqrt(sum); scale = 1 / norm if norm > 0;
//   3. all threads store diff * scale (or diff unchanged when norm is not
//      > 0) with coalesced stores.
// Every row is read before any row of the block is written, and blocks own
// disjoint rows, so `out` may alias `v`.  An assignment >= n_cent raises
// `status`, a word of pinned host memory that the host has cleared, and its row
// reads nothing (the outputs of such a call are unspecified; the host reports
// the error).  At HBM rate (1.52M x 64 in 148 us, 5.4 TB/s; a large copy
// reaches 5.2); clearing a device word before and copying it back after took
// 23 us more a call, the flag takes 13.
template <int VW>
__global__ __launch_bounds__(kResBlock) void residual_kernel(
    const float* v, const float* __restrict__ cent, const uint32_t* __restrict__ assign,
    float* out, float* __restrict__ norms, uint32_t* __restrict__ status, uint64_t n,
    uint32_t dim, uint32_t n_cent, uint32_t R) {
  extern __shared__ __attribute__((aligned(16))) float tile[];  // [R][dim + 1]
  const uint32_t ld = dim + 1;
  float* scale = tile + (size_t)R * ld;                          // [R]
  uint32_t* rowa = reinterpret_cast<uint32_t*>(scale + R);       // [R]
  const uint64_t row0 = (uint64_t)blockIdx.x * R;
  const uint32_t rows = (uint32_t)(n - row0 < R ? n - row0 : R);
  const uint32_t t = threadIdx.x;
  if (t < rows) {
    uint32_t a = assign[row0 + t];
    if (a >= n_cent) {
      __hip_atomic_store(status, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      a = kBadRow;
    }
    rowa[t] = a;
  }
  __syncthreads();

  const uint32_t q = dim / VW;        // units per row
  const uint32_t units = rows * q;
  constexpr int kUnroll = 4;
  for (uint32_t base = 0; base < units; base += kResBlock * kUnroll) {
    float dv[kUnroll][VW];
    uint32_t rr[kUnroll], cc[kUnroll];
#pragma unroll
    for (int k = 0; k < kUnroll; ++k) {
      const uint32_t u = base + k * kResBlock + t;
      rr[k] = u / q;
      cc[k] = u % q;
      if (u < units && rowa[rr[k]] != kBadRow) {
        const float* vp = v + (row0 + rr[k]) * dim + (uint64_t)cc[k] * VW;
        const float* cp = cent + (uint64_t)rowa[rr[k]] * dim + (uint64_t)cc[k] * VW;
        if constexpr (VW == 4) {
          const float4 a = *reinterpret_cast<const float4*>(vp);
          const float4 b = *reinterpret_cast<const float4*>(cp);
          dv[k][0] = a.x - b.x;
          dv[k][1] = a.y - b.y;
          dv[k][2] = a.z - b.z;
          dv[k][3] = a.w - b.w;
        } else {
#pragma unroll
          for (int j = 0; j < VW; ++j) dv[k][j] = vp[j] - cp[j];
        }
      } else {
#pragma unroll
        for (int j = 0; j < VW; ++j) dv[k][j] = __builtin_nanf("");
      }
    }
#pragma unroll
    for (int k = 0; k < kUnroll; ++k) {
      const uint32_t u = base + k * kResBlock + t;
      if (u < units) {
#pragma unroll
        for (int j = 0; j < VW; ++j) tile[rr[k] * ld + cc[k] * VW + j] = dv[k][j];
      }
    }
  }
  __syncthreads();

  if (t < rows) {
    const float* row = tile + (size_t)t * ld;
    float sum = 0.0f;
    for (uint32_t d = 0; d < dim; ++d) {
      const float x = row[d];
      const float sq = x * x;
      sum = sum + sq;
    }
    const float norm = sqrtf(sum);
    norms[row0 + t] = norm;
    // 1/norm >= +0 for every norm > 0 (+inf included); -1 marks "unscaled"
    scale[t] = norm > 0.0f ? 1.0f / norm : -1.0f;
  }
  __syncthreads();

  for (uint32_t base = 0; base < units; base += kResBlock) {
    const uint32_t u = base + t;
    if (u >= units) break;
    const uint32_t r = u / q, c = u % q;
    const float s = scale[r];
    float y[VW];
#pragma unroll
    for (int j = 0; j < VW; ++j) {
      const float x = tile[r * ld + c * VW + j];
      y[j] = s >= 0.0f ? x * s : x;
    }
    float* op = out + (row0 + r) * dim + (uint64_t)c * VW;
    if constexpr (VW == 4) {
      *reinterpret_cast<float4*>(op) = make_float4(y[0], y[1], y[2], y[3]);
    } else {
#pragma unroll
      for (int j = 0; j < VW; ++j) op[j] = y[j];
    }
  }
}

}  // namespace tacgpu

namespace tacgpu {

// ---------------------------------------------------------------------------
// .tac per-document layouts (src/index/storage.zig:674-686, :705-749).
// Each doc d occupies align8(4 + 4 n_d + n_d m cb) payload bytes:
//   u32 n_d | u32 centroid id x n_d | codes (n_d x m x cb bytes) | zeros.
// doc_index[d] is the payload offset of doc d; doc_index[n_docs] the total.
// ---------------------------------------------------------------------------
__device__ __forceinline__ uint64_t doc_bytes(uint64_t n_d, uint32_t m, uint32_t cb) {
  return (4 + 4 * n_d + n_d * m * cb + 7) & ~7ull;
}

constexpr int kScanBlock = 256;
constexpr int kScanPer = 4;  // elements per thread in the u64 scan
// Documents past kDocSlice tokens are written in slices of as many, each by a
// wave of its own: one wave would walk them alone long after the others are
// done.  Sound offsets make at most n_tokens / 256 slices.
constexpr uint64_t kDocSlice = 512;

struct DocSlice {
  uint64_t doc;
  uint64_t at;     // the document's offset within its scan block
  uint64_t first;  // the slice's first token
};
__host__ __device__ inline uint64_t doc_slices_most(uint64_t n_tokens) {
  return n_tokens / (kDocSlice / 2);
}

// State of a layout call on the device.  bad and n_slices are zero between
// calls: doc_sums_scan_kernel moves them to go and slices.
struct DocState {
  unsigned long long n_slices;  // slices listed
  unsigned long long slices;    // n_slices of this call
  uint32_t bad;                 // an offset decreases or passes n_tokens
  uint32_t go;                  // the payload fits and the offsets are sound
};

// Phase 1: per-block exclusive scan of doc sizes into doc_index, block totals
// into `sums`.
// Offsets that decrease or pass n_tokens raise st->bad (the writer then
// does not run) and count as empty documents; long documents' slices are listed.
__global__ __launch_bounds__(kScanBlock) void doc_sizes_scan_kernel(
    const uint64_t* __restrict__ doc_offsets, uint64_t n_docs, uint64_t n_tokens, uint32_t m,
    uint32_t cb, uint64_t* __restrict__ doc_index, uint64_t* __restrict__ sums,
    DocState* __restrict__ st, DocSlice* __restrict__ slices) {
  __shared__ uint64_t warp_tot[kScanBlock / 64];
  const uint64_t base = (uint64_t)blockIdx.x * kScanBlock * kScanPer + threadIdx.x * kScanPer;
  uint64_t v[kScanPer];
  uint64_t local = 0;
  uint32_t is_long = 0;
#pragma unroll
  for (int q = 0; q < kScanPer; ++q) {
    const uint64_t d = base + q;
    v[q] = 0;
    if (d < n_docs) {
      const uint64_t a = doc_offsets[d], b = doc_offsets[d + 1];
      if (b < a || b > n_tokens) {
        atomicOr(&st->bad, 1u);
      } else {
        v[q] = doc_bytes(b - a, m, cb);
        is_long |= b - a > kDocSlice ? 1u << q : 0u;
      }
    }
    local += v[q];
  }
  const uint32_t lane = threadIdx.x % 64, w = threadIdx.x / 64;
  uint64_t incl = local;
  for (int off = 1; off < 64; off <<= 1) {
    const uint64_t o = __shfl_up(incl, off, 64);
    if (lane >= (uint32_t)off) incl += o;
  }
  if (lane == 63) warp_tot[w] = incl;
  __syncthreads();
  uint64_t before = 0;
  for (uint32_t q = 0; q < w; ++q) before += warp_tot[q];
  uint64_t run = before + incl - local;
#pragma unroll
  for (int q = 0; q < kScanPer; ++q) {
    const uint64_t d = base + q;
    if (d < n_docs) doc_index[d] = run;
    if (is_long >> q & 1u) {
      const uint64_t n_d = doc_offsets[d + 1] - doc_offsets[d];
      const uint64_t count = (n_d + kDocSlice - 1) / kDocSlice;
      const uint64_t at = atomicAdd(&st->n_slices, (unsigned long long)count);
      for (uint64_t i = 0; i < count && at + i < doc_slices_most(n_tokens); ++i)
        slices[at + i] = DocSlice{d, run, i * kDocSlice};
    }
    run += v[q];
  }
  if (threadIdx.x == kScanBlock - 1) sums[blockIdx.x] = before + incl;
}

// Phase 2 (one block): exclusive scan of the block totals in place; the
// grand total lands in doc_index[n_docs].  Decides whether the writer runs and
// tells the host (host[0] bad offsets, host[1..2] the total).
__global__ __launch_bounds__(kScanBlock) void doc_sums_scan_kernel(
    uint64_t* __restrict__ sums, uint32_t nb, uint64_t* __restrict__ doc_index, uint64_t n_docs,
    uint64_t payload_len, DocState* __restrict__ st, uint32_t* __restrict__ host) {
  __shared__ uint64_t warp_tot[kScanBlock / 64];
  __shared__ uint64_t carry;
  if (threadIdx.x == 0) carry = 0;
  __syncthreads();
  const uint32_t lane = threadIdx.x % 64, w = threadIdx.x / 64;
  for (uint32_t b0 = 0; b0 < nb; b0 += kScanBlock) {
    const uint32_t b = b0 + threadIdx.x;
    const uint64_t x = b < nb ? sums[b] : 0;
    uint64_t incl = x;
    for (int off = 1; off < 64; off <<= 1) {
      const uint64_t o = __shfl_up(incl, off, 64);
      if (lane >= (uint32_t)off) incl += o;
    }
    if (lane == 63) warp_tot[w] = incl;
    __syncthreads();
    uint64_t before = carry;
    for (uint32_t q = 0; q < w; ++q) before += warp_tot[q];
    if (b < nb) sums[b] = before + incl - x;
    __syncthreads();
    if (threadIdx.x == kScanBlock - 1) carry = before + incl;
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    doc_index[n_docs] = carry;
    st->go = !st->bad && carry <= payload_len;
    st->slices = st->n_slices;
    __hip_atomic_store(host, st->bad, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __hip_atomic_store(host + 1, (uint32_t)carry, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __hip_atomic_store(host + 2, (uint32_t)(carry >> 32), __ATOMIC_RELAXED,
                       __HIP_MEMORY_SCOPE_SYSTEM);
    st->bad = 0;
    st->n_slices = 0;
  }
}

// Tokens [k0, k1) of a document of n_d tokens at p, by one wave: n_d (with the
// first token), the centroid ids, the codes (as 32-bit words when source and
// size allow; the id array is 4-aligned, as document starts are 8-aligned)
// and, behind the last token, zero padding.
__device__ __forceinline__ void doc_copy(uint32_t lane, uint64_t lo, uint64_t n_d, uint64_t k0,
                                         uint64_t k1, uint8_t* p, const uint32_t* assign,
                                         const uint8_t* codes, uint32_t m, uint32_t cb) {
  uint32_t* ids = reinterpret_cast<uint32_t*>(p + 4);
  if (lane == 0 && k0 == 0) *reinterpret_cast<uint32_t*>(p) = (uint32_t)n_d;
  for (uint64_t k = k0 + lane; k < k1; k += 64) ids[k] = assign[lo + k];
  const uint64_t row = (uint64_t)m * cb, nbytes = (k1 - k0) * row;
  const uint8_t* src = codes + (lo + k0) * row;
  uint8_t* dst = p + 4 + 4 * n_d + k0 * row;
  if ((((uintptr_t)src | (uintptr_t)dst | nbytes) & 3) == 0) {
    const uint32_t* s4 = reinterpret_cast<const uint32_t*>(src);
    uint32_t* d4 = reinterpret_cast<uint32_t*>(dst);
    for (uint64_t q = lane; q < nbytes / 4; q += 64) d4[q] = s4[q];
  } else {
    for (uint64_t q = lane; q < nbytes; q += 64) dst[q] = src[q];
  }
  if (k1 < n_d) return;
  const uint64_t total = doc_bytes(n_d, m, cb);
  for (uint64_t q = 4 + 4 * n_d + n_d * row + lane; q < total; q += 64) p[q] = 0;
}

// Phase 3: adds each scan block's carry-in to the document's offset and writes
// the layouts, one wave per slice or per `group` (at most 64) consecutive
// documents, whose offsets its lanes load at once (grid-stride).
__global__ __launch_bounds__(256) void doc_write_kernel(
    const uint64_t* __restrict__ doc_offsets, uint64_t n_docs, const uint32_t* __restrict__ assign,
    const uint8_t* __restrict__ codes, uint32_t m, uint32_t cb,
    const uint64_t* __restrict__ sums, uint64_t* __restrict__ doc_index,
    uint8_t* __restrict__ payload, uint32_t group, const DocState* __restrict__ st,
    const DocSlice* __restrict__ slices) {
  const uint32_t lane = threadIdx.x % 64;
  const uint64_t waves = (uint64_t)gridDim.x * (blockDim.x / 64);
  const uint64_t wave = (uint64_t)blockIdx.x * (blockDim.x / 64) + threadIdx.x / 64;
  const bool go = st->go != 0;
  const uint64_t n_slices = go ? st->slices : 0;
  for (uint64_t i = wave; i < n_slices; i += waves) {
    const DocSlice sl = slices[i];
    const uint64_t lo = doc_offsets[sl.doc], n_d = doc_offsets[sl.doc + 1] - lo;
    const uint64_t k1 = n_d - sl.first < kDocSlice ? n_d : sl.first + kDocSlice;
    doc_copy(lane, lo, n_d, sl.first, k1,
             payload + sl.at + sums[sl.doc / (kScanBlock * kScanPer)], assign, codes, m, cb);
  }
  for (uint64_t base = wave * group; base < n_docs; base += waves * group) {
    const uint32_t cnt = n_docs - base < group ? (uint32_t)(n_docs - base) : group;
    const uint64_t d = base + lane;
    uint64_t lo = 0, n_d = 0, at = 0;
    if (lane < cnt) {
      lo = doc_offsets[d];
      n_d = doc_offsets[d + 1] - lo;
      at = doc_index[d] + sums[d / (kScanBlock * kScanPer)];
      doc_index[d] = at;
    }
    if (!go) continue;
    for (uint32_t k = 0; k < cnt; ++k) {
      const uint64_t n_k = readlane_u64(n_d, k);
      if (n_k <= kDocSlice)
        doc_copy(lane, readlane_u64(lo, k), n_k, 0, n_k, payload + readlane_u64(at, k), assign,
                 codes, m, cb);
    }
  }
}

// ---------------------------------------------------------------------------
// CRC-32/ISO-HDLC of a device buffer (std.hash.Crc32, as storage.zig applies
// it to the whole image before the footer, :612-617, :782-786).
//
// Polynomials over GF(2) mod P, reflected: bit 31 holds the coefficient of
// x^0, so a little-endian word of the buffer is a polynomial as it stands.
// The CRC of n bytes B is B(x) x^32 + ones(x) x^(8n) mod P, complemented.
// The kernel evaluates B(x), padded with zero bytes to whole blocks, and the
// host applies x^32, the inverse of the padding and the preset.
//
// A block owns consecutive chunks of kCrcChunk bytes and walks them in steps
// of 8 KB: every lane loads 16 bytes a step (coalesced, a chunk's loads in
// flight at once) into four Horner sums of one word each, s <- s x^(8 * 8192)
// + word.  The product by a constant is four LDS table reads, one a byte of
// s.  What is left is the 8 KB polynomial of the block's 512 lanes: each lane
// joins its four words and multiplies by its own power of x, the block XORs
// the lanes and multiplies by x^(8 * bytes behind its chunks), and stores one
// word to pinned host memory, where the host XORs the blocks' words.
//
// Bound by the table reads in LDS (one a byte and lane, random banks) and by
// latency.  One leaf of 256 bytes a thread read the buffer 64 lines an
// instruction and built its tables in every block, and one more block joined
// the results in a chain: 20 + 25 us for 30.6 MB.  This kernel takes 14 us; with the lanes
// and waves folded in a tree by one wave and the blocks XORed by device
// atomics on one word it took 24.
// ---------------------------------------------------------------------------
constexpr uint32_t kCrcPoly = 0xEDB88320u;
constexpr uint32_t kCrcInvX = 0xDB710641u;  // x^-1 mod P
constexpr uint32_t kCrcOne = 0x80000000u;   // x^0
constexpr uint32_t kCrcThreads = 512;
constexpr uint32_t kCrcSteps = 8;  // loads of a lane in flight
constexpr uint32_t kCrcStepBytes = kCrcThreads * 16;
constexpr uint32_t kCrcChunk = kCrcSteps * kCrcStepBytes;
constexpr uint32_t kCrcBlocks = 1024;  // most blocks, a host word each

inline uint32_t crc_mulmod(uint32_t a, uint32_t b) {
  uint32_t p = 0;
  for (int i = 0; i < 32; ++i) {
    if ((a >> (31 - i)) & 1u) p ^= b;
    b = (b & 1u) ? (b >> 1) ^ kCrcPoly : b >> 1;
  }
  return p;
}

// base^e mod P.
inline uint32_t crc_pow(uint32_t base, uint64_t e) {
  uint32_t r = kCrcOne;
  for (; e; e >>= 1, base = crc_mulmod(base, base))
    if (e & 1u) r = crc_mulmod(r, base);
  return r;
}

// Device tables, in words: products of the four bytes of a word by x^(8 *
// kCrcStepBytes) and by x^32, entry [byte][value]; x^(128 i), the weight of
// the lane i places before the last; and the powers x^(8 kCrcChunk i 256^l),
// entry [l][i].
constexpr uint32_t kCrcTabStep = 0, kCrcTabWord = 1024, kCrcTabLane = 2048,
                   kCrcTabPow = kCrcTabLane + kCrcThreads, kCrcTabWords = kCrcTabPow + 1024;

inline void crc_tables_host(uint32_t* t) {
  const uint32_t x = kCrcOne >> 1;
  const uint32_t by[2] = {crc_pow(x, 8ull * kCrcStepBytes), crc_pow(x, 32)};
  for (uint32_t k = 0; k < 2; ++k)
    for (uint32_t b = 0; b < 4; ++b)
      for (uint32_t v = 0; v < 256; ++v)
        t[k * 1024 + b * 256 + v] = crc_mulmod(v << (8 * b), by[k]);
  uint32_t unit = crc_pow(x, 128), p = kCrcOne;
  for (uint32_t i = 0; i < kCrcThreads; ++i, p = crc_mulmod(p, unit)) t[kCrcTabLane + i] = p;
  unit = crc_pow(x, 8ull * kCrcChunk);
  for (uint32_t l = 0; l < 4; ++l) {
    p = kCrcOne;
    for (uint32_t i = 0; i < 256; ++i, p = crc_mulmod(p, unit)) t[kCrcTabPow + l * 256 + i] = p;
    unit = p;  // unit^256
  }
}

// The CRC of len bytes from the kernel's polynomial over the bytes and `pad`
// zero bytes behind them.
inline uint32_t crc_finish(uint32_t raw, uint32_t x32_over_pad, uint32_t preset) {
  return crc_mulmod(raw, x32_over_pad) ^ preset ^ 0xFFFFFFFFu;
}

// s times the table's constant.
__device__ __forceinline__ uint32_t crc_times(uint32_t s, const uint32_t* tab) {
  return tab[s & 0xFFu] ^ tab[256 + ((s >> 8) & 0xFFu)] ^ tab[512 + ((s >> 16) & 0xFFu)] ^
         tab[768 + (s >> 24)];
}

// a b mod P: the 64-bit carry-less product, its low word (the powers from
// x^32 on) reduced through the x^32 table.
__device__ __forceinline__ uint32_t crc_mul(uint32_t a, uint32_t b, const uint32_t* word_tab) {
  uint32_t lo = 0, hi = 0;  // of the product shifted left by one
#pragma unroll
  for (int i = 0; i < 32; ++i) {
    const uint32_t m = (uint32_t)((int32_t)(a << (31 - i)) >> 31);
    if (i < 31) lo ^= (b << (i + 1)) & m;
    hi ^= (b >> (31 - i)) & m;
  }
  return hi ^ crc_times(lo, word_tab);
}

// The 16 bytes at `pos` from base (16-byte aligned); bytes outside
// [first, end) are zero and not read.
__device__ __forceinline__ uint4 crc_load(const uint8_t* base, uint64_t pos, uint64_t first,
                                          uint64_t end) {
  if (pos >= first && pos + 16 <= end) return *reinterpret_cast<const uint4*>(base + pos);
  uint32_t v[4] = {0, 0, 0, 0};
  if (pos + 16 > first && pos < end)
    for (uint32_t b = 0; b < 16; ++b)
      if (pos + b >= first && pos + b < end) v[b / 4] |= (uint32_t)base[pos + b] << (8 * (b % 4));
  return make_uint4(v[0], v[1], v[2], v[3]);
}

// Bytes [first, end) from base, n_chunks chunks, `per` to a block; block b's
// word goes to host_out[b].
__global__ __launch_bounds__(kCrcThreads) void crc_kernel(
    const uint8_t* __restrict__ base, uint64_t first, uint64_t end, uint32_t n_chunks,
    uint32_t per, const uint32_t* __restrict__ tables, uint32_t* __restrict__ host_out) {
  __shared__ __attribute__((aligned(16))) uint32_t tab[2 * 1024];
  __shared__ uint32_t wave_word[kCrcThreads / 64];
  __shared__ uint32_t weight;
  const uint32_t t = threadIdx.x;
  const uint32_t c0 = blockIdx.x * per;
  const uint32_t c1 = n_chunks - c0 < per ? n_chunks : c0 + per;
  uint4 v[kCrcSteps];
  auto load = [&](uint32_t c) {
    const uint64_t lo = (uint64_t)c * kCrcChunk;
    if (lo >= first && lo + kCrcChunk <= end) {
      const uint4* p = reinterpret_cast<const uint4*>(base + lo) + t;
#pragma unroll
      for (uint32_t j = 0; j < kCrcSteps; ++j) v[j] = p[j * kCrcThreads];
    } else {
#pragma unroll
      for (uint32_t j = 0; j < kCrcSteps; ++j)
        v[j] = crc_load(base, lo + j * kCrcStepBytes + t * 16, first, end);
    }
  };
  load(c0);
  for (uint32_t f = t; f < 2 * 1024 / 4; f += kCrcThreads)
    reinterpret_cast<uint4*>(tab)[f] = reinterpret_cast<const uint4*>(tables)[f];
  const uint32_t lane_weight = tables[kCrcTabLane + kCrcThreads - 1 - t];
  // the chunks behind the block, in base 256: the last wave's first lane
  // multiplies their powers while the others fold
  const uint32_t behind = n_chunks - c1;
  uint32_t pw[4];
#pragma unroll
  for (uint32_t l = 0; l < 4; ++l)
    pw[l] = tables[kCrcTabPow + l * 256 + ((behind >> (8 * l)) & 0xFFu)];
  __syncthreads();
  uint32_t s[4] = {0, 0, 0, 0};
  for (uint32_t c = c0;;) {
#pragma unroll
    for (uint32_t j = 0; j < kCrcSteps; ++j) {
      const uint32_t word[4] = {v[j].x, v[j].y, v[j].z, v[j].w};
#pragma unroll
      for (int q = 0; q < 4; ++q) s[q] = crc_times(s[q], tab + kCrcTabStep) ^ word[q];
    }
    if (++c >= c1) break;
    load(c);
  }
  uint32_t r = s[0];
#pragma unroll
  for (int q = 1; q < 4; ++q) r = crc_times(r, tab + kCrcTabWord) ^ s[q];
  r = crc_mul(r, lane_weight, tab + kCrcTabWord);
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) r ^= __shfl_xor(r, off, 64);
  if (t % 64 == 0) wave_word[t / 64] = r;
  if (t == kCrcThreads - 64) {
    uint32_t f = pw[0];
    for (uint32_t l = 1; l < 4 && behind >> (8 * l); ++l)
      f = crc_mul(f, l == 1 ? pw[1] : l == 2 ? pw[2] : pw[3], tab + kCrcTabWord);
    weight = f;
  }
  __syncthreads();
  if (t != 0) return;
#pragma unroll
  for (uint32_t ww = 1; ww < kCrcThreads / 64; ++ww) r ^= wave_word[ww];
  __hip_atomic_store(host_out + blockIdx.x, crc_mul(r, weight, tab + kCrcTabWord),
                     __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

}  // namespace tacgpu
