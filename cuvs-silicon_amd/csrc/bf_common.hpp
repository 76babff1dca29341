// Definitions shared by the brute-force kernels of bf_search.hip (the
// streaming scan, sample, select, merge) and bf_gemm.hip (the register-
// blocked scan of large query batches): operand types, the candidate-list
// geometry and the list compaction, and the large-batch launcher.
#pragma once

#include <cstdint>

#include "cvs_internal.hpp"
#include "device_util.hpp"

namespace cvs {
namespace bf {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

#define CVS_INLINE __attribute__((always_inline))

constexpr uint64_t kSentinel = ~0ull;
// Buffer resource word 3 for raw (untyped) buffer access on gfx9-family
// targets, and the non-temporal cache policy for the streamed dataset.
constexpr int kRsrcWord3 = 0x00020000;
constexpr int kAuxNT = 2;

using rsrc4 = int __attribute__((ext_vector_type(4)));

// Buffer load straight to LDS (buffer_load ... lds): lane l writes kBytes at
// LDS byte address m0 + kBytes * l (m0 the same for every lane).  Written as
// inline assembly so that the compiler does not wait for every outstanding
// load before each later LDS read (it cannot tell which LDS bytes the load
// writes); the kernel orders these loads and the reads of their data with
// explicit s_waitcnt vmcnt and barriers.  M0 is an input operand, so the
// compiler knows it changes; one wait state separates its write from the
// load that reads it.
template <int kBytes, bool kNT>
__device__ CVS_INLINE void lds_dma(rsrc4 rs, int m0, uint32_t voff, int soff) {
  if constexpr (kBytes == 16 && kNT)
    asm volatile("s_nop 0\n\tbuffer_load_dwordx4 %0, %1, %2 offen nt lds"
                 :: "v"(voff), "s"(rs), "s"(soff), "{m0}"(m0) : "memory");
  else if constexpr (kBytes == 16)
    asm volatile("s_nop 0\n\tbuffer_load_dwordx4 %0, %1, %2 offen lds"
                 :: "v"(voff), "s"(rs), "s"(soff), "{m0}"(m0) : "memory");
  else
    asm volatile("s_nop 0\n\tbuffer_load_dword %0, %1, %2 offen lds"
                 :: "v"(voff), "s"(rs), "s"(soff), "{m0}"(m0) : "memory");
}

// Raw buffer descriptor: 48-bit base, stride 0, num_records bytes.
__device__ CVS_INLINE rsrc4 make_rsrc(const void* base, int bytes) {
  const uint64_t b = reinterpret_cast<uint64_t>(base);
  rsrc4 r;
  r.x = int(uint32_t(b));
  r.y = int(uint32_t(b >> 32) & 0xFFFFu);
  r.z = bytes;
  r.w = kRsrcWord3;
  return r;
}

// LDS byte address of p, in a scalar register.
__device__ CVS_INLINE int lds_addr(const void* p) {
  return __builtin_amdgcn_readfirstlane(
      int(uint32_t(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) const void*)p))));
}

enum { kModeScan = 0, kModeSample = 1 };

// List geometry per kp.  Each (workgroup, query) list is split into two
// halves, one per lane holding that query (lanes l and l + 32 see different
// rows of every tile), so each lane appends to its own half with a counter
// in a register and no atomics.  A lane adds at most one key between two
// fill checks; a half that fills up (HALF keys) rebalances the query's list
// to its kp smallest keys, kp/2 per half, so the slack HALF - kp/2 sets how
// many appends one compaction is amortized over.  Lists of kp <= 64 live in
// LDS (bounded by the 160 KiB budget next to the stage buffers); kp = 128
// lists (large k) live in global memory, one per (query, workgroup), since
// 128 queries x 192 keys exceed the LDS budget and appends are rare once the
// sampled threshold is in place.
template <int KP, int MODE>
struct Lists {
  static constexpr bool GL = MODE == 0 && KP > 64;  // lists in global memory
  static constexpr int HALF = MODE != 0 ? 1 : (KP == 16 ? 40 : (KP <= 64 ? 44 : 96));
  static constexpr int CAP = 2 * HALF;
  static constexpr int NS = (CAP + 63) / 64;  // list entries per lane in a compaction
  static_assert(MODE != 0 || HALF >= KP / 2 + 8, "list slack");
};

// Rewrites the two-half list of one query (c0 keys at list[0..), c1 keys at
// list[half..)) as its kp smallest keys, the first kp/2 in half 0 and the
// rest in half 1, and returns the order image of the kp-th smallest distance
// (0xffffffff when c0 + c1 <= kp: every key is kept and the threshold stays).
// All 64 lanes take part (list, c0 and c1 are wave-uniform); entry e lives in
// lane e % 64, slot e / 64.  Every entry is read before any is written.
template <int NS>
__device__ __forceinline__ uint32_t compact_query(uint64_t* list, int half, uint32_t c0, uint32_t c1,
                                                  int kp) {
  const int lane = __lane_id();
  const uint32_t cnt = c0 + c1;
  bool v[NS];
  uint64_t k[NS];
  uint32_t h[NS], l[NS];
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    const uint32_t e = uint32_t(lane + 64 * s);
    v[s] = e < uint32_t(half) ? e < c0 : (e - uint32_t(half)) < c1;
    k[s] = v[s] ? list[e] : kSentinel;
    h[s] = uint32_t(k[s] >> 32);
    l[s] = uint32_t(k[s]);
  }
  uint32_t kth_hi = 0xffffffffu, kth_lo = 0xffffffffu;
  if (cnt > uint32_t(kp)) {
    int need = kp;
    uint32_t pre = 0;
    for (int b = 31; b >= 0; --b) {
      int c = 0;
#pragma unroll
      for (int s = 0; s < NS; ++s) c += popc(__ballot(v[s] && ((h[s] ^ pre) >> b) == 0));
      if (c < need) {
        need -= c;
        pre |= 1u << b;
      }
    }
    kth_hi = pre;
    int lt = 0, eq = 0;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
      lt += popc(__ballot(v[s] && h[s] < kth_hi));
      eq += popc(__ballot(v[s] && h[s] == kth_hi));
    }
    if (eq > kp - lt) {  // ties on the distance word: select on the row id
      int need2 = kp - lt;
      uint32_t pre2 = 0;
      for (int b = 31; b >= 0; --b) {
        int c = 0;
#pragma unroll
        for (int s = 0; s < NS; ++s) c += popc(__ballot(v[s] && h[s] == kth_hi && ((l[s] ^ pre2) >> b) == 0));
        if (c < need2) {
          need2 -= c;
          pre2 |= 1u << b;
        }
      }
      kth_lo = pre2;
    }
  }
  const int kh = kp / 2;
  int base = 0;
#pragma unroll
  for (int s = 0; s < NS; ++s) {
    const bool keep = v[s] && (h[s] < kth_hi || (h[s] == kth_hi && l[s] <= kth_lo));
    const uint64_t m = __ballot(keep);
    const int p = base + mbcnt(m);
    if (keep) list[p < kh ? p : half + (p - kh)] = k[s];
    base += popc(m);
  }
  return cnt > uint32_t(kp) ? kth_hi : 0xffffffffu;
}

// ---------------------------------------------------------------------------
// Certificate of the fp16 selection.  A row's key is d~ = |q~|^2 + |x~|^2 -
// 2 q~.x~ in fp32, with q~, x~ the fp16 copies of s (q - mu), s (x - mu).  For
// the scaled exact distance D = s^2 |q - x|^2:
//   |d~ - |q~ - x~|^2| <= A = 2 (d + 16) 2^-24 (|q~| + rmax)^2
// (fp32 sums of d terms, including an MFMA accumulation that rounds twice
// per step, and the two final operations), and
//   | |q~ - x~| - sqrt(D) | <= E = |q~ - s(q - mu)| + dx
// (triangle inequality; dx bounds every row's rounding, measured when the
// dataset was made).  Hence D >= lb(d~) = (sqrt(d~ - A) - E)^2 when
// sqrt(d~ - A) > E, and 0 otherwise: a row whose key is at least T has an
// exact distance of at least lb(T) / s^2.
//
// The merge re-ranks the R smallest keys it holds exactly in fp32.  Every row
// not re-ranked has a key at or above T = min(key of the R-th candidate, the
// smallest final list threshold T*) (a list keeps every key of its range
// below its threshold).  If lb(T) exceeds s^2 d_k (1 + rho), with d_k the
// k-th exact distance and rho the relative error of the fp32 distances
// themselves, the result is the exact top k.  Otherwise the query
// escalates: every row with a key up to T_need = (sqrt(s^2 d_k (1 + rho)) +
// E)^2 + A (all of them are in the lists when T_need <= T*), or else every
// row of the dataset, is re-ranked exactly, and the top k of those is the
// answer.
// ---------------------------------------------------------------------------
struct Cert {
  float s2;              // scale^2: key units per squared distance unit
  float rmax;            // every row: |x~| <= rmax (scaled units)
  float dx;              // every row: |x~ - s (x - mu)| <= dx
  float a_coef;          // 2 (d + 16) 2^-24
  float rho;             // 2 (d + 8) 2^-24
  float qslack;          // sqrt(d) 2^-25 + fp32 error of a query's centring
  const float* qnorms;   // |q~|^2 per query
  const float* qerr;     // |q~ - s fl(q - mu)|^2 per query
  unsigned long long* counters;  // [0] escalated queries, [1] of them re-ranked over every row
};

enum { kCertPass = 0, kCertKeys = 1, kCertAll = 2 };

// Exact squared L2 distances of U rows to the query by the 64 lanes of the
// calling wave (ids >= n count as none and give 0).  The summation order is
// fixed: per lane, float4 partial sums over its 4-column pieces of 256-column
// chunks, then a butterfly, so a row always gets the same value.  All row
// loads of a 1024-column pass are issued before the first is used.
// Up to 128 columns the upper 32 lanes would add zeros: there each half of
// the wave takes a row of its own, for the same sums.
__device__ __forceinline__ float sum_sq4(const float4& a, const float4& b) {
  const float t0 = a.x - b.x, t1 = a.y - b.y, t2 = a.z - b.z, t3 = a.w - b.w;
  return __fadd_rn(__builtin_fmaf(t1, t1, __fmul_rn(t0, t0)), __builtin_fmaf(t3, t3, __fmul_rn(t2, t2)));
}

// One pass over NC chunks of 256 columns from column i0 (this lane's first).
template <int U, int NC>
__device__ __forceinline__ void exact_chunks(const uint32_t (&id)[U], const float* __restrict__ rows, int64_t n,
                                             int64_t d, const float* __restrict__ qv, int64_t i0, float (&acc)[U]) {
  float4 a4[NC], b4[NC][U];
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    const int64_t i = i0 + c * 256;
    a4[c] = i < d ? *reinterpret_cast<const float4*>(qv + i) : float4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < U; ++u)
      b4[c][u] = (i < d && int64_t(id[u]) < n) ? *reinterpret_cast<const float4*>(rows + int64_t(id[u]) * d + i)
                                               : float4{0.f, 0.f, 0.f, 0.f};
  }
#pragma unroll
  for (int c = 0; c < NC; ++c)
#pragma unroll
    for (int u = 0; u < U; ++u) acc[u] = __fadd_rn(acc[u], sum_sq4(a4[c], b4[c][u]));
}

template <int U>
__device__ __forceinline__ void wave_exact(const uint32_t (&id)[U], const float* __restrict__ rows, int64_t n,
                                           int64_t d, const float* __restrict__ qv, bool vec, float (&out)[U]) {
  static_assert(U % 2 == 0, "rows in pairs");
  const int lane = threadIdx.x & 63;
  if (vec && d <= 128) {
    uint32_t mine[U / 2];
    float acc[U / 2];
#pragma unroll
    for (int u = 0; u < U / 2; ++u) {
      mine[u] = lane < 32 ? id[2 * u] : id[2 * u + 1];
      acc[u] = 0.f;
    }
    exact_chunks<U / 2, 1>(mine, rows, n, d, qv, int64_t(lane & 31) * 4, acc);
#pragma unroll
    for (int u = 0; u < U / 2; ++u) {
#pragma unroll
      for (int o = 16; o >= 1; o >>= 1) acc[u] += xor_lanes_f(acc[u], o);
      out[2 * u] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(acc[u]), 0));
      out[2 * u + 1] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(acc[u]), 32));
    }
    return;
  }
  float acc[U];
#pragma unroll
  for (int u = 0; u < U; ++u) acc[u] = 0.f;
  if (vec) {
    for (int64_t c0 = 0; c0 < d; c0 += 4 * 256) {
      const int64_t i0 = c0 + int64_t(lane) * 4;
      if (d - c0 > 768)
        exact_chunks<U, 4>(id, rows, n, d, qv, i0, acc);
      else if (d - c0 > 512)
        exact_chunks<U, 3>(id, rows, n, d, qv, i0, acc);
      else if (d - c0 > 256)
        exact_chunks<U, 2>(id, rows, n, d, qv, i0, acc);
      else
        exact_chunks<U, 1>(id, rows, n, d, qv, i0, acc);
    }
  } else {
    // Rows that are not 16-byte aligned: one column per lane and load.  The
    // loads of eight columns of every row go out together, at clamped
    // indices so that none sits under a condition (each was waited for
    // before the next: the merge of 37 queries at d = 771 took 52.8 us, 27.3
    // us now); a value past the row is dropped after its load, and the sum runs
    // over the columns in the same order as one at a time.
    constexpr int C = 8;
    for (int64_t i0 = lane; i0 < d; i0 += 64 * C) {
      float a1[C], b1[C][U];
#pragma unroll
      for (int c = 0; c < C; ++c) {
        const int64_t i = i0 + 64 * c < d ? i0 + 64 * c : d - 1;
        a1[c] = qv[i];
#pragma unroll
        for (int u = 0; u < U; ++u) b1[c][u] = rows[(int64_t(id[u]) < n ? int64_t(id[u]) : 0) * d + i];
      }
#pragma unroll
      for (int c = 0; c < C; ++c)
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const float t = a1[c] - b1[c][u];
          acc[u] = i0 + 64 * c < d && int64_t(id[u]) < n ? acc[u] + t * t : acc[u];
        }
    }
  }
#pragma unroll
  for (int u = 0; u < U; ++u) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) acc[u] += xor_lanes_f(acc[u], o);
    out[u] = acc[u];
  }
}

constexpr int kExactU = 8;  // rows per wave and pass of the exact distances

// Exact keys ord(d) << 32 | id of the ids s_id[0..cnt) (a wave's own list),
// into s_key[0..cnt), by the calling wave.
__device__ __forceinline__ void wave_exact_keys(const uint32_t* s_id, int cnt, uint64_t* s_key, const float* rows,
                                                int64_t n, int64_t d, const float* qv, bool vec) {
  const int lane = threadIdx.x & 63;
  for (int c = 0; c < cnt; c += kExactU) {
    uint32_t id[kExactU];
#pragma unroll
    for (int u = 0; u < kExactU; ++u) id[u] = c + u < cnt ? s_id[c + u] : 0xffffffffu;
    float dd[kExactU];
    wave_exact<kExactU>(id, rows, n, d, qv, vec, dd);
#pragma unroll
    for (int u = 0; u < kExactU; ++u)
      if (lane == u && c + u < cnt) s_key[c + u] = (uint64_t(ord_f32(dd[u])) << 32) | id[u];
  }
}

// Certificate constants of a search over `ds` (defined in bf_search.hip).
Cert make_cert(cvs_context* ctx, const cvs_dataset* ds, const float* qnorms, const float* qerr);

// Converts q queries (device, q x d fp32) into q_rows / 32 query tiles of
// the dataset's layout and centring, their norms (q_rows, +inf past q) and
// squared rounding errors (q), on the context stream (bf_search.hip).
void launch_query_tiles(cvs_context* ctx, const cvs_dataset* ds, const float* queries, int64_t q, int64_t q_rows,
                        u32x4* qtiles, float* qnorms, float* qerr, hipEvent_t e0, hipEvent_t e1);

// Exact k-NN outside the fused scan's limits (d > 1024 or k > 112): fp16
// MFMA keys of a query chunk against every row, listed below a sampled
// per-query threshold (a radix select over the full key matrix where the list
// does not serve), and the certified exact re-rank (bf_wide.hip).  Device
// pointers, context stream.
void bf_wide_search(cvs_context* ctx, const cvs_dataset* ds, const float* queries, int64_t q, int64_t k,
                    uint32_t* nbr, float* dist);
constexpr int64_t kFusedMaxDim = 1024;  // the fused scan holds a query tile's operands for d <= 1024
constexpr int64_t kFusedMaxK = 112;     // and keeps up to 128 candidates per query

// Arguments of the register-blocked large-batch scan (bf_gemm.hip).  The
// candidate lists and their minima have the streaming scan's global-list
// layout: part[q][list][Lists<128, kModeScan>::CAP], first kp valid.
struct GemmArgs {
  const u32x4* tiles;   // dataset tiles (unit-padded; n_tiles a multiple of 64)
  const float* norms;   // dataset norms, 32 per tile
  int64_t n_rt;         // 128-row blocks of the dataset (n_tiles / 4)
  int ks;               // k-steps per tile (padded dimension / 16)
  const u32x4* qtiles;  // query tiles
  const float* qnorms;  // query norms, 32 per query tile
  int nq;
  int n_qtiles;         // number of 32-query tiles
  const float* thr0;    // per-query initial threshold
  uint64_t* part;       // [nq][n_lists][CAP] lists
  uint64_t* lmin;       // [nq][n_lists] smallest key of each list
  float* lcut;          // [nq][n_lists] final threshold of each list (rows it covers and does
                        // not hold have keys at or above it; +inf for an unused list)
  int n_lists;          // lists per query
};

// Launch shape of the register-blocked scan: n_wg workgroups (a multiple of
// 8) and n_lists candidate lists per query.  ok is false when the call is
// not one it handles (kp = 128 lists, 8 to 64 k-steps per tile, buffer and
// stage-count limits).
struct GemmPlan {
  bool ok = false;
  int n_wg = 0;
  int n_lists = 0;
};
GemmPlan plan_gemm_scan(int ks, int kp, int64_t n_rt, int n_qtiles, int compute_units);
// Launches it on the context stream; e0 / e1 (may be null) record the
// dispatch's start and end.
void launch_gemm_scan(cvs_context* ctx, const GemmArgs& args, int n_wg, hipEvent_t e0, hipEvent_t e1);

// Arguments of the large-batch scan over narrow rows (bf_batch.hip).  Its
// candidate lists are global for every kp: part[q][range][2 * batch_half(kp)],
// first kp valid at the end.
constexpr int batch_half(int kp) { return kp / 2 + 32; }
constexpr int kBatchMaxRanges = 128;
struct BatchArgs {
  const u32x4* tiles;   // dataset tiles
  const float* norms;   // dataset norms, 32 per tile
  int64_t n_tiles;
  const u32x4* qtiles;  // query tiles
  const float* qnorms;  // query norms, 32 per query tile
  int nq;
  int n_qtiles;
  const float* thr0;    // per-query initial threshold
  uint64_t* part;
  uint64_t* lmin;       // [nq][n_ranges] smallest key of each list
  float* lcut;          // [nq][n_ranges] final threshold of each list
  int n_ranges;
  int n_qblocks;
};
struct BatchPlan {
  bool ok = false;      // false: not a shape it handles, or not the faster scan there
  int n_ranges = 0;     // candidate lists per query
  int n_qblocks = 0;
};
BatchPlan plan_batch_scan(int ks, int kp, int64_t q, int64_t n, int64_t n_tiles, int compute_units);
void launch_batch_scan(cvs_context* ctx, const BatchArgs& args, int ks, int kp, hipEvent_t e0, hipEvent_t e1);

}  // namespace bf
}  // namespace cvs
