// Exact-search scan of large query batches over narrow rows (gfx950): 8 to 20
// k-steps per tile (d from 65 to 320), more than 1,024 queries, but for small
// calls (pays, below).
//
// With few k-steps per row tile the two other scans spend their time beside
// the matrix cores: the streaming scan (bf_search.hip) reads one LDS fragment
// per MFMA, and the register-blocked scan (bf_gemm.hip) has one wave per SIMD,
// whose epilogue (every distance formed and tested, candidates appended) then
// stands against only 4 k-steps' MFMAs with nothing to overlap it.  Here a
// wave keeps the operands of two query tiles for the whole dimension in
// registers (8 KS of them), so that a row fragment read from LDS serves two
// MFMAs and queries are read once, and two or three waves share a SIMD, one's
// epilogue under the others' MFMAs.
//
//  - A workgroup of 4 (8 k-steps) or 8 waves covers 256 or 512 queries and a
//    contiguous range of row tiles, streamed through two LDS buffers by loads
//    straight into LDS.
//  - Per 32 x 32 block a lane forms |x|^2 - 2 q.x for its 16 rows and their
//    minimum; only a block with a distance below some query's threshold is
//    looked at further, four rows at a time.  A passing lane appends
//    (distance, row) to its half of its query's list in global memory; a half
//    with less room than one block's 16 rows is first compacted to the kp
//    smallest keys.
//
// 10,000 queries, K = 100, 1M x 128: the register-blocked scan took 6.71 ms,
// this one 3.02 to 3.2 (2.56 TFLOP: 0.34 of the 2.5 PFLOP/s peak; the SIMDs'
// cycles: MFMA busy 0.42, other vector instructions 0.35).  What is left is
// latency that three waves do not hide: they wait 0.46 of their cycles.  Four query tiles per wave at two waves per SIMD
// took 3.28 ms (4.25 with the rows staged through registers, which spilled),
// and left small batches short of workgroups: 1,500 queries K = 10 1M x 128
// 717 us, 575 now, 1,314 as the streaming scan.
#include <algorithm>

#include "bf_common.hpp"

namespace cvs {
namespace bf {
namespace {

// Smallest of three; skips NaN, which passes no threshold either.  (fminf
// costs a canonicalising instruction per operand.)
__device__ CVS_INLINE float min3(float x, float y, float z) {
  float r;
  asm("v_min3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(x), "v"(y), "v"(z));
  return r;
}

template <int KS>
struct BatchCfg {
  static constexpr int QW = 2;                      // query tiles per wave
  static constexpr int TPS = 2;                     // row tiles per stage
  static constexpr int W = KS <= 8 ? 4 : 8;         // waves
  static constexpr int T = 64 * W;
  static constexpr int PER_SIMD = KS <= 8 ? 3 : 2;  // waves per SIMD
  static constexpr int VECS = KS * TPS * 64;        // 16-byte vectors per stage
  static constexpr int LPW = VECS / T;      // 1 KiB loads per wave and stage
  static constexpr int QB = W * QW * 32;      // queries per workgroup
  static_assert(VECS % T == 0, "whole loads");
};

template <int KS, int KP>
__global__ __launch_bounds__(BatchCfg<KS>::T, BatchCfg<KS>::PER_SIMD) void bf_batch_scan_kernel(BatchArgs a) {
  using C = BatchCfg<KS>;
  constexpr int QW = C::QW, TPS = C::TPS, kBThreads = C::T;
  constexpr int HALF = batch_half(KP), CAP = 2 * HALF;
  constexpr int NS = (CAP + 63) / 64;
  __shared__ u32x4 s_stage[2][C::VECS];
  __shared__ float s_dn[2][TPS * 32];
  const int tid = threadIdx.x, lane = tid & 63, half = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int G = a.n_ranges;
  const int x = int(blockIdx.x) / a.n_qblocks;  // range-major: a range's query blocks run together
  const int q0 = (int(blockIdx.x) % a.n_qblocks) * C::QB + wave * (QW * 32);  // first query of this wave

  // This workgroup's stages of TPS tiles (the tile count is a multiple of 64).
  const int64_t total = a.n_tiles / TPS;
  const int64_t st0 = total * x / G, st1 = total * (x + 1) / G;
  const int n_stages = int(st1 - st0);
  // Straight into LDS (no registers held): the loads of a stage are issued a
  // whole stage before the barrier that publishes it.  They are inline
  // assembly that the compiler does not count, so each wave waits for its own
  // at the end of a stage.  A stage past the last reads the last one again.
  const rsrc4 rs = make_rsrc(a.tiles + st0 * C::VECS, n_stages * C::VECS * 16);
  const rsrc4 ns = make_rsrc(a.norms + st0 * (TPS * 32), n_stages * TPS * 128);
  const int lds0 = lds_addr(&s_stage[0][wave * 64]), ldn0 = lds_addr(&s_dn[0][0]);
  const uint32_t voff = uint32_t(tid) * 16u, noff = uint32_t(lane) * 4u;
  auto load = [&](int j) CVS_INLINE {
    const int s = j < n_stages ? j : n_stages - 1, buf = j & 1;
#pragma unroll
    for (int i = 0; i < C::LPW; ++i)
      lds_dma<16, false>(rs, lds0 + buf * (C::VECS * 16) + i * (kBThreads * 16), voff + uint32_t(i * kBThreads * 16),
                         s * (C::VECS * 16));
    if (wave < TPS / 2)  // 64 norms each
      lds_dma<4, false>(ns, ldn0 + buf * (TPS * 128) + wave * 256, noff + uint32_t(wave) * 256u, s * (TPS * 128));
  };

  // Query operands, norms, thresholds; a query past the last has threshold
  // -inf (its tile may not exist: the last one is read instead).
  half8 qb[QW][KS];
  float qn[QW], thr[QW];
  uint32_t cnt[QW];
#pragma unroll
  for (int j = 0; j < QW; ++j) {
    const int qt = q0 / 32 + j;
    const u32x4* src = a.qtiles + int64_t(qt < a.n_qtiles ? qt : a.n_qtiles - 1) * (KS * 64) + lane;
#pragma unroll
    for (int s = 0; s < KS; ++s) qb[j][s] = __builtin_bit_cast(half8, src[s * 64]);
    const int q = q0 + 32 * j + (lane & 31);
    const bool ok = q < a.nq;
    qn[j] = ok ? a.qnorms[q] : INFINITY;
    thr[j] = ok ? nextafterf(a.thr0[q], INFINITY) : -INFINITY;
    cnt[j] = 0;
  }
  // List of query q0 + m in this range; a lane's half of its query's list in
  // tile j is at list0(32 j) + moff.
  auto list0 = [&](int m) CVS_INLINE -> uint64_t* { return a.part + (int64_t(q0 + m) * G + x) * CAP; };
  const uint32_t moff = uint32_t(lane & 31) * uint32_t(G) * uint32_t(CAP) + uint32_t(half) * uint32_t(HALF);

  // Compacts the lists of tile j that have a half over `limit` (or, at the
  // end, more than KP keys in all) to their KP smallest keys, which lowers
  // the query's threshold.
  auto compact = [&](int j, uint32_t& c, float& t, uint32_t limit, bool total_only) CVS_INLINE {
    const uint32_t both = c + xor_lanes<32>(c);
    const uint64_t over64 = __ballot(total_only ? both > uint32_t(KP) : c > limit);
    uint32_t over = uint32_t(over64) | uint32_t(over64 >> 32);
    if (over == 0) return;
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
    while (over) {
      const int i = __builtin_ctz(over);
      over &= over - 1;
      const uint32_t c0 = uint32_t(__builtin_amdgcn_readlane(int(c), i));
      const uint32_t c1 = uint32_t(__builtin_amdgcn_readlane(int(c), i + 32));
      const uint32_t kth = compact_query<NS>(list0(32 * j + i), HALF, c0, c1, KP);
      const uint32_t kept = c0 + c1 < uint32_t(KP) ? c0 + c1 : uint32_t(KP);
      if ((lane & 31) == i) {
        c = half == 0 ? (kept < uint32_t(KP / 2) ? kept : uint32_t(KP / 2))
                      : (kept > uint32_t(KP / 2) ? kept - uint32_t(KP / 2) : 0u);
        if (kth != 0xffffffffu) t = fminf(t, unord_f32(kth));
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
  };

  if (n_stages > 0) load(0);
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  for (int j = 0; j < n_stages; ++j) {
    load(j + 1);  // the other buffer was last read a stage ago, before the barrier
    const u32x4* sb = s_stage[j & 1] + lane;
    const float* dn = s_dn[j & 1] + 4 * half;
#pragma unroll 1
    for (int t = 0; t < TPS; ++t) {
      f32x16 acc[QW];
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const half8 av = __builtin_bit_cast(half8, sb[(t * KS + s) * 64]);
        const f32x16 zero = {};
#pragma unroll
        for (int w = 0; w < QW; ++w)
          acc[w] = __builtin_amdgcn_mfma_f32_32x32x16_f16(av, qb[w][s], s == 0 ? zero : acc[w], 0, 0, 0);
      }
      // Rows row0 + 8 (e / 4) + 4 half + e % 4.
      f32x4 dn4[4];
#pragma unroll
      for (int g = 0; g < 4; ++g) dn4[g] = *reinterpret_cast<const f32x4*>(dn + t * 32 + 8 * g);
      const uint32_t rbase = uint32_t((st0 + j) * TPS + t) * 32u + 4u * uint32_t(half);
#pragma unroll
      for (int w = 0; w < QW; ++w) {
        float mg[4];  // of rows 4 g .. 4 g + 3
#pragma unroll
        for (int g = 0; g < 4; ++g) {
#pragma unroll
          for (int e = 4 * g; e < 4 * g + 4; ++e) acc[w][e] = dn4[g][e & 3] - 2.0f * acc[w][e];
          mg[g] = min3(min3(acc[w][4 * g], acc[w][4 * g + 1], acc[w][4 * g + 2]), acc[w][4 * g + 3], INFINITY);
        }
        if (__ballot(qn[w] + min3(min3(mg[0], mg[1], mg[2]), mg[3], INFINITY) < thr[w]) == 0) continue;
        // Room for a block's 16 rows (a lane appends at most one key a row).
        if (__ballot(cnt[w] > uint32_t(HALF - 16)) != 0) compact(w, cnt[w], thr[w], uint32_t(HALF - 16), false);
        uint64_t* const mine = list0(32 * w) + moff;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          if (__ballot(qn[w] + mg[g] < thr[w]) == 0) continue;
#pragma unroll
          for (int e = 4 * g; e < 4 * g + 4; ++e) {
            const float d = qn[w] + acc[w][e];
            if (d < thr[w]) {
              mine[cnt[w]] = (uint64_t(ord_f32(d)) << 32) | (rbase + uint32_t(8 * g + (e & 3)));
              ++cnt[w];
            }
          }
        }
      }
    }
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
  }

  // The lists in place (first KP entries: half 0's keys, half 1's, then
  // sentinels), their minima and final thresholds.
#pragma unroll
  for (int w = 0; w < QW; ++w) compact(w, cnt[w], thr[w], 0u, true);
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
  constexpr int NE = (KP + 63) / 64;
#pragma unroll
  for (int w = 0; w < QW; ++w) {
#pragma unroll 4
    for (int i = 0; i < 32; ++i) {
      const int q = q0 + 32 * w + i;
      if (q >= a.nq) break;
      const uint32_t c0 = uint32_t(__builtin_amdgcn_readlane(int(cnt[w]), i));
      const uint32_t c1 = uint32_t(__builtin_amdgcn_readlane(int(cnt[w]), i + 32));
      uint64_t* const lst = list0(32 * w + i);
      uint64_t key[NE];
      uint64_t mn = kSentinel;
#pragma unroll
      for (int t = 0; t < NE; ++t) {
        const uint32_t e = uint32_t(lane + 64 * t);
        key[t] = e < c0 ? lst[e] : (e < c0 + c1 ? lst[HALF + (e - c0)] : kSentinel);
        mn = key[t] < mn ? key[t] : mn;
      }
      __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");  // every entry is read before any is written
#pragma unroll
      for (int t = 0; t < NE; ++t)
        if (lane + 64 * t < KP) lst[lane + 64 * t] = key[t];
#pragma unroll
      for (int o = 32; o >= 1; o >>= 1) {
        const uint64_t y = shfl_xor_u64(mn, o);
        mn = y < mn ? y : mn;
      }
      const float cut = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(thr[w]), i));
      if (lane == 0) {
        a.lmin[int64_t(q) * G + x] = mn;
        a.lcut[int64_t(q) * G + x] = cut;
      }
    }
  }
}

template <int KS>
void launch_ks(cvs_context* ctx, const BatchArgs& a, int kp, hipEvent_t e0, hipEvent_t e1) {
  const dim3 grid(unsigned(a.n_ranges) * unsigned(a.n_qblocks));
  auto go = [&](auto kernel) { hipExtLaunchKernelGGL(kernel, grid, dim3(BatchCfg<KS>::T), 0, ctx->stream, e0, e1, 0, a); };
  switch (kp) {
    case 16: go(bf_batch_scan_kernel<KS, 16>); break;
    case 32: go(bf_batch_scan_kernel<KS, 32>); break;
    case 64: go(bf_batch_scan_kernel<KS, 64>); break;
    case 128: go(bf_batch_scan_kernel<KS, 128>); break;
    default: fail(CVS_ERR_RUNTIME, "unsupported candidate count");
  }
}

// Fewest ranges of the dataset for lists of kp keys.  A list's final threshold
// is its kp-th key, and the smallest of them has to lie beyond the merge's
// R = 2 kp candidates: with one or two ranges it is the kp-th or so key of the
// whole dataset, and the queries that kp candidates do not certify are
// re-ranked over every row (131,072 queries, K = 10, 20,000 x 256 in tight
// clusters: a third of them).  These counts put kp of the 2 kp nearest rows
// into one range with a probability below 3e-6 (binomial; rows in an order that
// does not sort them by place).
int min_ranges(int kp) { return kp <= 16 ? 8 : (kp <= 32 ? 5 : (kp <= 64 ? 4 : 3)); }

// Whether this scan is the faster one (the other: the streaming scan, or for kp
// = 128 the register-blocked one, slower at all but one of 156 sizes).  Its
// workgroups finish 64 lists a wave however few rows they have seen, which
// small calls do not make up for.  Streaming scan against this one, K = 10, d =
// 96 / 256 / 320 (us, whole calls): 20,000 rows, 2,000 queries 135 / 164 / 190
// against 145 / 179 / 212, 4,000 queries 236 / 297 / 337 against 221 / 285 /
// 336; 40,000 rows, 1,100 queries 149 / 193 / 194 against 139 / 172 / 185.  The
// line lies lower for K = 24 (10,000 rows, 3,000 queries, d = 96 / 256: 214 /
// 227 against 192 / 219), and for K = 48 only calls whose rows fill most of one
// unit of 2,048 lie below it (2,000 rows, 1,100 queries: 1.05 to 1.2x slower
// here; 1,500 rows, up to 16 k-steps: 1.3 to 2.5x faster).
bool pays(int ks, int kp, int64_t q, int64_t n) {
  if (kp > 64) return true;
  if (kp == 64) return q >= 3000 || n > 2048 || (n <= 1700 && ks < 20);
  const double t = kp <= 16 ? 5500.0 : 3500.0;
  return n >= 4000 ? double(q) >= t * (1.0 - double(n) / 48000.0) : n >= 2000 && double(q) >= 1.5 * t;
}

}  // namespace

BatchPlan plan_batch_scan(int ks, int kp, int64_t q, int64_t n, int64_t n_tiles, int compute_units) {
  BatchPlan p;
  if (ks != 8 && ks != 12 && ks != 16 && ks != 20) return p;
  if (!pays(ks, kp, q, n)) return p;
  const int64_t qb = ks <= 8 ? BatchCfg<8>::QB : BatchCfg<12>::QB;
  const int64_t stages = n_tiles / (ks <= 8 ? BatchCfg<8>::TPS : BatchCfg<12>::TPS);
  const int64_t blocks = (q + qb - 1) / qb;
  if (blocks > (int64_t(1) << 20)) return p;
  // Ranges: the fewest (each list costs its workgroup a finish and the merge a
  // read) that leave at most 1/16 of the last round of workgroups' slots idle
  // (three per compute unit at 8 k-steps, one beyond), or else the best count;
  // no fewer than the certificate needs (min_ranges).
  const int64_t cu = std::max(1, compute_units) * (ks <= 8 ? 3 : 1);
  const int64_t most = std::min<int64_t>(kBatchMaxRanges, stages);
  double best = 0;
  for (int64_t g = std::min<int64_t>(min_ranges(kp), most); g <= most; ++g) {
    const int64_t w = g * blocks, rounds = (w + cu - 1) / cu;
    const double eff = double(w) / double(rounds * cu);
    if (eff > best + 1e-9) {
      best = eff;
      p.n_ranges = int(g);
    }
    if (eff >= 0.9375) break;
  }
  p.n_qblocks = int(blocks);
  // A range's tiles within one buffer resource (2 GiB).
  p.ok = p.n_ranges > 0 && (n_tiles / p.n_ranges + 64) * ks * int64_t(kStepBytes) < (int64_t(1) << 31);
  return p;
}

void launch_batch_scan(cvs_context* ctx, const BatchArgs& a, int ks, int kp, hipEvent_t e0, hipEvent_t e1) {
  switch (ks) {
    case 8: launch_ks<8>(ctx, a, kp, e0, e1); break;
    case 12: launch_ks<12>(ctx, a, kp, e0, e1); break;
    case 16: launch_ks<16>(ctx, a, kp, e0, e1); break;
    case 20: launch_ks<20>(ctx, a, kp, e0, e1); break;
    default: fail(CVS_ERR_RUNTIME, "unsupported padded dimension");
  }
  after_launch("bf_batch_scan_kernel");
}

}  // namespace bf
}  // namespace cvs
