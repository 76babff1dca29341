// CAGRA graph search for gfx950: one workgroup of 1-8 waves per query.
//
// Replaces the reference's `cagra_beam_search` kernel
// (shaders/cagra_kernels.metal:28-199, host src/metal_context.mm:918-1111)
// and its host-side entry-point selection (src/cagra.cpp:128-178).  The
// reference keeps an unsorted beam in device memory that thread 0 scans
// serially per neighbour, and a Q x N visited bitfield.  Here everything a
// query touches between iterations stays on chip:
//
//  - itopk list: sorted ascending 64-bit keys in registers, E = itopk/64 per
//    lane (position i = 64*slot + lane).  A key is
//        ord(distance) << 32 | id << 1 | expanded
//    so the order is (distance, id) and marking an entry expanded never
//    reorders the list.
//  - visited set: a bitmap of n bits in LDS when that is no larger than the
//    hash below (n <= 131,072 or 262,144); else an open-addressing hash of
//    2^hash_bits ids, filled to at most one half.  When the next iteration
//    could overflow the hash, it is cleared and the ids of the itopk list
//    re-inserted: an id that left the list can be evaluated again, but can
//    never re-enter it (its key is above the list's current worst), so the
//    list never holds duplicates and does not depend on which set is used.
//  - candidates: processed 64 at a time (one id per lane of the lead wave).
//    New ids pass the hash, are compacted into LDS, and their distances are
//    computed by the 16-lane teams of all waves (each lane reads 16 bytes at
//    a stride of 256 bytes, so a row is gathered in coalesced 256-byte
//    segments and one load instruction serves four rows).  The 64 keys are
//    sorted with a wave bitonic sort and merged into the itopk list with a
//    bitonic merge; candidates that cannot enter the list are dropped
//    before the sort.
//  - waves per query: 2 for large batches; 4 or 8 when the batch is small
//    and each query's chain of dependent gathers is the latency (Q = 1).
//    With long lists or wide searches (ahead_from) those small batches run
//    cagra_ahead_kernel, which shortens that chain: the rows of several
//    parents gathered in one step.
//
// Iteration: pick the first `width` unexpanded entries of the list as
// parents, mark them, evaluate their neighbours.  Stop when the list holds no
// unexpanded entry or after max_iterations.  The list is seeded with the
// index's seed nodes (the reference's navigation nodes, src/cagra.cpp:63-82:
// the reference starts from the single nearest one; here all of them enter
// the list, which contains that one); the free lanes of the last 64-id seed
// chunk (all 64 without seed nodes) take hashed ids led by the reference's
// fallback (q * 2654435761) mod n (shaders/cagra_kernels.metal:65-67).
//
// Distances are exact fp32 sums of squared differences (summation order of
// four 16-lane partial sums); outputs are sorted by (distance, id) and padded
// with UINT32_MAX / +inf (src/cagra.cpp:240-251).
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "cvs_internal.hpp"
#include "device_util.hpp"

namespace cvs {
namespace {

constexpr uint32_t kInvalidId = 0xffffffffu;
constexpr uint64_t kEmptyKey = ~0ull;
// Rows of up to kBigDim columns keep the query slice in registers; wider
// rows (up to CVS_CAGRA_MAX_DIM) keep it in LDS and are gathered in chunks
// of kBigDim columns.
constexpr int kBigDim = 1024;
constexpr int kMaxDv = kBigDim / 64;   // float4 per lane and row (fp32 traversal)
constexpr int kMaxDv8 = kBigDim / 128; // 8-column pieces per lane and row (fp16 traversal)

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));

struct SearchArgs {
  const float4* rows;     // n rows of dq float4, zero-padded
  const uint4* rows16;    // n rows of dq8 x 8 fp16 of scale * (row - mu) (traversal copy), zero-padded
  const float* mu;        // dpad column means subtracted in the traversal copy (zero-padded)
  float scale;            // power of two applied after centring
  const uint32_t* graph;  // n x g
  const uint32_t* seeds;  // n_seeds seed ids, or null
  const float* queries;   // q x d fp32
  uint32_t* out_nbr;      // q x k
  float* out_dist;        // q x k
  uint32_t* stats;        // q x 2: distance evaluations, iterations (or null)
  int64_t d;
  uint32_t n;
  int g;
  int dq;  // float4 per padded row (16 * dv)
  int dq8; // 8-column pieces per padded row (16 * dv8)
  int dv8; // 8-column pieces per lane and row
  int dv;  // float4 per lane and row
  int n_seeds;
  int seed_lanes;  // seed candidates in all: n_seeds, then hashed ids
  int k;
  int itopk;
  int width;
  int max_iter;
  int hash_bits;
  int bitmap_words;     // > 0: the visited set is a bitmap of this many words (n bits, rounded up)
  int teams;            // workgroups per query (block b = query b / teams, team b % teams)
  uint64_t* team_keys;  // teams > 1: (q * teams) x itopk list keys, merged afterwards
  uint32_t* record;     // or null: the ids of each query's distance evaluations, in order,
  int record_cap;       // the first record_cap of them per query (q x record_cap)
};

// Merges 64 sorted keys `c` (one per lane) into the sorted list `top` of
// 64*E keys, keeping the 64*E smallest.  min(top[i], c'[N-1-i]) with c'
// = c padded by empty keys is bitonic; half-cleaners then sort it.
template <int E>
__device__ __forceinline__ void merge_into(uint64_t (&top)[E], uint64_t c) {
  const int lane = __lane_id();
  const uint64_t cr = shfl_xor_u64(c, 63);  // lane 63 - lane
  top[E - 1] = top[E - 1] < cr ? top[E - 1] : cr;
#pragma unroll
  for (int s = E / 2; s >= 1; s >>= 1) {
#pragma unroll
    for (int e = 0; e < E; ++e) {
      if ((e & s) == 0) {
        const uint64_t lo = top[e] < top[e + s] ? top[e] : top[e + s];
        const uint64_t hi = top[e] < top[e + s] ? top[e + s] : top[e];
        top[e] = lo;
        top[e + s] = hi;
      }
    }
  }
#pragma unroll
  for (int stride = 32; stride >= 1; stride >>= 1) {
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const uint64_t y = shfl_xor_u64(top[e], stride);
      const bool lower = (lane & stride) == 0;
      top[e] = lower ? (top[e] < y ? top[e] : y) : (top[e] < y ? y : top[e]);
    }
  }
}

// The list's last kept key (position itopk - 1; the empty key while the list
// is not full).
template <int E>
__device__ __forceinline__ uint64_t last_key(const uint64_t (&top)[E], int itopk) {
  const int wpos = itopk - 1;
  uint64_t worst = kEmptyKey;
#pragma unroll
  for (int e = 0; e < E; ++e) {
    if (e == (wpos >> 6)) {  // uniform: one slot is read
      const uint32_t wlo = uint32_t(__builtin_amdgcn_readlane(int(uint32_t(top[e])), wpos & 63));
      const uint32_t whi = uint32_t(__builtin_amdgcn_readlane(int(uint32_t(top[e] >> 32)), wpos & 63));
      worst = (uint64_t(whi) << 32) | wlo;
    }
  }
  return worst;
}

// Inserts one key (uniform over the wave, not in the list) into the sorted
// list: entries above it move up by one position, the last one falls out.
// About 10 instructions per slot, where sorting a few candidates and merging
// them takes over 100 plus 60 per slot.
template <int E>
__device__ __forceinline__ void insert_key(uint64_t (&top)[E], uint64_t key) {
  constexpr int kWaveShr1 = 0x138;  // DPP: lane l takes lane l - 1, lane 0 keeps `old`
#pragma unroll
  for (int e = E - 1; e >= 0; --e) {
    const int lo = int(uint32_t(top[e])), hi = int(uint32_t(top[e] >> 32));
    int olo = 0, ohi = 0;
    if (e > 0) {
      olo = __builtin_amdgcn_readlane(int(uint32_t(top[e - 1])), 63);
      ohi = __builtin_amdgcn_readlane(int(uint32_t(top[e - 1] >> 32)), 63);
    }
    const uint32_t plo = uint32_t(__builtin_amdgcn_update_dpp(olo, lo, kWaveShr1, 0xF, 0xF, false));
    const uint32_t phi = uint32_t(__builtin_amdgcn_update_dpp(ohi, hi, kWaveShr1, 0xF, 0xF, false));
    const uint64_t prev = (uint64_t(phi) << 32) | plo;  // 0 before the first entry: below every key
    top[e] = top[e] < key ? top[e] : (prev < key ? key : prev);
  }
}

// Candidate keys (one per lane, the empty key for none) into the list.  A
// key at or above the list's last one cannot enter it (keys are unique; an
// unfilled list holds the empty key there), so such candidates are dropped
// first; a few are inserted one by one, more are compacted (through
// `scratch`, 32 keys of LDS that only this wave uses here), sorted and
// merged.  The list is the same either way.
constexpr int kInsertMax = 6;
template <int E>
__device__ __forceinline__ void add_keys(uint64_t (&top)[E], uint64_t key, int itopk, uint64_t* scratch) {
  const int lane = __lane_id();
  const uint64_t worst = last_key<E>(top, itopk);
  uint64_t m = __ballot(key < worst);
  if (m == 0) return;
  if (popc(m) <= kInsertMax) {
    do {
      const int b = __builtin_ctzll(m);
      m &= m - 1;
      const uint32_t lo = uint32_t(__builtin_amdgcn_readlane(int(uint32_t(key)), b));
      const uint32_t hi = uint32_t(__builtin_amdgcn_readlane(int(uint32_t(key >> 32)), b));
      insert_key<E>(top, (uint64_t(hi) << 32) | lo);
    } while (m != 0);
  } else {
    (void)sort_below(key, worst, kEmptyKey, scratch);
    merge_into<E>(top, key);
  }
#pragma unroll
  for (int e = 0; e < E; ++e)
    if (e * 64 + lane >= itopk) top[e] = kEmptyKey;
}

// A lane's slice of the query and its pieces of a row (d <= 1024).  fp32
// traversal: float4 columns tp + 16 j of the padded row.  fp16 traversal (and
// its fp32 re-rank): 8-column pieces tp + 16 j, so that a 16-lane team reads
// 256 contiguous bytes of an fp16 row (512 of an fp32 row) per piece.  The
// fp16 traversal keeps its slice of the centred, scaled query in fp16, as the
// rows are: a piece's distance is four packed differences and four
// fp32-accumulating dot2s, and the slice takes 32 VGPRs instead of 64.  The
// traversal's distances only steer the search; the list is re-ranked against
// the fp32 query and rows at the end.  The query comes from LDS, where
// stage_query put it with coalesced loads of any alignment (column clamped,
// the value masked by an AND of its bits, so that no load sits under a
// condition and all are in flight together): a lane's own loads of its 64
// scattered columns took 8 us of a single query's search.
__device__ __forceinline__ float masked(float x, bool in) {
  return __uint_as_float(__float_as_uint(x) & (in ? 0xffffffffu : 0u));
}

// Sum of the squares of four differences, in one rounding order wherever it
// is inlined, so that every kernel gives a row the same distance.
__device__ __forceinline__ float sum_sq4(float x, float y, float z, float w) {
  return __builtin_fmaf(x, x, __fmul_rn(y, y)) + __builtin_fmaf(z, z, __fmul_rn(w, w));
}

template <bool F16>
struct Slice;

template <>
struct Slice<false> {
  using Piece = float4;
  static constexpr int N = kMaxDv;
  float4 q[N];
  __device__ __forceinline__ void load(const float* s_q, int tp) {
#pragma unroll
    for (int j = 0; j < N; ++j) q[j] = reinterpret_cast<const float4*>(s_q)[tp + 16 * j];
  }
  __device__ __forceinline__ void fetch(const SearchArgs& a, uint32_t rid, int tp, float4 (&x)[N]) const {
    const float4* row = a.rows + int64_t(rid) * a.dq + tp;
#pragma unroll
    for (int j = 0; j < N; ++j)
      if (j < a.dv) x[j] = row[16 * j];
  }
  // This lane's part of the squared distance.
  __device__ __forceinline__ float part(const SearchArgs& a, const float4 (&x)[N]) const {
    float acc = 0.f;
#pragma unroll
    for (int j = 0; j < N; ++j) {
      if (j < a.dv) {
        acc = __fadd_rn(acc, sum_sq4(q[j].x - x[j].x, q[j].y - x[j].y, q[j].z - x[j].z, q[j].w - x[j].w));
      }
    }
    return acc;
  }
};

template <>
struct Slice<true> {
  using Piece = uint4;
  static constexpr int N = kMaxDv8;
  half8_t q[N];
  // From the centred, scaled query, rounded to fp16.
  __device__ __forceinline__ void load(const float* s_q, int tp) {
#pragma unroll
    for (int j = 0; j < N; ++j) {
      const float4* v = reinterpret_cast<const float4*>(s_q + (tp + 16 * j) * 8);
      const float4 x = v[0], y = v[1];
      q[j] = half8_t{_Float16(x.x), _Float16(x.y), _Float16(x.z), _Float16(x.w),
                     _Float16(y.x), _Float16(y.y), _Float16(y.z), _Float16(y.w)};
    }
  }
  __device__ __forceinline__ void fetch(const SearchArgs& a, uint32_t rid, int tp, uint4 (&x)[N]) const {
    const uint4* row = a.rows16 + int64_t(rid) * a.dq8 + tp;
#pragma unroll
    for (int j = 0; j < N; ++j)
      if (j < a.dv8) x[j] = row[16 * j];
  }
  __device__ __forceinline__ float part(const SearchArgs& a, const uint4 (&x)[N]) const {
    float acc = 0.f;
#pragma unroll
    for (int j = 0; j < N; ++j) {
      if (j < a.dv8) {
        const uint4 qw = __builtin_bit_cast(uint4, q[j]);
        const uint32_t qa[4] = {qw.x, qw.y, qw.z, qw.w}, xa[4] = {x[j].x, x[j].y, x[j].z, x[j].w};
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const half2_t d2 = __builtin_bit_cast(half2_t, qa[t]) - __builtin_bit_cast(half2_t, xa[t]);
          acc = __builtin_amdgcn_fdot2(d2, d2, acc, false);
        }
      }
    }
    return acc;
  }
};

// Sum over the 16 lanes of a team.
__device__ __forceinline__ float team_sum(float acc) {
  acc += xor_lanes_f(acc, 8);
  acc += xor_lanes_f(acc, 4);
  acc += xor_lanes_f(acc, 2);
  acc += xor_lanes_f(acc, 1);
  return acc;
}

// Exact part of the squared distance for the re-rank after fp16 traversal
// (d <= 1024): the fp32 row against the query as given, staged in LDS (zero
// past d as the rows are).
__device__ __forceinline__ float exact_part(const SearchArgs& a, const float* s_q, uint32_t rid, int tp) {
  const float4* row = a.rows + int64_t(rid) * a.dq + 2 * tp;
  const float4* qq = reinterpret_cast<const float4*>(s_q) + 2 * tp;
  float acc = 0.f;
  float4 x[2 * kMaxDv8];
#pragma unroll
  for (int j = 0; j < kMaxDv8; ++j) {
    if (j < a.dv8) {
      x[2 * j] = row[32 * j];
      x[2 * j + 1] = row[32 * j + 1];
    }
  }
#pragma unroll
  for (int j = 0; j < kMaxDv8; ++j) {
    if (j < a.dv8) {
      const float4 ql = qq[32 * j], qh4 = qq[32 * j + 1];
      const float4 lo = x[2 * j], hi = x[2 * j + 1];
      acc = __fadd_rn(acc, sum_sq4(ql.x - lo.x, ql.y - lo.y, ql.z - lo.z, ql.w - lo.w) +
                               sum_sq4(qh4.x - hi.x, qh4.y - hi.y, qh4.z - hi.z, qh4.w - hi.w));
    }
  }
  return acc;
}

// Writes a query's results (lead wave): the team's list for the merge of
// teams, else the k nearest and the counts.
template <int E>
__device__ __forceinline__ void write_list(const SearchArgs& a, const uint64_t (&top)[E], int64_t qi, uint32_t evals,
                                           int it) {
  const int lane = __lane_id();
  if (a.team_keys) {
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const int pos = e * 64 + lane;
      if (pos < a.itopk) a.team_keys[int64_t(blockIdx.x) * a.itopk + pos] = top[e];
    }
    return;
  }
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int pos = e * 64 + lane;
    if (pos < a.k) {
      const uint64_t key = top[e];
      a.out_nbr[qi * a.k + pos] = key == kEmptyKey ? kInvalidId : uint32_t(key) >> 1;
      a.out_dist[qi * a.k + pos] = key == kEmptyKey ? INFINITY : unord_f32(uint32_t(key >> 32));
    }
  }
  if (a.stats && lane == 0) {
    a.stats[2 * qi] = evals;
    a.stats[2 * qi + 1] = uint32_t(it);
  }
}

// fp16 traversal: the list's distances are recomputed exactly from the fp32
// rows (all W waves, 64 entries per round; `exact(id)` sums a row over the
// calling team) and the list re-sorted, so the output is the exact top-k of
// the visited rows in the list.
template <int E, int W, typename Exact>
__device__ __forceinline__ void rerank_list(uint64_t (&top)[E], bool lead, uint32_t* s_ids, float* s_dist,
                                            Exact exact) {
  const int lane = threadIdx.x & 63, team = threadIdx.x >> 4, tp = threadIdx.x & 15;
#pragma unroll
  for (int e = 0; e < E; ++e) {
    if (lead) s_ids[lane] = top[e] != kEmptyKey ? uint32_t(top[e]) >> 1 : 0u;
    __syncthreads();
    for (int r0 = 0; r0 < 64; r0 += 4 * W) {
      const float acc = exact(s_ids[r0 + team]);
      if (tp == 0) s_dist[r0 + team] = acc;
    }
    __syncthreads();
    if (lead && top[e] != kEmptyKey) top[e] = (uint64_t(ord_f32(s_dist[lane])) << 32) | (uint64_t(s_ids[lane]) << 1);
  }
  if (lead) wave_sort_e<E>(top);
}

// The query into LDS, kBigDim floats, zero past d: as given into s_q, and for
// fp16 traversal centred and scaled as the traversal copy is (its distances
// are scale^2 times the squared distance) into s_c.
template <bool F16>
__device__ __forceinline__ void stage_query(const SearchArgs& a, const float* qsrc, float* s_q, float* s_c,
                                            int threads) {
  for (int i = threadIdx.x; i < kBigDim; i += threads) {
    const int c = i < a.d ? i : int(a.d - 1);
    const float x = qsrc[c];
    s_q[i] = masked(x, i < a.d);
    if constexpr (F16) s_c[i] = masked((x - a.mu[c]) * a.scale, i < a.d);
  }
}

// One workgroup of W waves per query.  Wave 0 (the lead wave) owns the
// itopk list, the hash inserts, the sort and the merge; all 4W 16-lane teams
// gather candidate rows, so a chunk of 64 candidates costs ceil(64 / 4W)
// dependent gather rounds instead of 16.  The kernel also runs with W = 1 (no
// barriers between waves are needed then); the host launches W = 2 for large
// batches, where the other wave's gathers hide the lead wave's serial work,
// and W = 4 or 8 when few queries would leave most of the GPU idle.
// The large-batch fp16 instance (W = 2) runs four waves per SIMD (113 VGPRs):
// two queries per SIMD in flight instead of one and a half hide more of the
// lead wave's serial work.
template <int E, int W, bool F16, bool BIG>
__global__ __launch_bounds__(64 * W, (F16 && W == 2 && !BIG) ? 4 : 1) void cagra_search_kernel(SearchArgs a) {
  extern __shared__ uint32_t s_mem[];
  const bool bitmap = a.bitmap_words > 0;
  const int H = bitmap ? a.bitmap_words : 1 << a.hash_bits;  // visited-set words
  const uint32_t hmask = uint32_t(H) - 1u;
  const int hcap = bitmap ? (1 << 30) : H / 2;  // a bitmap is never cleared
  const uint32_t hempty = bitmap ? 0u : kInvalidId;
  uint32_t* s_hash = s_mem;
  uint32_t* s_ids = s_mem + (BIG || H > kBigDim ? H : kBigDim);  // 64 fresh ids
  float* s_dist = reinterpret_cast<float*>(s_ids + 64);  // their distances
  uint32_t* s_par = s_ids + 128;                         // parents of this iteration
  // Control words written by the lead wave and read by all after a barrier:
  // [0, 1] fresh-id count (alternating per chunk), [2] hash fill after a
  // reset, [3, 4] parent count (alternating per iteration).  Alternating slots
  // keep a write for the next step from racing a slow wave's read.
  uint32_t* s_ctl = s_par + CVS_CAGRA_MAX_WIDTH;
  // d > 1024 (BIG): the query stays in LDS, as given (s_q) and, for fp16
  // traversal, centred and scaled (s_qc); dpad floats each, after the
  // control words.  fp16 traversal with d <= 1024: s_q receives the query as
  // given (kBigDim floats, zero past d) for the final exact re-rank.
  float* s_q = reinterpret_cast<float*>(s_ctl + 8);
  float* s_qc = s_q + (BIG ? a.dq * 4 : 0);

  constexpr int kThreads = 64 * W;
  constexpr int kTeams = 4 * W;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const bool lead = W == 1 || __builtin_amdgcn_readfirstlane(tid >> 6) == 0;
  const int64_t qi = blockIdx.x / a.teams;
  const int tm = int(blockIdx.x - qi * a.teams);
  const int team = tid >> 4, tp = lane & 15;

  const float* qsrc = a.queries + qi * a.d;
  Slice<F16> slice;  // d <= 1024
  if constexpr (!BIG) {
    // Staged where the visited set will be (at least kBigDim words); fp16
    // traversal keeps the query as given in s_q for the final re-rank.
    float* const staged = reinterpret_cast<float*>(s_mem);
    stage_query<F16>(a, qsrc, F16 ? s_q : staged, staged, kThreads);
    __syncthreads();
    slice.load(staged, tp);
    __syncthreads();
  }
  for (int i = tid; i < H; i += kThreads) s_hash[i] = hempty;
  if constexpr (BIG) {
    const float* qg = a.queries + qi * a.d;
    for (int i = tid; i < 4 * a.dq; i += kThreads) {
      const float v = i < a.d ? qg[i] : 0.f;
      s_q[i] = v;
      if (F16) s_qc[i] = i < a.d ? (v - a.mu[i]) * a.scale : 0.f;
    }
  }

  // Squared distance of row rid to the query, summed over the 16 lanes of
  // this lane's team: from the traversal copy, or (exact) from the fp32 rows.
  auto team_dist = [&](uint32_t rid, bool exact) -> float {
    float acc = 0.f;
    if constexpr (BIG) {
      // Chunks of 1,024 columns: the row's pieces tp + 16 j of the chunk,
      // all loads of a chunk issued before the first is used; the query from
      // LDS.
      if (!F16 || exact) {
        // fp32 rows: float4 columns (F16: 8-column pieces as two float4).
        const float4* row = a.rows + int64_t(rid) * a.dq;
        const float4* qq = reinterpret_cast<const float4*>(s_q);
        for (int c0 = 0; c0 < a.dq; c0 += 256) {
          const int nj = (a.dq - c0) / 16 < 16 ? (a.dq - c0) / 16 : 16;
          float4 x[16];
#pragma unroll
          for (int j = 0; j < 16; ++j)
            if (j < nj) x[j] = row[c0 + tp + 16 * j];
#pragma unroll
          for (int j = 0; j < 16; ++j) {
            if (j < nj) {
              const float4 qj = qq[c0 + tp + 16 * j];
              const float dx = qj.x - x[j].x, dy = qj.y - x[j].y;
              const float dz = qj.z - x[j].z, dw = qj.w - x[j].w;
              acc += (dx * dx + dy * dy) + (dz * dz + dw * dw);
            }
          }
        }
      } else {
        // fp16 traversal copy: 8-column pieces against the centred query.
        const uint4* row = a.rows16 + int64_t(rid) * a.dq8;
        for (int c0 = 0; c0 < a.dq8; c0 += 128) {
          const int nj = (a.dq8 - c0) / 16 < 8 ? (a.dq8 - c0) / 16 : 8;
          uint4 x[8];
#pragma unroll
          for (int j = 0; j < 8; ++j)
            if (j < nj) x[j] = row[c0 + tp + 16 * j];
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            if (j < nj) {
              const half8_t h = __builtin_bit_cast(half8_t, x[j]);
              const float* qc = s_qc + 8 * (c0 + tp + 16 * j);
              float p[8];
#pragma unroll
              for (int t = 0; t < 8; ++t) {
                const float dt = qc[t] - float(h[t]);
                p[t] = dt * dt;
              }
              acc += ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
            }
          }
        }
      }
    } else if (F16 && exact) {
      acc = exact_part(a, s_q, rid, tp);
    } else {
      typename Slice<F16>::Piece x[Slice<F16>::N];
      slice.fetch(a, rid, tp, x);
      acc = slice.part(a, x);
    }
    return team_sum(acc);
  };

  uint64_t top[E];  // the list (lead wave)
#pragma unroll
  for (int e = 0; e < E; ++e) top[e] = kEmptyKey;
  int count = 0;       // ids in the hash table (workgroup-uniform)
  uint32_t evals = 0;  // distance evaluations (lead wave)
  int phase = 0;       // alternates the fresh-count slot
  __syncthreads();

  // Marks id (< n) visited; true if it was not.
  auto hash_insert = [&](uint32_t id) -> bool {
    if (bitmap) {
      const uint32_t bit = 1u << (id & 31u);
      return (atomicOr(&s_hash[id >> 5], bit) & bit) == 0u;
    }
    uint32_t h = (id * 0x9E3779B1u) >> (32 - a.hash_bits);
    for (;;) {
      const uint32_t old = atomicCAS(&s_hash[h], kInvalidId, id);
      if (old == kInvalidId) return true;
      if (old == id) return false;
      h = (h + 1u) & hmask;
    }
  };

  auto reset_hash = [&]() {
    __syncthreads();
    for (int i = tid; i < H; i += kThreads) s_hash[i] = hempty;
    __syncthreads();
    if (lead) {
      int c = 0;
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const bool v = top[e] != kEmptyKey;
        if (v) hash_insert(uint32_t(top[e]) >> 1);
        c += popc(__ballot(v));
      }
      if (lane == 0) s_ctl[2] = uint32_t(c);
    }
    __syncthreads();
    count = int(s_ctl[2]);
  };

  // Evaluates the candidate ids held one per lane of the lead wave
  // (kInvalidId for none) and merges the new ones into the list.
  auto process = [&](uint32_t id) {
    uint32_t* const s_nf = s_ctl + phase;
    phase ^= 1;
    if (lead) {
      const bool fresh = id < a.n && hash_insert(id);
      const uint64_t m = __ballot(fresh);
      if (fresh) s_ids[mbcnt(m)] = id;
      if (lane == 0) *s_nf = uint32_t(popc(m));
      if (a.record && fresh) {
        const uint32_t pos = evals + uint32_t(mbcnt(m));
        if (pos < uint32_t(a.record_cap)) a.record[qi * a.record_cap + pos] = id;
      }
    }
    __syncthreads();
    const int nf = int(*s_nf);
    if (nf == 0) return;
    count += nf;
    evals += uint32_t(nf);
    for (int r0 = 0; r0 < nf; r0 += kTeams) {
      const int r = r0 + team;
      const bool ok = r < nf;
      const float acc = team_dist(s_ids[ok ? r : 0], false);
      if (ok && tp == 0) s_dist[r] = acc;
    }
    __syncthreads();
    if (lead) {
      uint64_t key =
          lane < nf ? (uint64_t(ord_f32(s_dist[lane])) << 32) | (uint64_t(s_ids[lane]) << 1) : kEmptyKey;
      // (The id/distance slots are the scratch: every wave has finished
      // reading them.)
      add_keys<E>(top, key, a.itopk, reinterpret_cast<uint64_t*>(s_ids));
    }
    // With one wave, program order alone separates this chunk's LDS reads
    // from the next chunk's writes; with more, the lead wave writes the next
    // chunk's ids only after every wave has passed the barrier above.
    if (W == 1) __syncthreads();
  };

  // Seeds: seed_lanes candidates in chunks of 64, first the seed nodes, then
  // hashed ids led by the reference's fallback (q * 2654435761) mod n, so that
  // regions no seed node reaches (clusters the graph does not link) can still
  // be entered.  With several teams per query, team t takes the candidates
  // t, t + teams, t + 2 teams, ... of that sequence (the reference's teams
  // start from entry points rotated by n / teams,
  // shaders/cagra_kernels.metal:243-250).
  {
    const uint32_t h0 = uint32_t(qi) * 2654435761u;
    for (int c = 0; c < a.seed_lanes; c += 64) {
      if (count + 64 > hcap) reset_hash();
      const int i = (c + lane) * a.teams + tm;
      uint32_t id = kInvalidId;
      if (lead) {
        if (i < a.n_seeds)
          id = a.seeds[i];
        else if (uint32_t(i - a.n_seeds) < a.n)
          id = (h0 + uint32_t(i - a.n_seeds) * 0x9E3779B9u) % a.n;
      }
      process(id);
    }
  }

  // Iterations.
  int it = 0;
  for (; it < a.max_iter; ++it) {
    if (count + a.width * a.g > hcap) reset_hash();
    uint32_t* const s_np = s_ctl + 3 + (it & 1);
    if (lead) {
      int np = 0;
#pragma unroll
      for (int e = 0; e < E; ++e) {
        uint64_t m = __ballot(top[e] != kEmptyKey && (top[e] & 1ull) == 0);
        while (m != 0 && np < a.width) {
          const int b = __builtin_ctzll(m);
          m &= m - 1;
          if (lane == b) {
            s_par[np] = uint32_t(top[e]) >> 1;
            top[e] |= 1ull;
          }
          ++np;
        }
      }
      if (lane == 0) *s_np = uint32_t(np);
    }
    __syncthreads();
    const int np = int(*s_np);
    if (np == 0) break;
    const int total = np * a.g;
    for (int c = 0; c < total; c += 64) {
      const int f = c + lane;
      uint32_t id = kInvalidId;
      if (lead && f < total) {
        const int p = f / a.g;
        const int j = f - p * a.g;
        id = a.graph[int64_t(s_par[p]) * a.g + j];
      }
      process(id);
    }
  }

  if constexpr (F16) {
    rerank_list<E, W>(top, lead, s_ids, s_dist, [&](uint32_t rid) { return team_dist(rid, true); });
  }
  if (lead) write_list<E>(a, top, qi, evals, it);
}

// Smallest value of the wave, in every lane: v_min_u32 with DPP row shifts
// and row broadcasts (lanes without a source take the identity).
__device__ __forceinline__ uint32_t wave_min_u32(uint32_t x) {
  auto step = [&](auto ctrl, auto rows) {
    constexpr int kCtrl = decltype(ctrl)::value, kRows = decltype(rows)::value;
    const uint32_t y = uint32_t(__builtin_amdgcn_update_dpp(-1, int(x), kCtrl, kRows, 0xF, false));
    x = y < x ? y : x;
  };
  using std::integral_constant;
  step(integral_constant<int, 0x111>{}, integral_constant<int, 0xF>{});  // row_shr:1, 2, 4, 8
  step(integral_constant<int, 0x112>{}, integral_constant<int, 0xF>{});
  step(integral_constant<int, 0x114>{}, integral_constant<int, 0xF>{});
  step(integral_constant<int, 0x118>{}, integral_constant<int, 0xF>{});
  step(integral_constant<int, 0x142>{}, integral_constant<int, 0xA>{});  // row_bcast:15 into rows 1 and 3
  step(integral_constant<int, 0x143>{}, integral_constant<int, 0xC>{});  // row_bcast:31 into rows 2 and 3
  return uint32_t(__builtin_amdgcn_readlane(int(x), 63));
}

// The itopk list of cagra_ahead_kernel, split so that the steps of one wave
// take few dependent instructions however long the list is.  A fully sorted
// list is not needed for the search: the next parent is the smallest
// unexpanded key, and it is in the list iff fewer than itopk expanded keys lie
// below it (no other unexpanded key does).
//  - front: the nearest unexpanded keys, sorted, one per lane.
//  - buf: keys on their way into `rest` (LDS).  They stay there unsorted until
//    front is taken anew: by then most of them lie beyond the list.
//  - rest: the other keys, sorted, at most itopk; bit 0 is set in expanded ones.
// Every unexpanded key outside front is at or above flim, every one in it
// below.  Keys at or above `bound`, the last key of a full list, cannot be
// in it and are dropped; keys beyond the list that are kept are harmless, as
// the test above rejects them as parents and the list is cut to itopk keys at
// the end.  One wave uses the pool; every member but front and rest is uniform
// over it.
constexpr int kAhead = 8;           // entries that one step may expand
constexpr int kIds = kAhead * 64;   // candidates of one step at most

template <int E>
struct Pool {
  static constexpr int kFull = 512;  // buf is emptied before a step at this many keys
  // A step below that adds its parents and all its candidates (a candidate
  // goes into buf itself or displaces one key of front into it) with no look
  // at nbuf in between.  Emptying it between two adds instead, with room for
  // 144 keys, took 1.5% longer (itopk 512 Q=100 816 us, 805 with this room).
  static constexpr int kBuf = kFull + kAhead + kIds;
  static constexpr int kNear = 65;               // refill: the nearest unexpanded keys and one more
  static constexpr int kLds = kBuf + kNear + 64 * E;
  uint64_t front, rest[E];
  uint64_t bound, flim;
  int nbuf, expanded, itopk;
  uint64_t* buf;

  // The seeds go to `rest` (merge_sorted); flim = 0 makes front take them.
  __device__ __forceinline__ void init(int itopk_, uint64_t* lds) {
    front = kEmptyKey;
#pragma unroll
    for (int e = 0; e < E; ++e) rest[e] = kEmptyKey;
    bound = kEmptyKey;
    flim = 0;
    nbuf = expanded = 0;
    itopk = itopk_;
    buf = lds;
  }
  // 64 sorted keys into `rest`.
  __device__ __forceinline__ void merge_sorted(uint64_t key) {
    const int lane = __lane_id();
    merge_into<E>(rest, key);
#pragma unroll
    for (int e = 0; e < E; ++e)
      if (e * 64 + lane >= itopk) rest[e] = kEmptyKey;
  }
  // The whole list into `rest`: front first, then what of `buf` is still
  // below the list's last key.
  __device__ __forceinline__ void collect() {
    merge_sorted(front);
    front = kEmptyKey;
#pragma unroll 1
    for (int b = 0; b < nbuf; b += 64) {
      const int i = b + int(__lane_id());
      add_keys<E>(rest, i < nbuf ? buf[i] : kEmptyKey, itopk, buf + kBuf);
    }
    nbuf = 0;
    const uint64_t w = last_key<E>(rest, itopk);
    bound = w < bound ? w : bound;  // (refill takes keys out of `rest` again)
  }
  __device__ __forceinline__ void refill() {
    const int lane = __lane_id();
    collect();
    uint64_t* near = buf + kBuf;
    uint64_t* kept = near + kNear;
    int nu = 0, nk = 0;
#pragma unroll
    for (int e = 0; e < E; ++e) {
      const bool un = rest[e] != kEmptyKey && (rest[e] & 1ull) == 0;
      const uint64_t m = __ballot(un);
      const int r = nu + mbcnt(m);
      if (un && r < kNear) near[r] = rest[e];
      const bool keep = rest[e] != kEmptyKey && !(un && r < 64);
      const uint64_t mk = __ballot(keep);
      if (keep) kept[nk + mbcnt(mk)] = rest[e];
      nu += popc(m);
      nk += popc(mk);
    }
    front = lane < nu ? near[lane] : kEmptyKey;
    const uint64_t next = near[nu > 64 ? 64 : 0];
    flim = nu > 64 ? (uint64_t(uint32_t(__builtin_amdgcn_readfirstlane(int(uint32_t(next >> 32))))) << 32) |
                         uint32_t(__builtin_amdgcn_readfirstlane(int(uint32_t(next))))
                   : kEmptyKey;
#pragma unroll
    for (int e = 0; e < E; ++e) rest[e] = e * 64 + lane < nk ? kept[e * 64 + lane] : kEmptyKey;
  }
  // Number of entries in `front`, at least `want` if there are as many
  // unexpanded keys at all.
  __device__ __forceinline__ int ready(int want) {
    int c = popc(__ballot(front != kEmptyKey));
    if ((c < want && flim != kEmptyKey) || nbuf >= kFull) {
      refill();
      c = popc(__ballot(front != kEmptyKey));
    }
    return c;
  }
  // True if fewer than `limit` expanded keys lie below p, which is at or below
  // every unexpanded key but those before it in `front`.
  __device__ __forceinline__ bool fewer_below(uint64_t p, int limit) const {
    int below = 0;
    for (int c = 0; c < nbuf; c += 64) {
      const int i = c + int(__lane_id());
      below += popc(__ballot(i < nbuf && buf[i < nbuf ? i : 0] < p));
    }
#pragma unroll
    for (int e = 0; e < E; ++e) below += popc(__ballot(rest[e] < p));
    return below < limit;
  }
  // The first `count` entries of `front` are expanded.
  __device__ __forceinline__ void expand(int count) {
    const int lane = __lane_id();
    if (lane < count) buf[nbuf + lane] = front | 1ull;
    nbuf += count;
    expanded += count;
    const uint64_t up = shfl_u64(front, (lane + count) & 63);
    front = lane + count < 64 ? up : kEmptyKey;
  }
  // Keys on their way into `rest`, one per lane (the empty key for none).
  __device__ __forceinline__ void push(uint64_t key) {
    const uint64_t m = __ballot(key != kEmptyKey);
    if (m == 0) return;
    if (key != kEmptyKey) buf[nbuf + mbcnt(m)] = key;
    nbuf += popc(m);
    const uint32_t hi = wave_min_u32(uint32_t(key >> 32));
    const uint32_t lo = wave_min_u32(uint32_t(key >> 32) == hi ? uint32_t(key) : 0xffffffffu);
    const uint64_t low = (uint64_t(hi) << 32) | lo;
    flim = low < flim ? low : flim;
  }
  // Candidate keys, one per lane (the empty key for none).
  __device__ __forceinline__ void add(uint64_t key) {
    push(key < flim ? kEmptyKey : key);
    if (sort_below(key, flim, kEmptyKey, buf + kBuf) == 0) return;
    // The 64 smallest of both stay; min and max of one ascending and one
    // descending list are its halves, the lower one bitonic.
    const int lane = __lane_id();
    const uint64_t other = shfl_xor_u64(key, 63);  // lane 63 - lane
    const uint64_t up = front < other ? other : front;
    front = front < other ? front : other;
#pragma unroll
    for (int stride = 32; stride >= 1; stride >>= 1) {
      const uint64_t y = shfl_xor_u64(front, stride);
      front = ((lane & stride) == 0) == (front < y) ? front : y;
    }
    push(up);
  }
};

// The same search for batches that leave compute units idle (W = 4 or 8,
// d <= 1024, bitmap visited set, degree <= 64, width <= kAhead, one team),
// where one query's chain of dependent steps is the time: per expanded node
// the graph row, the visited test, the rows, the merge (3.1 us a node at
// N=100K D=1024 fp32, of which the row bytes take 0.45 us at one compute
// unit's load bandwidth).  Here one step serves several nodes:
//  - the lead wave takes the `ahead` nearest unexpanded entries;
//  - the neighbours of those whose neighbours are not at hand yet are
//    collected (one entry per wave) and their rows gathered together, and
//    their keys kept per entry in one of kAhead slots;
//  - as many of the entries are expanded as the search would have expanded
//    one iteration after the other: iteration i + 1 takes the next `width`
//    entries iff no candidate of the iterations before is nearer than the
//    last of them.  Their candidates join the visited set and the pool
//    together; the other entries go back, their keys stay in their slots.
// An entry near the head of the list is nearly always expanded soon, so few
// evaluations are lost.  Parents, visited set, list and counts are, iteration
// by iteration, those of cagra_search_kernel.
// A call at N=100K D=1024 fp32: itopk 64 Q=1 213 -> 185 us in 20 steps for 65
// nodes, itopk 512 Q=100 1611 -> 806 us in 81 steps for 512.  Of the latter's
// 21,600 cycles a step, 7,700 are the gathers (27 rows; the latency of one
// alone is 4,700), 4,500 the entries' choice and the pool's refills, 2,300
// the new candidates, 2,400 the run of iterations and the visited set, 1,900
// the graph rows: latencies of single instructions of one wave for the most
// part.
constexpr int kAheadHash = 2 * kIds;  // ids of one step: at most half full

template <int E, int W, bool F16>
__global__ __launch_bounds__(64 * W, 2) void cagra_ahead_kernel(SearchArgs a, int ahead) {
  extern __shared__ uint32_t s_mem[];
  constexpr int kThreads = 64 * W, kTeams = 4 * W;
  constexpr int kPerWave = kAhead / W;   // entries per wave and step
  static_assert(kPerWave * W == kAhead, "entries per wave");
  uint32_t* s_bits = s_mem;                               // visited rows (bitmap_words: whole 256-byte blocks)
  uint64_t* s_key = reinterpret_cast<uint64_t*>(s_bits + a.bitmap_words);  // [slot][64] keys
  uint32_t* s_ids = reinterpret_cast<uint32_t*>(s_key + kIds);
  float* s_dist = reinterpret_cast<float*>(s_ids + kIds);
  uint32_t* s_hid = reinterpret_cast<uint32_t*>(s_dist + kIds);  // ids of this step -> position in s_ids
  uint32_t* s_hpos = s_hid + kAheadHash;
  uint64_t* s_cand = reinterpret_cast<uint64_t*>(s_ids);  // candidates of a step's expanded entries (ids and distances are done with)
  uint64_t* s_pick = reinterpret_cast<uint64_t*>(s_hpos + kAheadHash);  // keys of this step's entries
  uint32_t* s_slot = reinterpret_cast<uint32_t*>(s_pick + kAhead);      // their slots
  uint32_t* s_min = s_slot + kAhead;  // smallest distance word among an entry's unvisited neighbours
  // [0] entries of this step, [1] mask of those to collect for, [2] how many of
  // the first `width` are in the list, [3] most entries to expand, [4, 5] the
  // pool's bound, [6] seeds, then candidates, [7] ids of this step, [8]
  // distance evaluations
  uint32_t* s_ctl = s_min + kAhead;
  uint64_t* s_pool = reinterpret_cast<uint64_t*>(s_ctl + 16);
  float* s_q = reinterpret_cast<float*>(s_pool + Pool<E>::kLds + 1);  // fp16 traversal: the query, kBigDim floats
  const int tid = threadIdx.x, lane = tid & 63, team = tid >> 4, tp = lane & 15;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const bool lead = wave == 0;
  const int64_t qi = blockIdx.x / a.teams;
  const int tm = int(blockIdx.x - qi * a.teams);
  const float* qsrc = a.queries + qi * a.d;

  for (int i = tid; i < a.bitmap_words; i += kThreads) s_bits[i] = 0u;
  for (int i = tid; i < kAheadHash; i += kThreads) s_hid[i] = kInvalidId;
  if (tid < 16) s_ctl[tid] = 0u;
  Slice<F16> slice;
  {
    // Staged where the entries' keys will be, two barriers on; fp16 traversal
    // keeps the query as given in s_q for the final re-rank.
    static_assert(kIds * 2 >= kBigDim, "room for a query");
    float* const staged = reinterpret_cast<float*>(s_key);
    stage_query<F16>(a, qsrc, F16 ? s_q : staged, staged, kThreads);
    __syncthreads();
    slice.load(staged, tp);
  }

  // Distances of the rows s_ids[0..nf) into s_dist, two rows in flight per team.
  auto evaluate = [&](int nf) {
    using Piece = typename Slice<F16>::Piece;
    int r0 = 0;
    for (; nf - r0 > kTeams; r0 += 2 * kTeams) {
      const int ra = r0 + team, rb = ra + kTeams;
      Piece xa[Slice<F16>::N], xb[Slice<F16>::N];
      slice.fetch(a, s_ids[ra], tp, xa);
      slice.fetch(a, s_ids[rb < nf ? rb : ra], tp, xb);
      const float da = team_sum(slice.part(a, xa)), db = team_sum(slice.part(a, xb));
      if (tp == 0) {
        s_dist[ra] = da;
        if (rb < nf) s_dist[rb] = db;
      }
    }
    if (r0 < nf) {
      const int r = r0 + team;
      Piece x[Slice<F16>::N];
      slice.fetch(a, s_ids[r < nf ? r : r0], tp, x);
      const float d = team_sum(slice.part(a, x));
      if (tp == 0 && r < nf) s_dist[r] = d;
    }
  };
  auto visit = [&](uint32_t id) -> bool {  // true if id was not visited
    const uint32_t bit = 1u << (id & 31u);
    return (atomicOr(&s_bits[id >> 5], bit) & bit) == 0u;
  };

  Pool<E> pool;  // the list (lead wave)
  pool.init(a.itopk, s_pool);
  uint32_t sp = kInvalidId;  // lead wave, lane l < kAhead: the entry whose neighbours' keys slot l holds

  // Seeds (the sequence of cagra_search_kernel), kIds at a time.
  const uint32_t h0 = uint32_t(qi) * 2654435761u;
  uint32_t* s_raw = reinterpret_cast<uint32_t*>(s_dist);
  for (int c0 = 0; c0 < a.seed_lanes; c0 += kIds) {
    const int cnt = a.seed_lanes - c0 < kIds ? a.seed_lanes - c0 : kIds;
    for (int i = tid; i < cnt; i += kThreads) {
      const int x = (c0 + i) * a.teams + tm;
      uint32_t id = kInvalidId;
      if (x < a.n_seeds)
        id = a.seeds[x];
      else if (uint32_t(x - a.n_seeds) < a.n)
        id = (h0 + uint32_t(x - a.n_seeds) * 0x9E3779B9u) % a.n;
      s_raw[i] = id;
    }
    __syncthreads();
    if (lead) {
      int nf = 0;
      for (int c = 0; c < cnt; c += 64) {  // cnt is a multiple of 64
        const uint32_t id = s_raw[c + lane];
        const bool fresh = id < a.n && visit(id);
        const uint64_t m = __ballot(fresh);
        if (fresh) s_ids[nf + mbcnt(m)] = id;
        nf += popc(m);
      }
      if (lane == 0) {
        s_ctl[6] = uint32_t(nf);
        s_ctl[8] += uint32_t(nf);
      }
    }
    __syncthreads();
    const int nf = int(s_ctl[6]);
    evaluate(nf);
    __syncthreads();
    // Each wave sorts its 64-key runs, the lead wave merges them.
    for (int b = wave * 64; b < nf; b += W * 64) {
      const int i = b + lane;
      s_key[i] = wave_sort_lanes<64>(
          i < nf ? (uint64_t(ord_f32(s_dist[i])) << 32) | (uint64_t(s_ids[i]) << 1) : kEmptyKey);
    }
    __syncthreads();
    if (lead)
      for (int b = 0; b < nf; b += 64) pool.merge_sorted(s_key[b + lane]);
    __syncthreads();  // the next seeds are staged over the distances
  }

  int it = 0;
  for (;;) {
    if (lead) {
      int n = 0, first = 0, most = 0;
      uint32_t miss = 0;
      if (it < a.max_iter) {
        n = min(pool.ready(ahead), ahead);
        // Of the first `width` entries, those are parents that are in the
        // list: with fewer than itopk expanded keys below, counting the
        // parents before.  Later iterations are taken only where that is
        // certain.
        const int w = n < a.width ? n : a.width;
        const int sure = a.itopk - pool.expanded;
        for (; first < w; ++first)
          if (first >= sure && !pool.fewer_below(shfl_u64(pool.front, first), a.itopk - first)) break;
        most = first < a.width ? first : max(first, min(sure, n));
        if (first == 0) n = 0;
        // Lane i finds the slot that holds entry i's keys; entries without
        // one get, in order, the slots that no entry of this step holds.
        const uint32_t id = lane < n ? uint32_t(pool.front) >> 1 : kInvalidId - 1;
        uint32_t slot = kAhead, keep = 0;
#pragma unroll
        for (int l = 0; l < kAhead; ++l) {
          const bool mine = id == uint32_t(__builtin_amdgcn_readlane(int(sp), l));
          slot = mine ? uint32_t(l) : slot;
          keep |= __ballot(mine) != 0 ? 1u << l : 0u;
        }
        miss = uint32_t(__ballot(lane < n && slot == uint32_t(kAhead)));
        if (miss != 0) {
          const bool free = lane < kAhead && ((keep >> (lane & 31)) & 1u) == 0u;
          const int nth = mbcnt(__ballot(free));  // slot `lane` is the nth free one,
          if (free) s_slot[nth] = uint32_t(lane);
          if (slot == uint32_t(kAhead) && lane < n) {
            slot = s_slot[mbcnt(uint64_t(miss))];
            s_min[slot] = id;  // and takes the nth of these entries
          }
          if (free && nth < popc(uint64_t(miss))) sp = s_min[lane];
        }
        if (lane < n) {
          s_pick[lane] = pool.front;
          s_slot[lane] = slot;
        }
      }
      if (lane == 0) {
        *reinterpret_cast<uint4*>(s_ctl) = uint4{uint32_t(n), miss, uint32_t(first), uint32_t(most)};
        *reinterpret_cast<uint4*>(s_ctl + 4) = uint4{uint32_t(pool.bound), uint32_t(pool.bound >> 32), 0u, 0u};
      }
    }
    __syncthreads();
    const uint4 ctl = *reinterpret_cast<const uint4*>(s_ctl);
    const int n = __builtin_amdgcn_readfirstlane(int(ctl.x));
    const uint32_t miss = uint32_t(__builtin_amdgcn_readfirstlane(int(ctl.y)));
    if (n == 0) break;
    // Each wave serves its entries of the step: the keys of their neighbours
    // from their slots, or collected and gathered.
    uint64_t key[kPerWave];
    uint32_t id[kPerWave], slot[kPerWave];
    int pos[kPerWave];  // collected: hash position, -1: no candidate
#pragma unroll
    for (int t = 0; t < kPerWave; ++t) {
      const int p = wave + t * W;
      key[t] = kEmptyKey;
      id[t] = kInvalidId;
      slot[t] = 0;
      if (p < n) {
        slot[t] = s_slot[p];
        if ((miss >> p) & 1u) {
          if (lane < a.g) id[t] = a.graph[int64_t(uint32_t(s_pick[p]) >> 1) * a.g + lane];
        } else {
          key[t] = s_key[slot[t] * 64 + lane];
          id[t] = uint32_t(key[t]) >> 1;  // >= n for none
        }
      }
    }
    bool open[kPerWave];  // not visited
#pragma unroll
    for (int t = 0; t < kPerWave; ++t)
      open[t] = id[t] < a.n && ((s_bits[id[t] < a.n ? id[t] >> 5 : 0] >> (id[t] & 31u)) & 1u) == 0u;
    if (miss != 0) {
      // Each id of the step once.
#pragma unroll
      for (int t = 0; t < kPerWave; ++t) {
        pos[t] = -1;
        if (((miss >> (wave + t * W)) & 1u) == 0) continue;
        bool first_seen = false;
        if (open[t]) {
          uint32_t h = (id[t] * 0x9E3779B1u) >> 22;  // kAheadHash positions
          for (;;) {
            const uint32_t old = atomicCAS(&s_hid[h], kInvalidId, id[t]);
            first_seen = old == kInvalidId;
            if (first_seen || old == id[t]) break;
            h = (h + 1u) & uint32_t(kAheadHash - 1);
          }
          pos[t] = int(h);
        }
        const uint64_t m = __ballot(first_seen);
        if (m != 0) {
          uint32_t base = 0;
          if (lane == 0) base = atomicAdd(&s_ctl[7], uint32_t(popc(m)));
          base = uint32_t(__builtin_amdgcn_readfirstlane(int(base)));
          if (first_seen) {
            const uint32_t at = base + uint32_t(mbcnt(m));
            s_ids[at] = id[t];
            s_hpos[pos[t]] = at;
          }
        }
      }
      __syncthreads();
      evaluate(int(s_ctl[7]));
      __syncthreads();
#pragma unroll
      for (int t = 0; t < kPerWave; ++t) {
        if (((miss >> (wave + t * W)) & 1u) == 0) continue;
        if (pos[t] >= 0) key[t] = (uint64_t(ord_f32(s_dist[s_hpos[pos[t]]])) << 32) | (uint64_t(id[t]) << 1);
        s_key[slot[t] * 64 + lane] = key[t];
      }
    }
    // The nearest unvisited neighbour of each entry.
#pragma unroll
    for (int t = 0; t < kPerWave; ++t) {
      const int p = wave + t * W;
      if (!open[t]) key[t] = kEmptyKey;
      const uint32_t mn = wave_min_u32(uint32_t(key[t] >> 32));
      if (lane == 0 && p < n) s_min[p] = mn;
    }
    __syncthreads();
    // The iterations that follow one another whatever their candidates are
    // (equal distances end the run; the next step then looks at the ids):
    // entry j ends an iteration that may follow if the nearest neighbour of
    // all iterations before it lies beyond it.
    int c = __builtin_amdgcn_readfirstlane(int(ctl.z)), iters = 1;
    {
      const int most = __builtin_amdgcn_readfirstlane(int(ctl.w));
      uint32_t before = lane < n ? s_min[lane & (kAhead - 1)] : 0xffffffffu;  // of entries 0 .. lane
      const uint32_t own = uint32_t(s_pick[lane & (kAhead - 1)] >> 32);
      // Running minimum by DPP row shifts (kAhead lanes of the first row).
      static_assert(kAhead == 8, "three row shifts");
      before = min(before, uint32_t(__builtin_amdgcn_update_dpp(-1, int(before), 0x111, 0xF, 0xF, false)));
      before = min(before, uint32_t(__builtin_amdgcn_update_dpp(-1, int(before), 0x112, 0xF, 0xF, false)));
      before = min(before, uint32_t(__builtin_amdgcn_update_dpp(-1, int(before), 0x114, 0xF, 0xF, false)));
      before = a.width == 1 ? uint32_t(__builtin_amdgcn_update_dpp(-1, int(before), 0x111, 0xF, 0xF, false))
                            : uint32_t(__shfl_up(int(before), a.width));
      const uint64_t ok = __ballot(lane >= a.width && lane < most && before > own);
      while (c + a.width <= most && it + iters < a.max_iter && ((ok >> (c + a.width - 1)) & 1ull)) {
        c += a.width;
        ++iters;
      }
    }
    it += iters;
    if (miss != 0)  // empty for the next step, which starts with a barrier
      for (int i = tid; i < kAheadHash; i += kThreads) s_hid[i] = kInvalidId;
    const uint64_t bound = *reinterpret_cast<const uint64_t*>(s_ctl + 4);
#pragma unroll
    for (int t = 0; t < kPerWave; ++t) {
      if (wave + t * W >= c) continue;
      const bool fresh = key[t] != kEmptyKey && visit(id[t]);
      const uint64_t m = __ballot(fresh && key[t] < bound);
      const int nfresh = popc(__ballot(fresh));
      uint32_t base = 0;
      if (lane == 0) {
        base = atomicAdd(&s_ctl[6], uint32_t(popc(m)));
        atomicAdd(&s_ctl[8], uint32_t(nfresh));
      }
      base = uint32_t(__builtin_amdgcn_readfirstlane(int(base)));
      if ((m >> lane) & 1ull) s_cand[base + mbcnt(m)] = key[t];
    }
    __syncthreads();
    if (lead) {
      const int nc = int(s_ctl[6]);
      // The expanded entries' slots are free.
      for (int i = 0; i < c; ++i) {
        const uint32_t x = uint32_t(__builtin_amdgcn_readlane(int(uint32_t(pool.front)), i)) >> 1;
        sp = sp == x ? kInvalidId : sp;
      }
      pool.expand(c);
      for (int b = 0; b < nc; b += 64) pool.add(b + lane < nc ? s_cand[b + lane] : kEmptyKey);
    }
  }

  if (lead) pool.collect();
  if constexpr (F16)
    rerank_list<E, W>(pool.rest, lead, s_ids, s_dist,
                      [&](uint32_t rid) { return team_sum(exact_part(a, s_q, rid, tp)); });
  if (lead) write_list<E>(a, pool.rest, qi, s_ctl[8], it);
}

// Waves per query (workgroups = queries x teams): 8 up to 128 workgroups, 4
// up to 512, else 2.  With 2 or more waves the lead wave's serial work (hash,
// sort, merge) overlaps other queries' gathers on the same SIMD without
// losing the gathering teams.  Wall time per batch at N=100K D=1024 itopk 64
// with the visited-hash sizes below (fp16 / fp32 traversal):
//   W=2: Q=1 0.28 / 0.33, Q=300 0.36 / 0.41, Q=1,000 0.42 / 0.63, Q=10,000 3.21 / 5.78 ms
//   W=4: Q=1 0.22 / 0.26, Q=300 0.28 / 0.36, Q=1,000 0.57 / 0.76, Q=10,000 3.96 / 5.69 ms
//   W=8: Q=1 0.23 / 0.26, Q=300 0.49 / 0.59, Q=1,000 1.00 / 1.20, Q=10,000 9.64 / 11.4 ms
// (one wave per query: Q=10,000 4.62 / 8.45 ms with the smallest table).
int waves_per_query(int64_t workgroups) {
  return workgroups <= 128 ? 8 : (workgroups <= 512 ? 4 : 2);
}

template <int E, bool F16>
void launch_search(int waves, bool big, int ahead, dim3 grid, size_t lds, hipStream_t stream, const SearchArgs& a,
                   hipEvent_t e0, hipEvent_t e1) {
  if (ahead > 0) {
    auto go = [&](auto kernel, int threads) {
      if (lds > 64 * 1024)  // fp16 traversal, itopk > 256, more than 253,952 rows
        CVS_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                    int(lds)));
      hipExtLaunchKernelGGL(kernel, grid, dim3(threads), lds, stream, e0, e1, 0, a, ahead);
    };
    if (waves == 8) {
      go(cagra_ahead_kernel<E, 8, F16>, 512);
      return;
    }
    if constexpr (E > 1) {
      go(cagra_ahead_kernel<E, 4, F16>, 256);
      return;
    }
  }
  if (big) {  // d > 1024: four waves per query at any batch size
    if (lds > 64 * 1024)
      CVS_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(cagra_search_kernel<E, 4, F16, true>),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, int(lds)));
    hipExtLaunchKernelGGL((cagra_search_kernel<E, 4, F16, true>), grid, dim3(256), lds, stream, e0, e1, 0, a);
    return;
  }
  switch (waves) {
    case 2: hipExtLaunchKernelGGL((cagra_search_kernel<E, 2, F16, false>), grid, dim3(128), lds, stream, e0, e1, 0, a); break;
    case 4: hipExtLaunchKernelGGL((cagra_search_kernel<E, 4, F16, false>), grid, dim3(256), lds, stream, e0, e1, 0, a); break;
    default: hipExtLaunchKernelGGL((cagra_search_kernel<E, 8, F16, false>), grid, dim3(512), lds, stream, e0, e1, 0, a); break;
  }
}

template <int E>
void launch_search(bool f16, int waves, bool big, int ahead, dim3 grid, size_t lds, hipStream_t stream,
                   const SearchArgs& a, hipEvent_t e0, hipEvent_t e1) {
  if (f16)
    launch_search<E, true>(waves, big, ahead, grid, lds, stream, a, e0, e1);
  else
    launch_search<E, false>(waves, big, ahead, grid, lds, stream, a, e0, e1);
}

// Merge of the teams' lists of one query (one wave per query): the teams x
// itopk keys are sorted, an id found by several teams is kept once (every
// team computes the same fp32 distance for it, so copies are adjacent once
// the expanded bit is ignored), and the k smallest are written, padded with
// UINT32_MAX / +inf.  The reference merges its teams' beams on the host with
// the same dedupe (src/metal_context.mm:1003-1035).
template <int E2>
__global__ __launch_bounds__(64) void team_merge_kernel(const uint64_t* __restrict__ keys, int total, int k,
                                                        uint32_t* __restrict__ out_nbr, float* __restrict__ out_dist) {
  const int64_t qi = blockIdx.x;
  const int lane = threadIdx.x;
  uint64_t v[E2];
#pragma unroll
  for (int e = 0; e < E2; ++e) {
    const int pos = e * 64 + lane;
    v[e] = pos < total ? (keys[qi * total + pos] | 1ull) : kEmptyKey;
  }
  wave_sort_e<E2>(v);
  int base = 0;
  uint32_t carry_lo = 0, carry_hi = 0;  // key at the previous slot's lane 63
#pragma unroll
  for (int e = 0; e < E2; ++e) {
    const uint32_t lo = uint32_t(v[e]), hi = uint32_t(v[e] >> 32);
    uint32_t plo = uint32_t(__shfl_up(int(lo), 1)), phi = uint32_t(__shfl_up(int(hi), 1));
    if (lane == 0) {
      plo = carry_lo;
      phi = carry_hi;
    }
    const uint64_t prev = (uint64_t(phi) << 32) | plo;
    const bool uniq = v[e] != kEmptyKey && ((e == 0 && lane == 0) || v[e] != prev);
    const uint64_t m = __ballot(uniq);
    const int rank = base + mbcnt(m);
    if (uniq && rank < k) {
      out_nbr[qi * k + rank] = uint32_t(v[e]) >> 1;
      out_dist[qi * k + rank] = unord_f32(uint32_t(v[e] >> 32));
    }
    base += popc(m);
    carry_lo = uint32_t(__builtin_amdgcn_readlane(int(lo), 63));
    carry_hi = uint32_t(__builtin_amdgcn_readlane(int(hi), 63));
  }
  for (int r = base + lane; r < k; r += 64) {
    out_nbr[qi * k + r] = kInvalidId;
    out_dist[qi * k + r] = INFINITY;
  }
}

// fp32 rows (n x dpad) -> the fp16 traversal copy of scale * (row - mu)
// (round to nearest even), 8 values per thread.  Centring keeps the fp16
// rounding proportional to the rows' spread, not their offset from the
// origin; the query is centred and scaled the same way in the search.
__global__ void rows_to_half_kernel(const float4* __restrict__ src, size_t pieces, int dpad8,
                                    const float4* __restrict__ mu, float scale, uint4* __restrict__ dst) {
  const size_t i = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i >= pieces) return;
  const size_t c = (i % size_t(dpad8)) * 2;  // float4 column of the piece
  const float4 lo = src[2 * i], hi = src[2 * i + 1];
  const float4 ml = mu[c], mh = mu[c + 1];
  half8_t h;
  h[0] = _Float16((lo.x - ml.x) * scale);
  h[1] = _Float16((lo.y - ml.y) * scale);
  h[2] = _Float16((lo.z - ml.z) * scale);
  h[3] = _Float16((lo.w - ml.w) * scale);
  h[4] = _Float16((hi.x - mh.x) * scale);
  h[5] = _Float16((hi.y - mh.y) * scale);
  h[6] = _Float16((hi.z - mh.z) * scale);
  h[7] = _Float16((hi.w - mh.w) * scale);
  dst[i] = __builtin_bit_cast(uint4, h);
}

// Exact squared L2 length of every graph edge (the reference's
// recompute_graph_distances, shaders/cagra_kernels.metal:658-681).  One
// workgroup per node: the node's row stays in registers (float4 columns
// tp + 16 j per lane of each 16-lane team) and the 16 teams gather the
// neighbour rows, 256 contiguous bytes per load instruction and team.  Rows
// wider than 1,024 columns (BIG) go in chunks of 1,024, the node's piece of
// each chunk loaded again (from the caches).  Entries that are not row ids
// (UINT32_MAX, or >= n) get +inf.
template <bool BIG>
__global__ __launch_bounds__(256) void edge_distances_kernel(const float4* __restrict__ rows, int dq, int dv,
                                                             const uint32_t* __restrict__ graph, int g, uint32_t n,
                                                             float* __restrict__ out) {
  const int64_t node = blockIdx.x;
  const int tid = threadIdx.x, team = tid >> 4, tp = tid & 15;
  float4 xv[kMaxDv];
  const float4* self = rows + node * dq + tp;
  if constexpr (!BIG) {
#pragma unroll
    for (int j = 0; j < kMaxDv; ++j)
      if (j < dv) xv[j] = self[16 * j];
  }
  for (int e = team; e < g; e += 16) {
    const uint32_t nb = graph[node * g + e];
    const bool valid = nb < n;
    const float4* row = rows + int64_t(valid ? nb : uint32_t(node)) * dq + tp;
    float acc = 0.f;
    for (int c0 = 0; c0 < (BIG ? dq : 1); c0 += 256) {
      const int nj = BIG ? ((dq - c0) / 16 < kMaxDv ? (dq - c0) / 16 : kMaxDv) : dv;
      if constexpr (BIG) {
#pragma unroll
        for (int j = 0; j < kMaxDv; ++j)
          if (j < nj) xv[j] = self[c0 + 16 * j];
      }
      float4 x[kMaxDv];
#pragma unroll
      for (int j = 0; j < kMaxDv; ++j)
        if (j < nj) x[j] = row[c0 + 16 * j];
#pragma unroll
      for (int j = 0; j < kMaxDv; ++j) {
        if (j < nj) {
          const float dx = xv[j].x - x[j].x, dy = xv[j].y - x[j].y;
          const float dz = xv[j].z - x[j].z, dw = xv[j].w - x[j].w;
          acc += (dx * dx + dy * dy) + (dz * dz + dw * dw);
        }
      }
    }
    acc += xor_lanes_f(acc, 8);
    acc += xor_lanes_f(acc, 4);
    acc += xor_lanes_f(acc, 2);
    acc += xor_lanes_f(acc, 1);
    if (tp == 0) out[node * g + e] = valid ? acc : INFINITY;
  }
}

// Gathers, for every query, the rows its search evaluated (recorded by
// cvs_cagra_search_record_async), with the search's row shape and no search
// work: one workgroup per query, 16 teams of 16 lanes, lane l reading the
// 16-byte pieces l, l + 16, ... of a row (256 contiguous bytes per team and
// load), two rows in flight per team.  The time of this launch is the
// search's data movement alone.
__global__ __launch_bounds__(256) void gather_replay_kernel(const uint4* __restrict__ rows, int row_vecs,
                                                            const uint32_t* __restrict__ record, int cap,
                                                            const uint32_t* __restrict__ stats,
                                                            uint32_t* __restrict__ sink) {
  const int64_t qi = blockIdx.x;
  const int team = threadIdx.x >> 4, tp = threadIdx.x & 15;
  const uint32_t ev = stats[2 * qi];
  const int cnt = int(ev < uint32_t(cap) ? ev : uint32_t(cap));
  const uint32_t* ids = record + qi * cap;
  uint32_t acc = 0;
  for (int i = team; i < cnt; i += 32) {
    const uint4* r0 = rows + int64_t(ids[i]) * row_vecs + tp;
    const uint4* r1 = rows + int64_t(ids[i + 16 < cnt ? i + 16 : i]) * row_vecs + tp;
    for (int c0 = 0; c0 < row_vecs; c0 += 256) {
      uint4 v0[16], v1[16];
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        const int c = c0 + tp + 16 * j;
        v0[j] = c < row_vecs ? r0[c0 + 16 * j] : uint4{0, 0, 0, 0};
        v1[j] = (c < row_vecs && i + 16 < cnt) ? r1[c0 + 16 * j] : uint4{0, 0, 0, 0};
      }
#pragma unroll
      for (int j = 0; j < 16; ++j) acc ^= v0[j].x ^ v0[j].w ^ v1[j].y ^ v1[j].z;
    }
  }
  if (acc == 0x9E3779B9u) sink[qi * 256 + threadIdx.x] = acc;
}

int ceil_log2(int64_t v) {
  int b = 0;
  while ((int64_t(1) << b) < v) ++b;
  return b;
}

// Shortest list with which cagra_ahead_kernel is faster than
// cagra_search_kernel (4 or 8 waves per query, up to 512 queries).  It saves
// the other kernel's steps, one per iteration, where most expansions are of
// entries that have been in the list for some time, and loses the rows that it
// gathers in vain.  Three things decide, all measured on both kernels at 15,000
// to 100,000 rows, d = 96 to 1,024, degree 16 to 64, fp32 and fp16 (ratios of
// the times, other kernel / this one; fp32, 100,000 x 768, degree 64 unless
// said otherwise):
//  - the list: width 1, Q = 1, itopk 48 0.99, 64 1.11, 128 1.50, 512 2.07.
//  - queries that share the caches' bandwidth: itopk 64, Q = 60 1.03 (15,000 x
//    256, Q = 30: 0.76), 128 0.87; with four waves (beyond 128 queries) Q = 300,
//    itopk 128 0.88, 256 1.16, 512 1.62.  A wide search gathers little in vain:
//    width 8, itopk 65, Q = 128 1.33, Q = 300 1.10.
//  - iterations of several parents with one chunk of 64 candidates: degree 32,
//    width 2, Q = 1, itopk 64 0.72, 128 0.90, 256 1.18, 512 1.40; degree 16,
//    width 4, itopk 512 0.91.
// Below the line the two differ little or the other kernel is faster.  A batch
// takes as long as its longest walk, so single ones lie on the other side
// (30,000 x 512, width 1, itopk 96 to 192, Q = 60, one walk of 384 nodes: 0.84).
int64_t ahead_from(int waves, int64_t q, int64_t n, int64_t width, int64_t degree) {
  const double parents = double(width) / double((width * degree + 63) / 64);  // per chunk
  if (parents > 2.0) return CVS_CAGRA_MAX_ITOPK + 1;
  double least;
  if (waves == 8) {
    const bool few = q <= 8 || (q <= 64 && n >= 32'768);
    least = width == 1 ? (few ? 64.0 : 96.0) * std::max(1.0, 32.0 / double(degree))
                       : (width <= 4 ? 64.0 : (width <= 6 ? 48.0 : 33.0));
  } else {
    least = width == 1 ? (q <= 384 ? 256.0 : 512.0)
                       : (width <= 3 ? 256.0 : (width == 4 ? 192.0 : (width <= 6 ? 128.0 : 65.0)));
  }
  return int64_t(std::min(512.0, least * parents * parents));
}

void cagra_search_device(cvs_context* ctx, const cvs_cagra_index* idx, const float* queries,
                         int64_t q, int64_t k, uint32_t itopk_size, uint32_t search_width,
                         uint32_t max_iterations, uint32_t* nbr, float* dist, uint32_t* stats, int teams = 1,
                         uint32_t* record = nullptr, int record_cap = 0) {
  if (!idx || idx->ctx != ctx) fail(CVS_ERR_INVALID_ARGUMENT, "index does not belong to context");
  if (!queries || !nbr || !dist) fail(CVS_ERR_INVALID_ARGUMENT, "null buffer");
  if (q <= 0) fail(CVS_ERR_INVALID_ARGUMENT, "query count must be positive");
  if (k <= 0) fail(CVS_ERR_INVALID_ARGUMENT, "k must be positive");
  if (q > int64_t(INT32_MAX)) fail(CVS_ERR_UNSUPPORTED, "too many queries in one call");
  const int64_t itopk = std::max<int64_t>(itopk_size ? itopk_size : 128, k);
  if (itopk > CVS_CAGRA_MAX_ITOPK)
    fail(CVS_ERR_UNSUPPORTED, "itopk_size (or k) exceeds CVS_CAGRA_MAX_ITOPK");
  if (teams < 1 || teams > CVS_CAGRA_MAX_TEAMS) fail(CVS_ERR_INVALID_ARGUMENT, "teams must be in [1, CVS_CAGRA_MAX_TEAMS]");
  if (teams > 1 && int64_t(teams) * itopk > CVS_CAGRA_MAX_ITOPK)
    fail(CVS_ERR_UNSUPPORTED, "teams * itopk_size exceeds CVS_CAGRA_MAX_ITOPK");
  if (q * teams > int64_t(INT32_MAX)) fail(CVS_ERR_UNSUPPORTED, "too many queries in one call");
  const int64_t width = search_width ? search_width : 1;
  if (width > CVS_CAGRA_MAX_WIDTH) fail(CVS_ERR_UNSUPPORTED, "search_width exceeds CVS_CAGRA_MAX_WIDTH");
  const int64_t per_iter = width * int64_t(idx->degree);
  if (per_iter > 2048) fail(CVS_ERR_UNSUPPORTED, "search_width * graph_degree exceeds 2048");
  const int e_slots = itopk <= 64 ? 1 : (itopk <= 128 ? 2 : (itopk <= 256 ? 4 : 8));
  int64_t iters = max_iterations;
  if (iters == 0) iters = std::max<int64_t>(200, 2 * itopk / width);
  const bool big = idx->d > kBigDim;
  const int waves = big ? 4 : waves_per_query(q * teams);
  // The visited hash at twice (W=2) or four times (W=4, 8) the size that
  // keeps it half empty, up to 2^13 entries (32 KiB): the lead wave's probe
  // chains stay short, and fewer mid-search clears mean fewer rows evaluated
  // twice.  W=2 serves the large batches, where a 2^13 table would cost
  // workgroups per CU (fp16 traversal, Q=10,000: 3.21 ms at 2^12, 3.70 ms at
  // 2^13, 4.43 ms at 2^11).
  int hash_bits = std::max(11, ceil_log2(2 * (64 * e_slots + std::max<int64_t>(64, per_iter))));
  hash_bits = std::max(hash_bits, std::min(hash_bits + (waves >= 4 ? 2 : 1), 13));
  // A bitmap of the n rows where it takes no more LDS than the hash: one
  // atomic per id, no probing, never cleared.  Whole 256-byte blocks keep the
  // words after it 8-byte aligned.
  const int64_t bitmap_words = (idx->n + 2047) / 2048 * 64;
  const bool use_bitmap = bitmap_words <= (int64_t(1) << hash_bits);
  const size_t visit_words = use_bitmap ? size_t(bitmap_words) : (size_t(1) << hash_bits);
  // (The visited set's words hold the query first, see cagra_search_kernel.)
  // Small batches gather for several entries at a time (cagra_ahead_kernel)
  // where that is the faster way (ahead_from).  Teams walk from scattered seeds
  // with short lists (8 teams x 32, Q=1: 123 us without it, 175 with it; 4 x 64:
  // 213 / 250; not taken).  Six entries are best for one key per lane (4: 196,
  // 8: 192 us at Q=1), eight for longer lists.
  int ahead = 0;
  if (waves >= 4 && !big && use_bitmap && idx->degree <= 64 && width <= kAhead && teams == 1 && !record &&
      itopk >= ahead_from(waves, q, idx->n, width, idx->degree))
    ahead = std::max(itopk > 64 ? kAhead : 6, int(width));
  const bool f16 = idx->traversal_bits == 16;
  size_t lds = (big ? visit_words : std::max<size_t>(visit_words, kBigDim)) * 4 + (64 + 64 + CVS_CAGRA_MAX_WIDTH + 8) * 4 +
               (big ? size_t(idx->dpad) * 4 * (f16 ? 2 : 1) : (f16 ? size_t(kBigDim) * 4 : 0));
  if (ahead > 0)  // the kernel's arrays, in its order
    lds = visit_words * 4 + size_t(kIds) * 16 + size_t(kAheadHash) * 8 + (4 * kAhead + 16) * 4 +
          size_t(Pool<1>::kLds + 64 * (e_slots - 1) + 1) * 8 + (f16 ? size_t(kBigDim) * 4 : 0);

  SearchArgs a{};
  a.rows = reinterpret_cast<const float4*>(idx->rows);
  a.graph = idx->graph;
  a.seeds = idx->seeds;
  a.queries = queries;
  a.out_nbr = nbr;
  a.out_dist = dist;
  a.stats = stats;
  a.d = idx->d;
  a.n = uint32_t(idx->n);
  a.g = int(idx->degree);
  a.rows16 = reinterpret_cast<const uint4*>(idx->rows16);
  a.mu = idx->mu;
  a.scale = idx->scale;
  a.dq = int(idx->dpad / 4);
  a.dv = int(idx->dpad / 64);
  a.dq8 = int(idx->dpad / 8);
  a.dv8 = int(idx->dpad / 128);
  a.n_seeds = int(idx->n_seeds);
  // At least itopk candidates (all seed nodes, then hashed ids; each team its
  // share of the seed nodes), in whole chunks of 64: a list of itopk entries
  // starts from as many distinct rows.
  const int64_t team_seeds = (int64_t(idx->n_seeds) + teams - 1) / teams;
  a.seed_lanes = int((std::max<int64_t>({team_seeds, itopk, 1}) + 63) / 64 * 64);
  a.k = int(k);
  a.itopk = int(itopk);
  a.width = int(width);
  a.max_iter = int(std::min<int64_t>(iters, INT32_MAX));
  a.hash_bits = hash_bits;
  a.bitmap_words = use_bitmap ? int(bitmap_words) : 0;
  a.teams = teams;
  a.record = teams == 1 ? record : nullptr;
  a.record_cap = record_cap;
  if (teams > 1) {
    ctx->ws_teams.reserve(size_t(q) * size_t(teams) * size_t(itopk) * sizeof(uint64_t));
    a.team_keys = ctx->ws_teams.as<uint64_t>();
    a.stats = nullptr;
  }

  const TimerSpan t0 = timer_span(ctx, "cagra_search");
  const dim3 grid(static_cast<unsigned>(q * teams));
  // The search kernel starts the span; the team merge (if any) ends it.
  hipEvent_t e1 = teams > 1 ? nullptr : t0.stop;
  switch (e_slots) {
    case 1: launch_search<1>(f16, waves, big, ahead, grid, lds, ctx->stream, a, t0.start, e1); break;
    case 2: launch_search<2>(f16, waves, big, ahead, grid, lds, ctx->stream, a, t0.start, e1); break;
    case 4: launch_search<4>(f16, waves, big, ahead, grid, lds, ctx->stream, a, t0.start, e1); break;
    default: launch_search<8>(f16, waves, big, ahead, grid, lds, ctx->stream, a, t0.start, e1); break;
  }
  after_launch("cagra_search_kernel");
  if (teams > 1) {
    const int total = int(teams * itopk);
    const uint64_t* keys = a.team_keys;
    const dim3 mg{unsigned(q)}, mb{64};
    if (total <= 64)
      hipExtLaunchKernelGGL(team_merge_kernel<1>, mg, mb, 0, ctx->stream, nullptr, t0.stop, 0, keys, total, int(k), nbr, dist);
    else if (total <= 128)
      hipExtLaunchKernelGGL(team_merge_kernel<2>, mg, mb, 0, ctx->stream, nullptr, t0.stop, 0, keys, total, int(k), nbr, dist);
    else if (total <= 256)
      hipExtLaunchKernelGGL(team_merge_kernel<4>, mg, mb, 0, ctx->stream, nullptr, t0.stop, 0, keys, total, int(k), nbr, dist);
    else
      hipExtLaunchKernelGGL(team_merge_kernel<8>, mg, mb, 0, ctx->stream, nullptr, t0.stop, 0, keys, total, int(k), nbr, dist);
    after_launch("team_merge_kernel");
  }
}

}  // namespace
}  // namespace cvs

using namespace cvs;

extern "C" {

int cvs_cagra_nav_nodes(int64_t n, uint32_t* out_ids, int64_t* out_count) {
  return guarded([&] {
    if (!out_count) fail(CVS_ERR_INVALID_ARGUMENT, "null out_count");
    if (n <= 0) fail(CVS_ERR_INVALID_ARGUMENT, "row count must be positive");
    if (n > int64_t(UINT32_MAX)) fail(CVS_ERR_UNSUPPORTED, "row ids must fit in uint32");
    // min(200, floor(sqrt(n))) rows, row i at floor(i * (n / n_nav)) with the
    // spacing taken in double (src/cagra.cpp:65-72).
    int64_t n_nav = static_cast<int64_t>(std::sqrt(static_cast<double>(n)));
    if (n_nav > 200) n_nav = 200;
    *out_count = n_nav;
    if (out_ids) {
      const double step = static_cast<double>(n) / static_cast<double>(n_nav);
      for (int64_t i = 0; i < n_nav; ++i) out_ids[i] = static_cast<uint32_t>(static_cast<double>(i) * step);
    }
  });
}

int cvs_cagra_index_create(cvs_context* ctx, const float* rows, int64_t n, int64_t d,
                           int rows_on_device, const uint32_t* graph, uint32_t degree,
                           int graph_on_device, const uint32_t* seeds, uint32_t n_seeds,
                           cvs_cagra_index** out_index) {
  return guarded([&] {
    bind(ctx);
    if (!out_index) fail(CVS_ERR_INVALID_ARGUMENT, "null out_index");
    *out_index = nullptr;
    if (!rows || n <= 0 || d <= 0) fail(CVS_ERR_INVALID_ARGUMENT, "dataset must be non-null and non-empty");
    if (!graph || degree == 0) fail(CVS_ERR_INVALID_ARGUMENT, "graph must be non-null with degree > 0");
    if (n_seeds > 0 && !seeds) fail(CVS_ERR_INVALID_ARGUMENT, "null seed ids");
    if (n > int64_t(INT32_MAX)) fail(CVS_ERR_UNSUPPORTED, "graph search needs n < 2^31");
    if (d > CVS_CAGRA_MAX_DIM) fail(CVS_ERR_UNSUPPORTED, "dimension exceeds CVS_CAGRA_MAX_DIM");
    if (degree > 1024) fail(CVS_ERR_UNSUPPORTED, "graph degree exceeds 1024");
    for (uint32_t i = 0; i < n_seeds; ++i)
      if (seeds[i] >= uint64_t(n)) fail(CVS_ERR_INVALID_ARGUMENT, "seed id out of range");
    auto* ix = new cvs_cagra_index();
    ix->ctx = ctx;
    ix->n = n;
    ix->d = d;
    ix->dpad = (d + 127) / 128 * 128;
    ix->degree = degree;
    ix->n_seeds = n_seeds;
    try {
      const size_t row_bytes = size_t(n) * size_t(ix->dpad) * sizeof(float);
      CVS_HIP(hipMalloc(&ix->rows, row_bytes));
      CVS_HIP(hipMalloc(&ix->graph, size_t(n) * degree * sizeof(uint32_t)));
      if (n_seeds) CVS_HIP(hipMalloc(&ix->seeds, size_t(n_seeds) * sizeof(uint32_t)));
      if (ix->dpad != d) CVS_HIP(hipMemsetAsync(ix->rows, 0, row_bytes, ctx->stream));
      upload_rows(ctx, ix->rows, ix->dpad, rows, n, d, rows_on_device);
      CVS_HIP(hipMalloc(&ix->rows16, size_t(n) * size_t(ix->dpad) * 2));
      CVS_HIP(hipMalloc(&ix->mu, size_t(ix->dpad) * sizeof(float)));
      ix->scale = centre_rows(ctx, ix->rows, n, ix->dpad, ix->dpad, ix->mu);
      hipLaunchKernelGGL(rows_to_half_kernel, dim3(unsigned((size_t(n) * size_t(ix->dpad) / 8 + 255) / 256)), dim3(256),
                         0, ctx->stream, reinterpret_cast<const float4*>(ix->rows), size_t(n) * size_t(ix->dpad) / 8,
                         int(ix->dpad / 8), reinterpret_cast<const float4*>(ix->mu), ix->scale,
                         reinterpret_cast<uint4*>(ix->rows16));
      after_launch("rows_to_half_kernel");
      CVS_HIP(hipMemcpyAsync(ix->graph, graph, size_t(n) * degree * sizeof(uint32_t),
                             graph_on_device ? hipMemcpyDeviceToDevice : hipMemcpyHostToDevice, ctx->stream));
      if (n_seeds)
        CVS_HIP(hipMemcpyAsync(ix->seeds, seeds, size_t(n_seeds) * sizeof(uint32_t), hipMemcpyHostToDevice,
                               ctx->stream));
      CVS_HIP(hipStreamSynchronize(ctx->stream));
    } catch (...) {
      if (ix->rows) (void)hipFree(ix->rows);
      if (ix->rows16) (void)hipFree(ix->rows16);
      if (ix->mu) (void)hipFree(ix->mu);
      if (ix->graph) (void)hipFree(ix->graph);
      if (ix->seeds) (void)hipFree(ix->seeds);
      delete ix;
      throw;
    }
    ++ctx->live_children;
    *out_index = ix;
  });
}

int cvs_cagra_index_destroy(cvs_cagra_index* index) {
  return guarded([&] {
    if (!index) return;
    bind(index->ctx);
    (void)hipStreamSynchronize(index->ctx->stream);
    (void)hipFree(index->rows);
    (void)hipFree(index->rows16);
    (void)hipFree(index->mu);
    (void)hipFree(index->graph);
    if (index->seeds) (void)hipFree(index->seeds);
    --index->ctx->live_children;
    delete index;
  });
}

int cvs_cagra_index_edge_distances(cvs_context* ctx, const cvs_cagra_index* index, float* out_distances,
                                   int out_on_device) {
  return guarded([&] {
    bind(ctx);
    if (!index || index->ctx != ctx) fail(CVS_ERR_INVALID_ARGUMENT, "index does not belong to context");
    if (!out_distances) fail(CVS_ERR_INVALID_ARGUMENT, "null buffer");
    const size_t count = size_t(index->n) * index->degree;
    float* dst = out_distances;
    if (!out_on_device) {
      ctx->ws_io.reserve(count * sizeof(float));
      dst = ctx->ws_io.as<float>();
    }
    const TimerSpan t0 = timer_span(ctx, "cagra_edge_distances");
    auto kern = index->d > kBigDim ? edge_distances_kernel<true> : edge_distances_kernel<false>;
    hipExtLaunchKernelGGL(kern, dim3(unsigned(index->n)), dim3(256), 0, ctx->stream, t0.start,
                          t0.stop, 0, reinterpret_cast<const float4*>(index->rows), int(index->dpad / 4),
                          int(index->dpad / 64), static_cast<const uint32_t*>(index->graph), int(index->degree),
                          uint32_t(index->n), dst);
    after_launch("edge_distances_kernel");
    if (!out_on_device) {
      CVS_HIP(hipMemcpyAsync(out_distances, dst, count * sizeof(float), hipMemcpyDeviceToHost, ctx->stream));
      CVS_HIP(hipStreamSynchronize(ctx->stream));
    }
  });
}

int cvs_cagra_index_set_traversal(cvs_cagra_index* index, int bits) {
  return guarded([&] {
    if (!index) fail(CVS_ERR_INVALID_ARGUMENT, "null index");
    if (bits != 16 && bits != 32) fail(CVS_ERR_INVALID_ARGUMENT, "traversal precision must be 16 or 32 bits");
    index->traversal_bits = bits;
  });
}

int cvs_cagra_search_async(cvs_context* ctx, const cvs_cagra_index* index, const float* queries_dev,
                           int64_t q, int64_t k, uint32_t itopk_size, uint32_t search_width,
                           uint32_t max_iterations, uint32_t* out_neighbors_dev,
                           float* out_distances_dev, uint32_t* out_stats_dev) {
  return guarded([&] {
    bind(ctx);
    cagra_search_device(ctx, index, queries_dev, q, k, itopk_size, search_width, max_iterations,
                        out_neighbors_dev, out_distances_dev, out_stats_dev);
  });
}

int cvs_cagra_search_teams_async(cvs_context* ctx, const cvs_cagra_index* index, const float* queries_dev,
                                 int64_t q, int64_t k, uint32_t itopk_size, uint32_t search_width,
                                 uint32_t max_iterations, uint32_t teams, uint32_t* out_neighbors_dev,
                                 float* out_distances_dev) {
  return guarded([&] {
    bind(ctx);
    cagra_search_device(ctx, index, queries_dev, q, k, itopk_size, search_width, max_iterations,
                        out_neighbors_dev, out_distances_dev, nullptr, int(std::min<uint32_t>(teams, 1u << 20)));
  });
}

int cvs_cagra_search_record_async(cvs_context* ctx, const cvs_cagra_index* index, const float* queries_dev,
                                  int64_t q, int64_t k, uint32_t itopk_size, uint32_t search_width,
                                  uint32_t max_iterations, uint32_t* out_neighbors_dev, float* out_distances_dev,
                                  uint32_t* out_stats_dev, uint32_t* record_dev, uint32_t record_cap) {
  return guarded([&] {
    bind(ctx);
    if (!record_dev || record_cap == 0 || !out_stats_dev)
      fail(CVS_ERR_INVALID_ARGUMENT, "recording needs a record buffer, a positive capacity and stats");
    if (record_cap > (1u << 20)) fail(CVS_ERR_UNSUPPORTED, "record_cap above 2^20");
    cagra_search_device(ctx, index, queries_dev, q, k, itopk_size, search_width, max_iterations, out_neighbors_dev,
                        out_distances_dev, out_stats_dev, 1, record_dev, int(record_cap));
  });
}

int cvs_cagra_replay_gathers(cvs_context* ctx, const cvs_cagra_index* index, const uint32_t* record_dev,
                             uint32_t record_cap, const uint32_t* stats_dev, int64_t q, int bits, int reps,
                             double* out_ms) {
  return guarded([&] {
    bind(ctx);
    if (!index || index->ctx != ctx) fail(CVS_ERR_INVALID_ARGUMENT, "index does not belong to context");
    if (!record_dev || !stats_dev || !out_ms || record_cap == 0 || q <= 0 || reps < 1)
      fail(CVS_ERR_INVALID_ARGUMENT, "bad replay arguments");
    if (bits != 16 && bits != 32) fail(CVS_ERR_INVALID_ARGUMENT, "bits must be 16 or 32");
    if (q > int64_t(INT32_MAX)) fail(CVS_ERR_UNSUPPORTED, "too many queries");
    const int row_vecs = int(index->dpad * (bits / 8) / 16);
    const uint4* rows = bits == 16 ? static_cast<const uint4*>(index->rows16)
                                   : reinterpret_cast<const uint4*>(index->rows);
    void* sink = nullptr;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    auto cleanup = [&] {
      if (e0) (void)hipEventDestroy(e0);
      if (e1) (void)hipEventDestroy(e1);
      if (sink) (void)hipFree(sink);
    };
    try {
      CVS_HIP(hipMalloc(&sink, size_t(q) * 256 * sizeof(uint32_t)));
      CVS_HIP(hipEventCreate(&e0));
      CVS_HIP(hipEventCreate(&e1));
      auto launch = [&] {
        hipLaunchKernelGGL(gather_replay_kernel, dim3(unsigned(q)), dim3(256), 0, ctx->stream, rows, row_vecs,
                           record_dev, int(record_cap), stats_dev, static_cast<uint32_t*>(sink));
        after_launch("gather_replay_kernel");
      };
      launch();  // warm-up
      CVS_HIP(hipEventRecord(e0, ctx->stream));
      for (int i = 0; i < reps; ++i) launch();
      CVS_HIP(hipEventRecord(e1, ctx->stream));
      CVS_HIP(hipEventSynchronize(e1));
      float ms = 0.f;
      CVS_HIP(hipEventElapsedTime(&ms, e0, e1));
      *out_ms = double(ms) / reps;
    } catch (...) {
      cleanup();
      throw;
    }
    cleanup();
  });
}

int cvs_cagra_search_teams(cvs_context* ctx, const cvs_cagra_index* index, const float* queries, int64_t q,
                           int64_t k, uint32_t itopk_size, uint32_t search_width, uint32_t max_iterations,
                           uint32_t teams, uint32_t* out_neighbors, float* out_distances) {
  return guarded([&] {
    bind(ctx);
    if (!index || !queries || !out_neighbors || !out_distances) fail(CVS_ERR_INVALID_ARGUMENT, "null buffer");
    if (index->ctx != ctx) fail(CVS_ERR_INVALID_ARGUMENT, "index does not belong to context");
    if (q <= 0 || k <= 0) fail(CVS_ERR_INVALID_ARGUMENT, "query count and k must be positive");
    const size_t qbytes = size_t(q) * size_t(index->d) * sizeof(float);
    const size_t obytes = size_t(q) * size_t(k) * sizeof(float);
    host_call(ctx, queries, qbytes, out_neighbors, out_distances, obytes, [&](const float* dq, uint32_t* dn, float* dd) {
      cagra_search_device(ctx, index, dq, q, k, itopk_size, search_width, max_iterations, dn, dd, nullptr,
                          int(std::min<uint32_t>(teams, 1u << 20)));
    });
  });
}

int cvs_cagra_search(cvs_context* ctx, const cvs_cagra_index* index, const float* queries, int64_t q,
                     int64_t k, uint32_t itopk_size, uint32_t search_width, uint32_t max_iterations,
                     uint32_t* out_neighbors, float* out_distances) {
  return guarded([&] {
    bind(ctx);
    if (!index || !queries || !out_neighbors || !out_distances) fail(CVS_ERR_INVALID_ARGUMENT, "null buffer");
    if (index->ctx != ctx) fail(CVS_ERR_INVALID_ARGUMENT, "index does not belong to context");
    if (q <= 0 || k <= 0) fail(CVS_ERR_INVALID_ARGUMENT, "query count and k must be positive");
    const size_t qbytes = size_t(q) * size_t(index->d) * sizeof(float);
    const size_t obytes = size_t(q) * size_t(k) * sizeof(float);
    host_call(ctx, queries, qbytes, out_neighbors, out_distances, obytes, [&](const float* dq, uint32_t* dn, float* dd) {
      cagra_search_device(ctx, index, dq, q, k, itopk_size, search_width, max_iterations, dn, dd, nullptr);
    });
  });
}

}  // extern "C"
