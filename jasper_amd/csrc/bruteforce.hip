// bruteforce.hip -- exact k-NN by brute force on the matrix cores
// (the reference's ground-truth utility, python/jasper/__init__.py:828-926).
//
// Arithmetic as the reference computes it: L2 = (||q||^2 + ||v||^2) - 2 q.v in
// fp32, clamped at 0; IP = -(q.v) where the fp16 matmul's result is rounded to
// fp16 before the negation. q.v comes from v_mfma_f32_32x32x16_f16 (fp16
// products are exact in fp32, accumulation in fp32, K ascending on every path);
// the squared norms are fp32 sums, in element order for rows of up to 128 values
// and in the order of bf_long_sqnorm_kernel for longer ones. So a pair's
// distance is the same bits in every call. Ties are ordered by (distance, id).
//
// One-pass path, used for small bases (the line is in bruteforce_knn) and for
// queries that the rounds path leaves over:
// bf_scan_kernel: one wave owns 32 queries and one chunk of the base. It
// holds the A fragments of its queries in registers and walks the chunk 32
// vectors at a time (one 32x32 output tile, K over the padded dim), loading
// the next 32 vectors while the current ones are on the matrix cores. A
// score enters a per-query candidate buffer in LDS only if it beats the
// query's current k-th best; a buffer that could overflow in the next step
// is compacted (sorted, cut to k), which also lowers the threshold. At the
// end each (query, chunk) writes its best k, sorted. bf_merge_kernel: one
// wave per query merges the chunk lists. Rows longer than 32 K steps (512
// values, config 4's 960) take the same kernel with the query and base
// fragments read per slice of 8 K steps.
// The rounds path for larger bases is described before bf_tile_kernel.
#include "bruteforce.hpp"
#include "common.hpp"
#include "graph.hpp"
#include "mfma_gemm.hpp"

#include <algorithm>
#include <cfloat>
#include <cstdlib>
#include <stdexcept>
#include <type_traits>

namespace jasper_amd {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float float16v __attribute__((ext_vector_type(16)));

constexpr int kBfMaxK = 128;         // k the fused scan supports
constexpr int kBfStep = 32;          // vectors per step = most keys a query can gain per step
constexpr int kBfScratch = 256;      // compaction scratch: holds a full buffer (k + kBfStep <= 160)
constexpr uint32_t kBfMaxDp = 4096;  // longest padded row
constexpr int kBfSlice = 8;          // K steps per slice of the long-row scan (KS = 0)

__device__ uint4 kBfZeroChunk = {0u, 0u, 0u, 0u};  // never written

__device__ __forceinline__ half8 u4_as_h8(uint4 v) {
  half8 h;
  __builtin_memcpy(&h, &v, 16);
  return h;
}

// ||x||^2 per row, fp32 fma in element order. A block of 256 rows stages
// them 64 values at a time in LDS with coalesced loads (eight threads per
// 128-byte row segment), and each thread continues its own row's fma chain
// from there: the per-row order of the one-thread-per-row loop, with the
// memory access of a stream (the strided per-thread reads had run at about
// a sixth of the bandwidth). Row stride in LDS 136 bytes (34 words): at most
// two rows of a wave share a bank when they read the same column.
constexpr uint32_t kSqnRows = 256, kSqnChunk = 64, kSqnStride = kSqnChunk * 2 + 8;  // bytes
__global__ __launch_bounds__(kSqnRows) void row_sqnorm_kernel(const uint16_t* __restrict__ x, int64_t n,
                                                              uint32_t dp, uint32_t dim, float* __restrict__ out) {
  __shared__ __align__(16) uint8_t tile[kSqnRows * kSqnStride];  // 34,816 bytes
  const uint32_t t = threadIdx.x;
  const int64_t r0 = (int64_t)blockIdx.x * kSqnRows;
  const int64_t i = r0 + t;
  float s = 0.0f;
  for (uint32_t c0 = 0; c0 < dim; c0 += kSqnChunk) {
    // 256 rows x 8 segments of 16 bytes: each thread loads 8 of them
#pragma unroll
    for (uint32_t k = 0; k < 8; ++k) {
      const uint32_t e = k * kSqnRows + t;    // segment index in the tile
      const uint32_t rr = e >> 3, seg = e & 7u;
      const int64_t row = r0 + rr;
      const uint32_t col = c0 + seg * 8u;   // first value of the segment
      uint4 v = make_uint4(0u, 0u, 0u, 0u);
      if (row < n && col < dp) v = *reinterpret_cast<const uint4*>(x + (size_t)row * dp + col);
      uint2* dst = reinterpret_cast<uint2*>(tile + rr * kSqnStride + seg * 16u);  // 8-byte aligned
      dst[0] = make_uint2(v.x, v.y);
      dst[1] = make_uint2(v.z, v.w);
    }
    __syncthreads();
    const uint8_t* mine = tile + t * kSqnStride;
#pragma unroll
    for (uint32_t j = 0; j < kSqnChunk; ++j) {
      if (c0 + j < dim) {
        _Float16 hv;
        __builtin_memcpy(&hv, mine + 2u * j, 2);
        const float f = (float)hv;
        s = __builtin_fmaf(f, f, s);
      }
    }
    __syncthreads();
  }
  if (i < n) out[i] = s;
}

// ||x||^2 per row of more than 128 values, in the order that bf_tile_kernel sums
// it from its fragments: chunk c (8 values) to sum c mod 8, sums 2w and 2w + 1
// joined to part w, and the parts added from 0 to 3. Every path takes long rows'
// norms in this order, so that a pair's distance does not depend on the call it
// is computed in. Eight lanes per row, one per sum (128 contiguous bytes).
__global__ __launch_bounds__(256) void bf_long_sqnorm_kernel(const uint16_t* __restrict__ x, int64_t n, uint32_t dp,
                                                             float* __restrict__ out,
                                                             const uint32_t* __restrict__ wanted) {
  if (wanted && !*wanted) return;  // the norms are for queries left over, and there are none
  const int64_t row = (int64_t)blockIdx.x * 32 + (threadIdx.x >> 3);
  const uint32_t lane = threadIdx.x & 63u, j = lane & 7u;
  float s = 0.0f;
  if (row < n)
    for (uint32_t c = j; c < dp / 8; c += 8)
      s = gemm_sq_add(u4_as_h8(reinterpret_cast<const uint4*>(x + (size_t)row * dp)[c]), s);
  const float part = s + __shfl_xor(s, 1, 64);
  float sum = 0.0f;
#pragma unroll
  for (uint32_t w = 0; w < 4; ++w) sum += __shfl(part, (int)((lane & ~7u) + 2 * w), 64);
  if (row < n && j == 0) out[row] = sum;
}

// ||x||^2 of every row. wanted (long rows): nothing is computed if it is zero.
static void bf_sqnorms(const void* x, int64_t n, uint32_t dp, uint32_t dim, float* out, const uint32_t* wanted,
                       hipStream_t s) {
  if (dp > 128)
    hipLaunchKernelGGL(bf_long_sqnorm_kernel, dim3((uint32_t)((n + 31) / 32)), dim3(256), 0, s, (const uint16_t*)x, n,
                       dp, out, wanted);
  else
    hipLaunchKernelGGL(row_sqnorm_kernel, dim3((uint32_t)((n + kSqnRows - 1) / kSqnRows)), dim3(kSqnRows), 0, s,
                       (const uint16_t*)x, n, dp, dim, out);
  hip_check(hipGetLastError(), "launch row norms");
}

// Sort key: order-preserving distance bits (high) and id (low).
__device__ __forceinline__ uint64_t bf_key(float d, uint32_t id) { return ((uint64_t)dist_to_ord(d) << 32) | id; }

// Compact one query's buffer through the wave's kBfScratch-entry scratch:
// sort the cnt (<= kBfScratch) keys, keep min(cnt, k) in buf; returns that
// count and the k-th key (~0 when fewer than k remain). Wave-wide.
__device__ uint32_t bf_compact(uint64_t* buf, uint32_t cnt, uint32_t k, uint64_t* scratch, uint64_t* kth) {
  const uint32_t lane = lane_id();
  if (cnt <= 64) {
    // one key per lane, sorted in registers
    uint64_t x = lane < cnt ? buf[lane] : ~0ull;
    x = wave_bitonic_sort<64>(x);
    const uint32_t keep = min(cnt, k);
    const uint64_t kk = (uint64_t)__shfl((long long)x, (int)(k - 1), 64);
    if (lane < keep) buf[lane] = x;
    *kth = keep == k ? kk : ~0ull;
    lds_wave_sync();
    return keep;
  }
  const uint32_t N = pow2_ceil(cnt);
  for (uint32_t i = lane; i < N; i += 64) scratch[i] = i < cnt ? buf[i] : ~0ull;
  wave_sync();
  lds_bitonic_sort(scratch, N);
  const uint32_t keep = min(cnt, k);
  for (uint32_t i = lane; i < keep; i += 64) buf[i] = scratch[i];
  *kth = keep == k ? scratch[k - 1] : ~0ull;
  wave_sync();
  return keep;
}

template <int KS, int METRIC>
__global__ __launch_bounds__(64) void bf_scan_kernel(const uint16_t* __restrict__ base, int64_t n, uint32_t dp,
                                                     const uint16_t* __restrict__ queries, int64_t nq,
                                                     const float* __restrict__ vsq, const float* __restrict__ qsq,
                                                     uint32_t k, uint32_t cap, int64_t chunk, uint32_t n_chunks,
                                                     uint64_t* __restrict__ out /* [nq][n_chunks][k] */,
                                                     const uint8_t* __restrict__ tile_flags) {
  // cap >= k + kBfStep (a multiple of 8): candidate slots per query.
  // KS = 0: rows longer than 32 K steps; the query and base fragments are
  // read per slice of kBfSlice steps instead of held in registers.
  extern __shared__ uint64_t bf_lds[];
  uint64_t* cand = bf_lds;                 // [32][cap]
  uint64_t* scratch = bf_lds + 32 * cap;   // [kBfScratch]
  __shared__ uint32_t cnt[32];
  __shared__ uint64_t thr[32];
  const uint32_t lane = threadIdx.x;
  const int64_t q0 = (int64_t)blockIdx.x * 32;
  const uint32_t ci = blockIdx.y;
  const int64_t v_begin = (int64_t)ci * chunk;
  const int64_t v_end = min(n, v_begin + chunk);
  const uint32_t nck = dp / 8;  // 16-byte chunks per row
  if (tile_flags && !tile_flags[blockIdx.x]) return;  // only the flagged query tiles

  if (lane < 32) {
    cnt[lane] = 0;
    thr[lane] = ~0ull;
  }
  wave_sync();

  // A fragments: lane holds query q0 + (lane % 32), K slice 8 * (lane / 32).
  const uint32_t am = lane & 31u, ah = lane >> 5;
  const int64_t aq = q0 + am;
  constexpr int KR = KS > 0 ? KS : 1;  // K steps held in registers
  uint4 af[KR];
  if constexpr (KS > 0) {
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const uint32_t c = (uint32_t)s * 2 + ah;
      af[s] = (aq < nq && c < nck) ? reinterpret_cast<const uint4*>(queries + (size_t)aq * dp)[c]
                                   : make_uint4(0, 0, 0, 0);
    }
  }
  // long rows: this lane's query row (a row of zeros past nq)
  const uint4* qrow = aq < nq ? reinterpret_cast<const uint4*>(queries + (size_t)aq * dp) : nullptr;
  const uint32_t nks = (dp + 15) / 16;  // K steps (the last may be half empty)
  // the query rows of this lane's accumulators: m = 8g + 4*(lane/32) + j.
  // thd[r] is the distance of row r's current k-th key (+inf until known);
  // a score passes the cheap test d <= thd[r] and then the exact key test.
  float qs[16], thd[16];
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int64_t q = q0 + 8 * (r >> 2) + 4 * ah + (r & 3);
    qs[r] = (METRIC == kL2 && q < nq) ? qsq[q] : 0.0f;
    thd[r] = __builtin_inff();
  }

  // one 32-vector tile per step, double-buffered by hand so that a step's
  // MFMAs wait only for its own rows: the next tile's rows (and squared
  // norms) load while this one is on the matrix cores
  // a K slot past the row (dp % 16 == 8) reads the zero chunk: no per-lane
  // branch in the loop, and the product stays an exact 0 (the query side is
  // zero there too)
  auto load_step = [&](int64_t v0, uint4 (&nb)[KR], float& nvs) {
    const int64_t v = v0 + am;
    const int64_t vr = v < v_end ? v : v_begin;
    if constexpr (METRIC == kL2) nvs = vsq[vr];
    if constexpr (KS > 0) {
      const uint4* rv = reinterpret_cast<const uint4*>(base + (size_t)vr * dp);
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        const uint32_t c = (uint32_t)s * 2 + ah;
        nb[s] = *(c < nck ? rv + c : &kBfZeroChunk);
      }
    }
  };
  auto step = [&](int64_t v0, const uint4 (&cb)[KR], float vs) {
    float16v acc = {};
    if constexpr (KS > 0) {
#pragma unroll
      for (int s = 0; s < KS; ++s)
        acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(u4_as_h8(af[s]), u4_as_h8(cb[s]), acc, 0, 0, 0);
    } else {
      // K in slices: both fragments of a slice read together, then its
      // chain of kBfSlice matrix-core steps (the query rows stay in cache)
      const int64_t v = v0 + am;
      const uint4* rv = reinterpret_cast<const uint4*>(base + (size_t)(v < v_end ? v : v_begin) * dp);
      for (uint32_t s0 = 0; s0 < nks; s0 += kBfSlice) {
        uint4 a8[kBfSlice], b8[kBfSlice];
#pragma unroll
        for (int t = 0; t < kBfSlice; ++t) {
          const uint32_t c = (s0 + (uint32_t)t) * 2 + ah;
          a8[t] = qrow && c < nck ? qrow[c] : make_uint4(0u, 0u, 0u, 0u);
          b8[t] = *(c < nck ? rv + c : &kBfZeroChunk);
        }
#pragma unroll
        for (int t = 0; t < kBfSlice; ++t)
          acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(u4_as_h8(a8[t]), u4_as_h8(b8[t]), acc, 0, 0, 0);
      }
    }
    // lane holds column n = lane % 32 (vector) and rows 8g + 4*(lane/32) + j
    const int64_t v = v0 + am;
    if (v < v_end) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        float d;
        if constexpr (METRIC == kL2) {
          d = __builtin_fmaf(-2.0f, acc[r], qs[r] + vs);  // == (qs + vs) - 2 dot: 2 dot is exact
        } else {
          d = -__half2float(__float2half_rn(acc[r]));
        }
        if (d <= thd[r]) {
          if constexpr (METRIC == kL2) d = d < 0.0f ? 0.0f : d;
          const uint32_t m = 8u * (r >> 2) + 4u * ah + (r & 3);
          const uint64_t key = bf_key(d, (uint32_t)v);
          if (key < thr[m]) {
            const uint32_t slot = atomicAdd(&cnt[m], 1u);
            cand[m * cap + slot] = key;
          }
        }
      }
    }
    lds_wave_sync();
    // compact the buffers that could overflow in the next step (32 new keys at most)
    uint64_t full = ballot(lane < 32 && cnt[lane] > cap - kBfStep);
    if (full) {
      while (full) {
        const uint32_t m = (uint32_t)__builtin_ctzll(full);
        full &= full - 1;
        uint64_t kth;
        const uint32_t keep = bf_compact(cand + m * cap, cnt[m], k, scratch, &kth);
        if (lane == 0) {
          cnt[m] = keep;
          thr[m] = kth;
        }
        lds_wave_sync();
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const uint64_t t = thr[8u * (r >> 2) + 4u * ah + (r & 3)];
        thd[r] = t == ~0ull ? __builtin_inff() : ord_to_dist((uint32_t)(t >> 32));
      }
    }
  };
  // two tiles per iteration; tiles past v_end load a clamped row and add no
  // candidates (v < v_end fails), so the loop needs no mid-iteration exit
  uint4 ba[KR], bb[KR];
  float vsa = 0.0f, vsb = 0.0f;
  if (v_begin < v_end) load_step(v_begin, ba, vsa);
  for (int64_t v0 = v_begin; v0 < v_end; v0 += 64) {
    load_step(v0 + 32, bb, vsb);
    step(v0, ba, vsa);
    load_step(v0 + 64, ba, vsa);
    step(v0 + 32, bb, vsb);
  }
  // final: best k of each query, sorted, padded with ~0
  for (uint32_t m = 0; m < 32; ++m) {
    const int64_t q = q0 + m;
    if (q >= nq) break;
    uint64_t kth;
    const uint32_t keep = bf_compact(cand + m * cap, cnt[m], k, scratch, &kth);
    uint64_t* dst = out + ((size_t)q * n_chunks + ci) * k;
    for (uint32_t i = lane; i < k; i += 64) dst[i] = i < keep ? cand[m * cap + i] : ~0ull;
    wave_sync();
  }
}

// Merge the n_chunks sorted lists of one query (one wave per query).
__global__ __launch_bounds__(64) void bf_merge_kernel(const uint64_t* __restrict__ lists, int64_t nq,
                                                      uint32_t n_chunks, uint32_t k, int32_t* __restrict__ out_ids,
                                                      float* __restrict__ out_d, const uint8_t* __restrict__ q_flags) {
  __shared__ uint64_t buf[256];
  const int64_t q = blockIdx.x;
  if (q >= nq) return;
  if (q_flags && !q_flags[q]) return;
  const uint32_t lane = threadIdx.x;
  const uint64_t* src = lists + (size_t)q * n_chunks * k;
  const size_t total = (size_t)n_chunks * k;
  // running best: buf[0, k) sorted; fill buf[k, 256) with the next keys
  for (uint32_t i = lane; i < 256; i += 64) buf[i] = ~0ull;
  wave_sync();
  const uint32_t room = 256 - k;
  for (size_t off = 0; off < total; off += room) {
    for (uint32_t i = lane; i < room; i += 64) buf[k + i] = off + i < total ? src[off + i] : ~0ull;
    wave_sync();
    lds_bitonic_sort(buf, 256);
  }
  for (uint32_t i = lane; i < k; i += 64) {
    const uint64_t key = buf[i];
    out_ids[(size_t)q * k + i] = key == ~0ull ? -1 : (int32_t)(uint32_t)key;
    out_d[(size_t)q * k + i] = key == ~0ull ? FLT_MAX : ord_to_dist((uint32_t)(key >> 32));
  }
}

constexpr uint32_t kBfCandCap = 1024;  // keys a query's list holds between rounds
// The tests' cheap form reads ||v||^2 shrunk by 2^-20 (bf_tile_kernel).
constexpr float kBfVsShrink = 1.0f - 0x1p-20f;

// ------------------------------------------------------------ rounds path
// The base is scored in rounds over units of UNIT rows, in an order that spreads
// every round over the whole base: place i of the order is unit
// i * mul mod n_units, mul coprime to n_units. Round 0 (kBfFirst rows) writes
// every distance; after each round a trim kernel keeps a query's best k keys
// and its k-th distance T_q, and the next round, 4 or 16 times as many rows,
// appends only keys with d <= T_q: about k * (ratio - 1) of them.
// Rows stored cluster by cluster: until k rows of a query's cluster have been
// met, T_q is another cluster's and units of its own enter the list whole, up
// to more keys than it holds. The rounds then go on with the k best that it
// holds (T_q still bounds the true k-th distance, and later rounds tighten it),
// and such queries are scored once more over the whole base against their last
// T_q, which lists little more than k rows. Only work-groups that hold such a
// query run then; the others return at once. k = 100, rows in clusters: 1,000
// queries of 1M x 960 in clusters of 1,000 rows 50.6 -> 5.6 ms (in one pass ->
// once more; 3.7 ms shuffled), 10k of 1M x 128, 4,000 rows, 85 -> 6.6 ms (6.2).
constexpr uint32_t kBfFirst = 4096;  // rows of round 0
// A query's slots in the scratch: round 0's distances, then, once its trim has
// read them, the list in the first half.
constexpr uint32_t kBfListStride = kBfFirst / 2;
constexpr int64_t kBfBlock = 16384;  // queries scored together
static_assert(kBfListStride >= kBfCandCap, "the list fits in the distances' place");
static_assert(kBfBlock * kBfListStride < (1ll << 32), "list slots have 32-bit numbers");

struct BfOrder {
  uint32_t mul, n_units;
  __device__ __forceinline__ uint32_t at(uint32_t place) const { return (uint32_t)(((uint64_t)place * mul) % n_units); }
  // the unit `by` (< n_units) further in the base, cyclically; by = places * mul mod n_units
  __device__ __forceinline__ uint32_t on(uint32_t unit, uint32_t by) const {
    unit += by;
    return unit >= n_units ? unit - n_units : unit;
  }
  __device__ __forceinline__ uint32_t step(uint32_t places) const {  // places * mul mod n_units, few places
    uint32_t x = 0;
    for (uint32_t i = 0; i < places; ++i) x = on(x, mul);
    return x;
  }
};

enum BfQuery : uint8_t { kBfDone, kBfLeftOver, kBfLost };  // kBfDone: or in work

// What the kernels know of the queries' states, in one piece of the scratch.
struct BfState {
  uint32_t* any;  // [2] is any query left over, has any lost keys
  uint8_t* tile;  // [ceil(nq / 32)] holds a query left over
  uint8_t* q;     // [nq] BfQuery
  __host__ __device__ BfState(uint32_t* a, int64_t nq)
      : any(a), tile(reinterpret_cast<uint8_t*>(a + 2)), q(tile + (nq + 31) / 32) {}
};

// A round's start: round 0 clears what its trim does not write; with nothing to
// score again, the work-group returns.
__device__ __forceinline__ bool bf_begin(uint32_t* any, int64_t nq, bool first, bool again) {
  if (first && blockIdx.x == 0) {
    const BfState state(any, nq);
    for (uint32_t i = threadIdx.x; i < (uint32_t)((nq + 31) / 32); i += blockDim.x) state.tile[i] = 0;
    if (threadIdx.x < 2) any[threadIdx.x] = 0;
  }
  return !again || any[1] != 0;
}

// The order's mul: near the golden ratio of the units, the coprime number whose
// ratio to them has the smallest largest partial quotient (any run of places
// then falls evenly over the base, and any run of units over the places).
static uint32_t bf_order_step(uint32_t n_units) {
  const uint32_t golden = (uint32_t)(0.6180339887 * n_units);
  uint32_t best = 1, worst = ~0u;
  for (uint32_t i = 0; i < 128 && worst > 3; ++i) {
    const uint32_t mul = i & 1u ? golden - (i + 1) / 2 : golden + i / 2;
    uint32_t a = n_units, b = mul, largest = 0;
    while (b != 0) {
      uint32_t quotient = a / b;
      const uint32_t rest = a % b;
      if (rest == 0 && b != 1) quotient = ~0u;  // not coprime
      if (rest == 0 && b == 1) --quotient;      // (.., q) is (.., q - 1, 1)
      largest = std::max(largest, quotient);
      a = b;
      b = rest;
    }
    if (largest < worst) {
      worst = largest;
      best = mul;
    }
  }
  return best;
}

// Work-group barrier for LDS alone: loads in flight (the next tile's) go on.
__device__ __forceinline__ void lds_block_sync() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// Rows of more than 128 values: units of a matrix tile's columns. With units of
// whole tiles (256 rows) nearly every query of a base in clusters loses keys.
constexpr uint32_t kBfTileUnit = 32;

// One round over the order's tiles [t0, t1) (of G::TN / 32 places) with the
// product loop of mfma_gemm.hpp: G::TM queries per work-group, n_ch
// work-groups per query block taking contiguous parts of the round. The work
// order is XCD-aware: work-groups are dealt to the 8 XCDs round-robin by id, so
// work-group p takes item p / 8 of XCD p % 8's share, and the query blocks of one
// part run on one XCD and share its L2's copy of the tiles. The base rows' squared
// norms are summed from the fragments the products read (v_dot2, in the
// shadow of the MFMAs, in the order of bf_long_sqnorm_kernel; the WAM waves that
// read the same fragments share the K steps), so the base is read once, without
// a pass of its own for the norms. dense: round 0, every distance to its own slot of
// dist [nq][kBfFirst] (NaN for rows past the base). again: the queries whose
// threshold is a number are scored again (none, most often).
// L2 scores first take a cheap conservative test: y = fl(2 q.v - vs') >= c_q,
// with vs' = fl(||v||^2 (1 - 2^-20)) and c_q <= (||q||^2 - T_q) - 2^-19
// (||q||^2 + |T_q|). Whenever the exact score d = fl(fl(||q||^2 + ||v||^2) -
// 2 q.v) satisfies d <= T_q, y passes: with u = 2^-24, d <= T_q gives 2 q.v -
// ||v||^2 >= ||q||^2 - T_q - (||q||^2 + ||v||^2 + 2 |T_q|) u for the same
// computed q.v and norms, and vs' leaves 14 u ||v||^2, c_q 32 u (||q||^2 +
// |T_q|) of room. Only a 32 x 32 block in which some lane's test passes
// computes exact scores, and of its 16 rows per lane those that passed.
template <class G>
struct BfTileLds {
  static constexpr uint32_t kLocal = 11;  // keys staged per query
  // after the loop's buffers, per query: staged keys, norm, threshold, the
  // cheap test's bound, a count; then the norms' parts. 256 x 256: 161,792
  // of 163,840 bytes
  static constexpr size_t bytes = G::kLds + (size_t)G::TM * (8 * kLocal + 4 * 4) + (size_t)4 * G::TN * 4;
};

template <class G, int METRIC>
__global__ __launch_bounds__(G::kThreads, 2) void bf_tile_kernel(
    const uint16_t* __restrict__ base, int64_t n, uint32_t dp, const uint16_t* __restrict__ queries, int64_t nq,
    const float* __restrict__ qsq, const float* __restrict__ qthr, uint32_t t0, uint32_t t1, BfOrder order,
    uint32_t n_ch, uint32_t qblocks, float* __restrict__ dense, uint32_t* __restrict__ qcount,
    uint64_t* __restrict__ qcand, uint32_t* __restrict__ any, bool again) {
  if (!bf_begin(any, nq, dense != nullptr, again)) return;
  // K step j's squares go to part j mod 4 of the norm: the waves that share a
  // column take one step of each slice (four waves) or every other slice (two)
  static_assert((G::KC == 8 && G::WAM == 4) || (G::KC == 4 && G::WAM == 2), "every K step is some wave's");
  constexpr int kParts = 4 / G::WAM;  // of a wave
  extern __shared__ uint4 bf_tile_lds[];
  constexpr uint32_t kLocal = BfTileLds<G>::kLocal;
  char* lds = reinterpret_cast<char*>(bf_tile_lds);
  uint64_t* lbuf = reinterpret_cast<uint64_t*>(lds + G::kLds);         // [TM][kLocal]
  float* sqs = reinterpret_cast<float*>(lbuf + (size_t)G::TM * kLocal);  // [TM] query norms
  float* sth = sqs + G::TM;                                              // [TM] thresholds
  float* scr = sth + G::TM;                                              // [TM] the cheap test's c_q
  uint32_t* lcnt = reinterpret_cast<uint32_t*>(scr + G::TM);             // [TM]
  float* part = reinterpret_cast<float*>(lcnt + G::TM);                  // [4][TN] parts of the rows' norms
  const uint32_t W = gridDim.x, p = blockIdx.x, xcd = p & 7u, per = W >> 3, extra = W & 7u;
  const uint32_t L = xcd * per + min(xcd, extra) + (p >> 3);
  const uint32_t qblock = L % qblocks, ch = L / qblocks;
  // part ch of the round: its tiles differ by at most one between parts
  const uint32_t total = t1 - t0, each = total / n_ch, more = total % n_ch;
  const uint32_t first = t0 + ch * each + min(ch, more), count = each + (ch < more ? 1u : 0u);
  const int64_t qbase = (int64_t)qblock * G::TM;
  bool wanted = false;
  for (uint32_t r = threadIdx.x; r < (uint32_t)G::TM; r += G::kThreads) {
    const int64_t q = qbase + r;
    // a NaN threshold passes nothing (rows past the last query)
    const float qn = (METRIC == kL2 && q < nq) ? qsq[q] : 0.0f;
    const float th = q >= nq ? __builtin_nanf("") : dense ? __builtin_inff() : qthr[q];
    sqs[r] = qn;
    sth[r] = th;
    wanted = wanted || th == th;
    // IP: fp16(q.v) >= -T_q needs q.v >= -T_q less half an fp16 step; a whole
    // step (or the subnormal step) here.
    const double t = (double)th;
    const double c = METRIC == kL2 ? ((double)qn - t) - ((double)qn + fabs(t)) * 0x1p-19
                                   : -t - fabs(t) * 0x1p-10 - 0x1p-24;
    scr[r] = (float)(c - fabs(c) * 0x1p-22);
    lcnt[r] = 0u;
  }
  if (!__syncthreads_or(wanted)) return;
  const uint32_t lane = threadIdx.x & 63u, wave = uniform(threadIdx.x >> 6), am = lane & 31u, ah = lane >> 5;
  const uint32_t wm = wave % G::WAM, wn = wave / G::WAM;
  float vs[kParts][G::WTN];  // this lane's parts of its columns' squared norms
#pragma unroll
  for (int e = 0; e < kParts; ++e)
#pragma unroll
    for (int b = 0; b < G::WTN; ++b) vs[e][b] = 0.0f;
  // the units being loaded (load j of this wave lies in one) and, by column
  // blocks, being tested
  constexpr uint32_t kUnits = G::TN / kBfTileUnit;
  const uint32_t tile_step = order.step(kUnits);
  const uint32_t unit0 = order.at(first * kUnits);
  uint32_t next[G::kLoadsB], here = order.on(unit0, order.step(wn * G::WTN));
#pragma unroll
  for (int j = 0; j < G::kLoadsB; ++j) next[j] = order.on(unit0, order.step(G::load_row(j, wave) / kBfTileUnit));
  // a place's rows; past the base for places beyond the last
  auto unit_row = [&](uint32_t unit, uint32_t place) {
    return (int64_t)(place < order.n_units ? unit : order.n_units) * kBfTileUnit;
  };
  gemm_walk<G>(
      lds, queries, dp / 8, qbase, nq - 1, base, dp / 8, n - 1, dp / 8, &kBfZeroChunk, count,
      [&](uint32_t t, int j, uint32_t r) {
        const int64_t row = unit_row(next[j], (first + t) * kUnits + r / kBfTileUnit) + r % kBfTileUnit;
        next[j] = order.on(next[j], tile_step);
        return row;
      },
      [&](uint32_t k, int step, const gemm_half8 (&y)[G::WTN]) {
        if (METRIC == kL2 && (G::WAM == 4 ? (uint32_t)step : k & 1u) == wm) {
          float(&part_vs)[G::WTN] = vs[G::WAM == 4 ? 0 : step];
#pragma unroll
          for (int b = 0; b < G::WTN; ++b) part_vs[b] = gemm_sq_add(y[b], part_vs[b]);
        }
      },
      [&](uint32_t t, const gemm_acc (&acc)[G::WTM][G::WTN]) {
        uint32_t unit = here;
        const uint32_t place = (first + t) * kUnits + wn * G::WTN;
        int64_t v0[G::WTN];
#pragma unroll
        for (int b = 0; b < G::WTN; ++b) {
          v0[b] = unit_row(unit, place + b);
          unit = order.on(unit, order.mul);
        }
        here = order.on(here, tile_step);
        float vn[G::WTN];
#pragma unroll
        for (int b = 0; b < G::WTN; ++b) vn[b] = 0.0f;
        if constexpr (METRIC == kL2) {
          // the last tile's readers are past the barriers of this tile's slices
#pragma unroll
          for (int e = 0; e < kParts; ++e)
#pragma unroll
            for (int b = 0; b < G::WTN; ++b) {
              const float x = vs[e][b] + __shfl_xor(vs[e][b], 32, 64);
              if (ah == 0) part[(wm * kParts + e) * G::TN + wn * G::WTN * 32 + 32 * b + am] = x;
              vs[e][b] = 0.0f;
            }
          lds_block_sync();
#pragma unroll
          for (int b = 0; b < G::WTN; ++b)
#pragma unroll
            for (int w = 0; w < 4; ++w) vn[b] += part[w * G::TN + wn * G::WTN * 32 + 32 * b + am];
        }
#pragma unroll
        for (int a = 0; a < G::WTM; ++a) {
          // rows r0 + 8g + j of this lane; opaque, or the compiler reads every
          // row's values once for the whole walk and spills
          uint32_t r0 = wm * G::WTM * 32 + 32 * a + 4 * ah;
          asm volatile("" : "+v"(r0));
          float cq[16];
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            const float4 c4 = *reinterpret_cast<const float4*>(scr + r0 + 8 * g);
            cq[4 * g] = c4.x, cq[4 * g + 1] = c4.y, cq[4 * g + 2] = c4.z, cq[4 * g + 3] = c4.w;
          }
#pragma unroll
          for (int b = 0; b < G::WTN; ++b) {
            const float vsm = vn[b] * kBfVsShrink;
            uint64_t any = 0;  // lanes with a passing score
#pragma unroll
            for (int i = 0; i < 16; ++i) {
              const float y = METRIC == kL2 ? __builtin_fmaf(2.0f, acc[a][b][i], -vsm) : acc[a][b][i];
              any |= ballot(y >= cq[i]);
            }
            if (any == 0 && !dense) continue;
            const int64_t v = v0[b] + am;
            uint32_t re = r0;
            asm volatile("" : "+v"(re));
#pragma unroll
            for (int i = 0; i < 16; ++i) {
              const float y = METRIC == kL2 ? __builtin_fmaf(2.0f, acc[a][b][i], -vsm) : acc[a][b][i];
              if (!dense && ballot(y >= cq[i]) == 0) continue;
              const uint32_t r = re + 8 * (i >> 2) + (i & 3);
              float d;
              if constexpr (METRIC == kL2) d = __builtin_fmaf(-2.0f, acc[a][b][i], sqs[r] + vn[b]);
              else d = -__half2float(__float2half_rn(acc[a][b][i]));
              const bool pass = v < n && d <= sth[r];
              if constexpr (METRIC == kL2) d = d < 0.0f ? 0.0f : d;
              if (dense) {
                const int64_t q = qbase + r;
                if (q < nq)
                  dense[(size_t)q * kBfFirst + (first + t) * G::TN + wn * G::WTN * 32 + 32 * b + am] =
                      pass ? d : __builtin_nanf("");
              } else if (pass) {
                const uint64_t key = bf_key(d, (uint32_t)v);
                const uint32_t s = atomicAdd(&lcnt[r], 1u);
                if (s < kLocal) lbuf[(size_t)r * kLocal + s] = key;
                else {
                  // (inline: a call would save every accumulator around it)
                  const uint32_t q = (uint32_t)qbase + r;
                  const uint32_t at = atomicAdd(&qcount[q], 1u);
                  if (at < kBfCandCap) qcand[q * kBfListStride + at] = key;
                }
              }
            }
          }
        }
      });
  if (dense) return;
  // flush the staged keys: one reservation in the query's list
  __syncthreads();
  for (uint32_t r = threadIdx.x; r < (uint32_t)G::TM; r += G::kThreads) {
    const uint32_t c = min(lcnt[r], kLocal);
    if (qbase + r >= nq || c == 0) continue;
    const uint32_t at = atomicAdd(&qcount[qbase + r], c);
    for (uint32_t i = 0; i < c && at + i < kBfCandCap; ++i)
      qcand[(size_t)(qbase + r) * kBfListStride + at + i] = lbuf[(size_t)r * kLocal + i];
  }
}

// Rows of up to 128 values: the whole row fits registers, so a wave holds the
// fragments of 64 queries (64 VGPRs at 128 values) and only the base goes
// through LDS: 64-row tiles, loaded straight into it two tiles ahead of use
// (three buffers), each read by the block's four waves (2 x 2 MFMA tiles per
// wave: 64 bytes of LDS per cycle and CU at the matrix cores' rate, of 128).
// Two blocks per CU, so one's tests run beside the other's products.
// L2's cheap test costs 9 VALU instructions per 32 x 32 scores instead of 32:
// the products start from -c_q / 2 in place of zero and the largest of a
// lane's 16 sums is compared with ||v||^2 / 2. A block of scores that passes
// is multiplied again from zero for its exact sums (the
// scan's, bit for bit). The test's sums carry at most 136 roundings
// (8 chains of 16 products and the start) of at most (|c_q| + ||q||^2 +
// ||v||^2) / 2 each, the exact ones as many: with u = 2^-24, c_q <= ||q||^2 -
// T_q less 2048 u (||q||^2 + |T_q|) and ||v||^2 taken 1024 u smaller leave
// room for 2 * 136 u (|c_q| + ||q||^2 + ||v||^2) and the distance's own three.
// IP compares each sum with its bound (its error has no bound without norms).
// 10k x 1M x 128, k = 10, L2, the whole call: 4.71 ms with thresholds from a
// scan of 65,536 rows and 32 queries per wave, 3.3 ms this way (the last round
// 1,002 TFLOP/s); k = 100 by inner product at 96 values 40 -> 6.1 ms.
template <int KS>
struct BfStream {
  static constexpr int TM = 256, TN = 64, kWaves = 4, kThreads = 256, kBuffers = 3;
  static constexpr uint32_t kLocal = 11;                      // keys staged per query
  static constexpr int kLoads = (2 * KS + 3) / 4;             // per wave and tile: 1 KB each (nck = 2 KS or one less)
  static size_t bytes(uint32_t nck) {
    return (size_t)kBuffers * (TN * nck * 16 + TN * 4) + (size_t)TM * (8 * kLocal + 4 * 4);
  }
};

template <class G, int KS, int METRIC>
__global__ __launch_bounds__(256, 2) void bf_stream_kernel(
    const uint16_t* __restrict__ base, int64_t n, uint32_t dp, const uint16_t* __restrict__ queries, int64_t nq,
    const float* __restrict__ qsq, const float* __restrict__ vsq, const float* __restrict__ qthr, uint32_t t0,
    uint32_t t1, BfOrder order, uint32_t n_ch, uint32_t qblocks, float* __restrict__ dense,
    uint32_t* __restrict__ qcount, uint64_t* __restrict__ qcand, uint32_t* __restrict__ any, bool again) {
  if (!bf_begin(any, nq, dense != nullptr, again)) return;
  extern __shared__ uint4 bf_stream_lds[];
  constexpr uint32_t kLocal = G::kLocal;
  const uint32_t nck = dp / 8, tile_bytes = G::TN * nck * 16;
  char* rows = reinterpret_cast<char*>(bf_stream_lds);                                   // [3][TN][nck]
  float* norms = reinterpret_cast<float*>(rows + (size_t)G::kBuffers * tile_bytes);     // [3][TN]
  uint64_t* lbuf = reinterpret_cast<uint64_t*>(norms + G::kBuffers * G::TN);            // [TM][kLocal]
  float* sqs = reinterpret_cast<float*>(lbuf + (size_t)G::TM * kLocal);                 // [TM] query norms
  float* sth = sqs + G::TM;                                                             // [TM] thresholds
  float* scr = sth + G::TM;                                                             // [TM] the products' start
  uint32_t* lcnt = reinterpret_cast<uint32_t*>(scr + G::TM);                            // [TM]
  const uint32_t W = gridDim.x, p = blockIdx.x, xcd = p & 7u, per = W >> 3, extra = W & 7u;
  const uint32_t L = xcd * per + min(xcd, extra) + (p >> 3);
  const uint32_t qblock = L % qblocks, ch = L / qblocks;
  const uint32_t total = t1 - t0, each = total / n_ch, more = total % n_ch;
  const uint32_t first = t0 + ch * each + min(ch, more), count = each + (ch < more ? 1u : 0u);
  const int64_t qbase = (int64_t)qblock * G::TM;
  bool wanted = false;
  for (uint32_t r = threadIdx.x; r < (uint32_t)G::TM; r += G::kThreads) {
    const int64_t q = qbase + r;
    // a NaN threshold passes nothing (rows past the last query)
    const float qn = (METRIC == kL2 && q < nq) ? qsq[q] : 0.0f;
    const float th = q >= nq ? __builtin_nanf("") : dense ? __builtin_inff() : qthr[q];
    sqs[r] = qn;
    sth[r] = th;
    wanted = wanted || th == th;
    const double t = (double)th;
    if (METRIC == kL2) {
      const double c = ((double)qn - t) - ((double)qn + fabs(t)) * 0x1p-13;
      scr[r] = dense ? 0.0f : (float)(-0.5 * c);
    } else {
      const double c = -t - fabs(t) * 0x1p-10 - 0x1p-24;
      scr[r] = (float)(c - fabs(c) * 0x1p-22);
    }
    lcnt[r] = 0u;
  }
  if (!__syncthreads_or(wanted)) return;
  const uint32_t lane = threadIdx.x & 63u, wave = uniform(threadIdx.x >> 6), am = lane & 31u, ah = lane >> 5;
  // a row's chunk c sits at slot (c + f(r)) mod nck, which spreads eight
  // consecutive rows' equal chunks over the banks: row starts repeat every
  // 8 / g rows (mod 128 bytes), g = gcd(nck, 8)
  const uint32_t g8 = nck & (0u - nck), g = min(g8, 8u), gshift = 3u - (uint32_t)__builtin_ctz(g);
  auto turn = [&](uint32_t r) { return (r >> gshift) & (g - 1u); };
  uint32_t off[G::kLoads], lrow[G::kLoads];  // this lane's piece of load j: byte offset in a whole tile, row
#pragma unroll
  for (int j = 0; j < G::kLoads; ++j) {
    const uint32_t e = min((uint32_t)j * G::kWaves + wave, nck - 1u) * 64u + lane;  // (the last kilobyte again)
    const uint32_t r = e / nck, slot = e % nck, f = turn(r) % nck;
    const uint32_t c = slot >= f ? slot - f : slot + nck - f;
    lrow[j] = r;
    off[j] = (r * nck + c) * 16u;
  }
  auto issue = [&](uint32_t tile, uint32_t buf) {
    const int64_t v0 = (int64_t)tile * G::TN;
    const char* tb = reinterpret_cast<const char*>(base) + (size_t)v0 * nck * 16;
    const bool whole = v0 + G::TN <= n;
#pragma unroll
    for (int j = 0; j < G::kLoads; ++j) {
      uint32_t o = off[j];
      if (!whole && v0 + lrow[j] >= n) o -= (uint32_t)(v0 + lrow[j] - (n - 1)) * nck * 16u;  // the last row again
      const uint32_t kb = min((uint32_t)j * G::kWaves + wave, nck - 1u);
      gemm_load_lds16(tb + o, rows + (size_t)buf * tile_bytes + kb * 1024u);
    }
    if constexpr (METRIC == kL2)
      __builtin_amdgcn_global_load_lds((gemm_glb_void*)(vsq + min(v0 + (int64_t)lane, n - 1)),
                                       (gemm_lds_void*)(norms + buf * G::TN), 4, 0, 0);
  };
  half8 af[2][KS];
#pragma unroll
  for (int t = 0; t < 2; ++t) {
    const int64_t aq = qbase + 64 * wave + 32 * t + am;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const uint32_t c = (uint32_t)s * 2 + ah;
      af[t][s] = u4_as_h8((aq < nq && c < nck) ? reinterpret_cast<const uint4*>(queries + (size_t)aq * dp)[c]
                                               : make_uint4(0, 0, 0, 0));
    }
  }
  const uint32_t fr = turn(am) % nck, fr32 = turn(am + 32u) % nck;
  const bool odd = (nck & 1u) != 0;
  auto frag = [&](uint32_t buf, int u, int s) {
    const uint32_t f = u ? fr32 : fr;
    uint32_t slot = (uint32_t)s * 2 + ah + f;
    slot = slot >= nck ? slot - nck : slot;
    slot = slot >= nck ? 0u : slot;  // (the K slot past an odd row)
    half8 b = *reinterpret_cast<const half8*>(rows + (size_t)buf * tile_bytes + ((32u * u + am) * nck + slot) * 16u);
    if (s == KS - 1 && odd && ah) b = half8{};
    return b;
  };
  __syncthreads();
  float16v start[2];  // L2: -c_q / 2 of this lane's rows; IP: the bounds themselves
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int i = 0; i < 16; ++i) start[t][i] = scr[64 * wave + 32 * t + 8 * (i >> 2) + 4 * ah + (i & 3)];
  uint32_t next = order.at(first), here = next;
  uint32_t nb = 0, cb = 0;
  for (uint32_t k = 0; k < 2 && k < count; ++k) {
    issue(next, nb);
    next = order.on(next, order.mul);
    nb = nb == 2 ? 0 : nb + 1;
  }
  for (uint32_t it = 0; it < count; ++it) {
    // this tile's loads have landed (the next one's may be in flight), and
    // every wave is done with the buffer that the one after goes to
    constexpr int kInFlight = G::kLoads + (METRIC == kL2 ? 1 : 0);
    if (it + 1 < count) __builtin_amdgcn_s_waitcnt(kInFlight | 0x70);
    else __builtin_amdgcn_s_waitcnt(0x70);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (it + 2 < count) {
      issue(next, nb);
      next = order.on(next, order.mul);
      nb = nb == 2 ? 0 : nb + 1;
    }
    float16v acc[2][2];
    half8 b[2][2];
#pragma unroll
    for (int u = 0; u < 2; ++u) b[0][u] = frag(cb, u, 0);
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      if (s + 1 < KS) {
#pragma unroll
        for (int u = 0; u < 2; ++u) b[(s + 1) & 1][u] = frag(cb, u, s + 1);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int u = 0; u < 2; ++u)
          acc[t][u] = __builtin_amdgcn_mfma_f32_32x32x16_f16(
              af[t][s], b[s & 1][u], s ? acc[t][u] : METRIC == kL2 ? start[t] : float16v{}, 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int64_t v = (int64_t)here * G::TN + 32 * u + am;
      const float vn = METRIC == kL2 ? norms[cb * G::TN + 32 * u + am] : 0.0f;
      const float half = 0.5f * (vn * (1.0f - 0x1p-14f));
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        bool hit;
        if constexpr (METRIC == kL2) {
          float m = acc[t][u][0];
#pragma unroll
          for (int i = 1; i < 16; ++i) m = fmaxf(m, acc[t][u][i]);
          hit = m >= half;
        } else {
          hit = false;
#pragma unroll
          for (int i = 0; i < 16; ++i) hit = hit || acc[t][u][i] >= start[t][i];
        }
        if (ballot(hit) == 0 && !dense) continue;
        float16v sum = {};
        if constexpr (METRIC == kL2) {
#pragma unroll
          for (int s = 0; s < KS; ++s)
            sum = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[t][s], frag(cb, u, s), sum, 0, 0, 0);
        } else {
          sum = acc[t][u];
        }
        // rows r0 + 8g + j of this lane; opaque, or the compiler forms every
        // row's addresses once for the whole walk and spills
        uint32_t r0 = 64 * wave + 32 * t + 4 * ah;
        asm volatile("" : "+v"(r0));
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          // most of a passing block's 16 rows have no passing score
          if (!dense && ballot(METRIC == kL2 ? acc[t][u][i] >= half : acc[t][u][i] >= start[t][i]) == 0) continue;
          const uint32_t r = r0 + 8 * (i >> 2) + (i & 3);
          float d;
          if constexpr (METRIC == kL2) d = __builtin_fmaf(-2.0f, sum[i], sqs[r] + vn);
          else d = -__half2float(__float2half_rn(sum[i]));
          const bool pass = v < n && d <= sth[r];
          if constexpr (METRIC == kL2) d = d < 0.0f ? 0.0f : d;
          if (dense) {
            const int64_t q = qbase + r;
            if (q < nq)
              dense[(size_t)q * kBfFirst + (first + it) * G::TN + 32 * u + am] = pass ? d : __builtin_nanf("");
          } else if (pass) {
            const uint64_t key = bf_key(d, (uint32_t)v);
            const uint32_t s = atomicAdd(&lcnt[r], 1u);
            if (s < kLocal) lbuf[(size_t)r * kLocal + s] = key;
            else {
              const uint32_t q = (uint32_t)qbase + r;
              const uint32_t at = atomicAdd(&qcount[q], 1u);
              if (at < kBfCandCap) qcand[q * kBfListStride + at] = key;
            }
          }
        }
      }
    }
    here = order.on(here, order.mul);
    cb = cb == 2 ? 0 : cb + 1;
  }
  if (dense) return;
  // flush the staged keys: one reservation in the query's list
  __syncthreads();
  for (uint32_t r = threadIdx.x; r < (uint32_t)G::TM; r += G::kThreads) {
    const uint32_t c = min(lcnt[r], kLocal);
    if (qbase + r >= nq || c == 0) continue;
    const uint32_t at = atomicAdd(&qcount[qbase + r], c);
    for (uint32_t i = 0; i < c && at + i < kBfCandCap; ++i)
      qcand[(size_t)(qbase + r) * kBfListStride + at + i] = lbuf[(size_t)r * kLocal + i];
  }
}

// After a round, a work-group per query: finds the query's k-th key and keeps
// the k smallest in the list (in any order), their k-th distance as the
// threshold. The k-th is found by bits, from the top: a key's word takes a 0
// where at least k keys are then no larger (keys in registers, 16 per lane);
// the id word only where the k-th distance ties. That needs no sort of the
// list (1,024 keys sorted through LDS by a wave took 216 us for 10k queries);
// only the last round sorts, and only k keys. Four waves for round 0's 4,096
// keys: with 64 per lane the unrolled code ran once per wave from a cold
// instruction cache (272 us for 10k queries).
// A list that overflowed marks its query as having lost keys; the last round
// leaves such a query its threshold and an empty list, and after it is scored
// again, STAGE kBfAgain takes its results. One that overflows even then (ties),
// or with fewer than k keys of finite distance (infinite or NaN rows), is
// flagged for the one-pass kernels, and a NaN threshold keeps later rounds from
// appending to it.
// STAGE kBfDense: the keys are round 0's distances and the ids those of the
// order's first places, of UNIT rows.
enum BfStage { kBfDense, kBfRound, kBfLast, kBfAgain };
constexpr int kBfTrimRows = kBfCandCap / 64;  // keys per lane

template <BfStage STAGE, uint32_t UNIT>
__global__ __launch_bounds__(STAGE == kBfDense ? 256 : 64) void bf_trim_kernel(
    uint64_t* qcand, BfOrder order, uint32_t* __restrict__ qcount, uint32_t k, BfState state,
    float* __restrict__ qthr, int32_t* __restrict__ out_ids, float* __restrict__ out_d) {
  constexpr bool DENSE = STAGE == kBfDense;
  constexpr int kWaves = DENSE ? 4 : 1;
  static_assert(!DENSE || kBfFirst == 64 * kBfTrimRows * kWaves, "round 0 fills the registers");
  static_assert(UNIT == 32 || UNIT == 64, "a lane's slots are 64 apart");
  if (STAGE == kBfAgain && !state.any[1]) return;
  __shared__ uint64_t best[128];
  __shared__ uint32_t red[2][4];
  __shared__ uint32_t taken;
  const int64_t q = blockIdx.x;
  const uint32_t lane = threadIdx.x & 63u, wave = uniform(threadIdx.x >> 6);
  const uint8_t was = DENSE ? (uint8_t)kBfDone : state.q[q];
  if (was == kBfLeftOver || (STAGE == kBfAgain && was != kBfLost)) return;
  const uint32_t cnt = DENSE ? kBfFirst : uniform(qcount[q]);
  uint64_t* list = qcand + (size_t)q * kBfListStride;
  const float* dense = reinterpret_cast<const float*>(list);  // (read whole before the list is written)
  uint32_t hi[kBfTrimRows], lo[kBfTrimRows];  // empty slots and NaN: all ones
  const uint32_t rows = DENSE ? (uint32_t)kBfTrimRows : min((cnt + 63u) / 64u, (uint32_t)kBfTrimRows);
  // DENSE: slots 64 (wave kBfTrimRows + j) + lane, UNIT to a place
  uint32_t unit = DENSE ? order.at(wave * (uint32_t)kBfTrimRows * (64u / UNIT)) : 0u;
  const uint32_t step = DENSE ? order.step(64u / UNIT) : 0u;
#pragma unroll
  for (int j = 0; j < kBfTrimRows; ++j) {
    hi[j] = lo[j] = ~0u;
    if constexpr (DENSE) {
      const float d = dense[(wave * kBfTrimRows + (uint32_t)j) * 64u + lane];
      lo[j] = (lane < UNIT ? unit : order.on(unit, order.mul)) * UNIT + lane % UNIT;
      unit = order.on(unit, step);
      if (d == d) hi[j] = dist_to_ord(d);
    } else if ((uint32_t)j < rows && (uint32_t)j * 64u + lane < cnt) {
      const uint64_t key = list[(uint32_t)j * 64u + lane];
      hi[j] = (uint32_t)(key >> 32);
      lo[j] = (uint32_t)key;
    }
  }
  uint32_t turn = 0;
  // f(a, b) over the work-group's values
  auto reduce = [&](uint32_t x, auto f) {
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) x = f(x, (uint32_t)__shfl_xor((int)x, m, 64));
    if constexpr (kWaves > 1) {
      if (lane == 0) red[turn][wave] = x;
      __syncthreads();
      x = f(f(red[turn][0], red[turn][1]), f(red[turn][2], red[turn][3]));
      turn ^= 1u;
    }
    return uniform(x);
  };
  auto add = [](uint32_t a, uint32_t b) { return a + b; };
  auto larger = [](uint32_t a, uint32_t b) { return max(a, b); };
  auto smaller = [](uint32_t a, uint32_t b) { return min(a, b); };
  auto count_to = [&](uint32_t top) {  // keys whose distance word is at most top
    uint32_t c = 0;
#pragma unroll
    for (int j = 0; j < kBfTrimRows; ++j)
      if ((uint32_t)j < rows) c += hi[j] <= top ? 1u : 0u;
    return reduce(c, add);
  };
  // the k-th smallest distance word: below the bits that all words share
  // (most of a float's top bits), and only until a word has exactly k below it
  uint32_t mn = ~0u, mx = 0u;
#pragma unroll
  for (int j = 0; j < kBfTrimRows; ++j) {
    mn = min(mn, hi[j]);
    if (hi[j] != ~0u) mx = max(mx, hi[j]);
  }
  mn = reduce(mn, smaller);
  mx = reduce(mx, larger);
  uint32_t v = ~0u, below = 0;  // below: keys smaller than v
  bool exact = false;           // no key beyond the k-th ties with it
  if (mn != ~0u && count_to(mx) >= k) {
    int bit = mn == mx ? -1 : 31 - __builtin_clz(mn ^ mx);
    v = bit < 0 ? mn : mn & ~((2u << bit) - 1u);
    for (; bit >= 0; --bit) {
      const uint32_t top = v | ((1u << bit) - 1u);  // the largest word with a 0 here
      const uint32_t c = count_to(top);
      if (c == k) {
        uint32_t x = 0;
#pragma unroll
        for (int j = 0; j < kBfTrimRows; ++j)
          if (hi[j] <= top) x = max(x, hi[j]);
        v = reduce(x, larger);
        exact = true;
        break;
      }
      if (c < k) {
        v |= 1u << bit;
        below = c;
      }
    }
  }
  const float t = ord_to_dist(v);
  const bool over = cnt > 64u * kBfTrimRows * kWaves;
  if ((over && STAGE == kBfAgain) || v == ~0u || !(fabsf(t) < __builtin_inff())) {
    if (threadIdx.x == 0) {
      state.q[q] = kBfLeftOver;
      state.tile[q >> 5] = 1;
      state.any[0] = 1;
      qthr[q] = __builtin_nanf("");
    }
    return;
  }
  if (DENSE && threadIdx.x == 0) state.q[q] = kBfDone;
  if (over && threadIdx.x == 0) {
    state.q[q] = kBfLost;
    state.any[1] = 1;
  }
  if (STAGE == kBfLast) {
    const bool again = over || was == kBfLost;
    if (threadIdx.x == 0) {
      qthr[q] = again ? t : __builtin_nanf("");
      qcount[q] = 0;
    }
    if (again) return;
  }
  // ties at it: the smallest k - below ids
  uint32_t w = ~0u;
  if (!exact && count_to(v) > k) {
    w = 0;
    for (int bit = 31; bit >= 0; --bit) {
      const uint32_t top = w | ((1u << bit) - 1u);
      uint32_t c = 0;
#pragma unroll
      for (int j = 0; j < kBfTrimRows; ++j) c += hi[j] == v && lo[j] <= top ? 1u : 0u;
      if (below + reduce(c, add) < k) w |= 1u << bit;
    }
  }
  if (threadIdx.x == 0) taken = 0;
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kBfTrimRows; ++j) {
    if (hi[j] < v || (hi[j] == v && lo[j] <= w)) {
      const uint64_t key = ((uint64_t)hi[j] << 32) | lo[j];
      const uint32_t at = atomicAdd(&taken, 1u);  // exactly k in all
      if (STAGE == kBfLast || STAGE == kBfAgain) best[at] = key;
      else list[at] = key;
    }
  }
  if (STAGE == kBfDense || STAGE == kBfRound) {  // (round 0 is never the last)
    if (threadIdx.x == 0) {
      qcount[q] = k;
      qthr[q] = t;
    }
    return;
  }
  if (STAGE == kBfAgain && threadIdx.x == 0) state.q[q] = kBfDone;
  const uint32_t N = max(pow2_ceil(k), 2u);
  for (uint32_t i = k + lane; i < N; i += 64u) best[i] = ~0ull;
  wave_sync();
  lds_bitonic_sort(best, N);
  for (uint32_t i = lane; i < k; i += 64) {
    out_ids[(size_t)q * k + i] = (int32_t)(uint32_t)best[i];
    out_d[(size_t)q * k + i] = ord_to_dist((uint32_t)(best[i] >> 32));
  }
}

// How the one-pass path cuts the base.
struct BfChunks {
  int64_t chunk;      // rows
  uint32_t n_chunks;
  size_t list_bytes;  // of the chunks' results

  BfChunks(int64_t n, int64_t nq, uint32_t k) {
    // chunks: each a multiple of 64 vectors (a whole number of 32-vector steps)
    // about 2,048 work-groups (single waves): longer chunks spend fewer of
    // their steps filling and compacting the buffers before the threshold
    // settles (65,536 x 128 rows, 10k queries: 8,192 work-groups took 0.80 ms
    // longer, 4,096 0.18, 1,024 0.33);
    // JASPER_BF_SCAN_WGS overrides it (tuning)
    static const int64_t target = [] {
      const char* e = std::getenv("JASPER_BF_SCAN_WGS");
      return e ? std::max<int64_t>(1, std::atoll(e)) : 2048;
    }();
    int64_t want = std::max<int64_t>(1, target / ((nq + 31) / 32));
    want = std::min<int64_t>(want, (n + 63) / 64);
    chunk = ((n + want - 1) / want + 63) / 64 * 64;
    n_chunks = (uint32_t)((n + chunk - 1) / chunk);
    list_bytes = (size_t)nq * n_chunks * k * 8;
  }
};

// The one-pass path (scan + merge) over base rows [0, n), for all queries or
// only the flagged ones. lists: BfChunks::list_bytes of scratch.
static void bf_one_pass(const void* base, int64_t n, uint32_t dp, const void* queries, int64_t nq, uint32_t k,
                        int metric, const float* vsq, const float* qsq, uint64_t* lists, int32_t* out_ids,
                        float* out_d, const uint8_t* tile_flags, const uint8_t* q_flags, hipStream_t s) {
  const uint32_t ks = (dp + 15) / 16;  // 16-wide K steps (the last may be half empty)
  const BfChunks cut(n, nq, k);
  const dim3 grid((uint32_t)((nq + 31) / 32), cut.n_chunks);
  // at least 64 slots: a buffer is compacted (a 64-key register sort, then
  // every row's threshold reloaded) once it holds more than cap - kBfStep
  // keys, so at k = 10 the 48 slots of k + kBfStep compacted each query
  // after every 6 or so new candidates; 64 allow 22 between compactions
  // and keep the 1,878 work-groups of 10k queries resident (18.4 KB of LDS
  // each): 65,536 x 128 rows 0.90 -> 0.77 ms
  const uint32_t cap = std::max<uint32_t>((k + kBfStep + 7u) & ~7u, 64u);
  const size_t lds = ((size_t)32 * cap + kBfScratch) * 8;
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, grid, dim3(64), lds, s, (const uint16_t*)base, n, dp, (const uint16_t*)queries, nq,
                       vsq, qsq, k, cap, cut.chunk, cut.n_chunks, lists, tile_flags);
  };
#define JA_BF_CASE(K)                                              \
  case K:                                                          \
    if (metric == kL2) go(bf_scan_kernel<K, kL2>);                 \
    else go(bf_scan_kernel<K, kIP>);                               \
    break;
  switch (ks > 32 ? 0u : ks) {
    JA_BF_CASE(0)
    JA_BF_CASE(1) JA_BF_CASE(2) JA_BF_CASE(3) JA_BF_CASE(4) JA_BF_CASE(5) JA_BF_CASE(6) JA_BF_CASE(7)
    JA_BF_CASE(8) JA_BF_CASE(9) JA_BF_CASE(10) JA_BF_CASE(11) JA_BF_CASE(12) JA_BF_CASE(13) JA_BF_CASE(14)
    JA_BF_CASE(15) JA_BF_CASE(16) JA_BF_CASE(17) JA_BF_CASE(18) JA_BF_CASE(19) JA_BF_CASE(20) JA_BF_CASE(21)
    JA_BF_CASE(22) JA_BF_CASE(23) JA_BF_CASE(24) JA_BF_CASE(25) JA_BF_CASE(26) JA_BF_CASE(27) JA_BF_CASE(28)
    JA_BF_CASE(29) JA_BF_CASE(30) JA_BF_CASE(31) JA_BF_CASE(32)
    default: throw std::invalid_argument("bruteforce_knn: unsupported dim");
  }
#undef JA_BF_CASE
  hip_check(hipGetLastError(), "launch bf_scan_kernel");
  hipLaunchKernelGGL(bf_merge_kernel, dim3((uint32_t)nq), dim3(64), 0, s, (const uint64_t*)lists, nq, cut.n_chunks, k,
                     out_ids, out_d, q_flags);
  hip_check(hipGetLastError(), "launch bf_merge_kernel");
}

// Scratch of the rounds path, one allocation (with eight, back-to-back calls of
// 300 queries and 65,536 x 128 rows, k = 1, took 254 us each instead of 113, and
// the first of 10k queries and 1M rows 4.2 ms instead of 3.5): per query its
// distances' and list's slots, whose place the one-pass lists take after the
// last round; a count, a threshold, a norm and a state; then the base's norms.
struct BfScratch {
  uint64_t* qcand;
  float* vsq;
  uint32_t* qcount;
  float *qthr, *qsq;
  uint32_t* any;  // BfState

  // for blocks of `block` of nq queries
  static size_t slots(int64_t n, int64_t nq, int64_t block, uint32_t k) {
    size_t most = (size_t)block * kBfListStride * 8;
    for (int64_t part : {block, nq % block})
      if (part > 0) most = std::max(most, BfChunks(n, part, k).list_bytes);
    return most;
  }
  static size_t bytes(int64_t n, int64_t nq, int64_t block, uint32_t k, bool norms) {
    return slots(n, nq, block, k) + (norms ? (size_t)n * 4 : 0) + (size_t)block * (3 * 4 + 1) +
           (size_t)(block + 31) / 32 + 8;
  }
  BfScratch(void* mem, int64_t n, int64_t nq, int64_t block, uint32_t k, bool norms) {
    qcand = (uint64_t*)mem;
    vsq = (float*)((char*)mem + slots(n, nq, block, k));
    qcount = (uint32_t*)(vsq + (norms ? n : 0));
    qthr = (float*)(qcount + block);
    qsq = qthr + block;
    any = (uint32_t*)(qsq + block);
  }
};

// Scores the whole base in rounds and writes the results; the scratch's state
// names the queries that are left to the one-pass kernels. G: the tiles, of
// units of UNIT rows; round(parts, qblocks, t0, t1, order, dist, again):
// launches one round.
template <class G, uint32_t UNIT, class Round>
static void bf_rounds(int64_t n, int64_t nq, uint32_t k, const BfScratch& m, int32_t* out_ids, float* out_d,
                      hipStream_t s, Round round) {
  const uint32_t n_tiles = (uint32_t)((n + G::TN - 1) / G::TN);
  const uint32_t qblocks = (uint32_t)((nq + G::TM - 1) / G::TM);
  const uint32_t n_units = (uint32_t)((n + UNIT - 1) / UNIT);
  const BfOrder order{bf_order_step(n_units), n_units};
  // work-groups the chip holds at once: eight waves per CU (two per SIMD)
  constexpr uint32_t kResident = 256u * (8 / G::kWaves);
  constexpr uint32_t kFirstTiles = kBfFirst / G::TN;
  static_assert(kFirstTiles * G::TN == kBfFirst, "round 0 is whole tiles");
  auto score = [&](uint32_t t0, uint32_t t1, float* dist, bool again) {
    round(gemm_parts(qblocks, t1 - t0, kResident), qblocks, t0, t1, order, dist, again);
    hip_check(hipGetLastError(), "launch a brute-force round");
  };
  auto trim = [&](auto kern, uint32_t threads) {
    hipLaunchKernelGGL(kern, dim3((uint32_t)nq), dim3(threads), 0, s, m.qcand, order, m.qcount, k, BfState(m.any, nq), m.qthr,
                       out_ids, out_d);
    hip_check(hipGetLastError(), "launch bf_trim_kernel");
  };
  uint32_t t0 = 0, t1 = kFirstTiles;  // n >= 4 kBfFirst
  score(t0, t1, (float*)m.qcand, false);
  trim(bf_trim_kernel<kBfDense, UNIT>, 256);
  while (t1 < n_tiles) {
    // fourfold: about 3 k candidates per query and round, few where most rows
    // are. With few queries, where a round is mostly its launches, one step of
    // 16 (a list holds 16 k keys with room at k <= 32); with 10k queries it
    // cost 0.25 ms more in exact scores than the round it saves
    const uint64_t grow = k <= 32 && nq <= 1024 && (uint64_t)t1 * 64 <= n_tiles ? 16 : 4;
    t0 = t1;
    t1 = (uint32_t)std::min<uint64_t>(n_tiles, (uint64_t)t1 * grow);
    score(t0, t1, nullptr, false);
    if (t1 < n_tiles) trim(bf_trim_kernel<kBfRound, UNIT>, 64);
    else trim(bf_trim_kernel<kBfLast, UNIT>, 64);
  }
  score(0, n_tiles, nullptr, true);
  trim(bf_trim_kernel<kBfAgain, UNIT>, 64);
}

// The rounds path for one block of queries: the rounds, and the one-pass kernels
// for the queries they left over (none, in the ordinary case: they then end at
// once). The base's norms are computed (rows of up to 128 values) or there is
// space for them.
static void bf_in_rounds(const void* base, int64_t n, uint32_t dim, uint32_t dp, const void* queries, int64_t nq,
                         uint32_t k, int metric, const BfScratch& m, int32_t* out_ids, float* out_d, hipStream_t s) {
  const BfState state(m.any, nq);
  const uint16_t* base16 = (const uint16_t*)base;
  const uint16_t* queries16 = (const uint16_t*)queries;
  if (metric == kL2) bf_sqnorms(queries, nq, dp, dim, m.qsq, nullptr, s);
  if (dp <= 128) {
    auto go = [&](auto tag) {
      constexpr int KS = decltype(tag)::value;
      using G = BfStream<KS>;
      const size_t lds = G::bytes(dp / 8);
      auto kern = metric == kL2 ? bf_stream_kernel<G, KS, kL2> : bf_stream_kernel<G, KS, kIP>;
      if (lds > 64 * 1024)
        hip_check(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds), "LDS");
      bf_rounds<G, G::TN>(n, nq, k, m, out_ids, out_d, s,
                   [&](uint32_t parts, uint32_t qblocks, uint32_t t0, uint32_t t1, BfOrder order, float* dist, bool again) {
                     hipLaunchKernelGGL(kern, dim3(qblocks * parts), dim3(G::kThreads), lds, s, base16, n, dp,
                                        queries16, nq, (const float*)m.qsq, (const float*)m.vsq, (const float*)m.qthr,
                                        t0, t1, order, parts, qblocks, dist, m.qcount, m.qcand, m.any, again);
                   });
    };
    switch ((dp + 15) / 16) {
      case 1: go(std::integral_constant<int, 1>{}); break;
      case 2: go(std::integral_constant<int, 2>{}); break;
      case 3: go(std::integral_constant<int, 3>{}); break;
      case 4: go(std::integral_constant<int, 4>{}); break;
      case 5: go(std::integral_constant<int, 5>{}); break;
      case 6: go(std::integral_constant<int, 6>{}); break;
      case 7: go(std::integral_constant<int, 7>{}); break;
      default: go(std::integral_constant<int, 8>{}); break;
    }
  } else {
    auto go = [&](auto tile) {
      using G = decltype(tile);
      constexpr size_t lds = BfTileLds<G>::bytes;
      auto kern = metric == kL2 ? bf_tile_kernel<G, kL2> : bf_tile_kernel<G, kIP>;
      hip_check(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds), "LDS");
      bf_rounds<G, kBfTileUnit>(n, nq, k, m, out_ids, out_d, s,
                   [&](uint32_t parts, uint32_t qblocks, uint32_t t0, uint32_t t1, BfOrder order, float* dist, bool again) {
                     hipLaunchKernelGGL(kern, dim3(qblocks * parts), dim3(G::kThreads), lds, s, base16, n, dp,
                                        queries16, nq, (const float*)m.qsq, (const float*)m.qthr, t0, t1, order, parts,
                                        qblocks, dist, m.qcount, m.qcand, m.any, again);
                   });
    };
    // 256 queries per work-group at 991 TFLOP/s or 128 at 850 (mfma_gemm.hpp),
    // whichever finishes the padded queries first
    const uint64_t by256 = (uint64_t)((nq + 255) / 256) * 256 * 850, by128 = (uint64_t)((nq + 127) / 128) * 128 * 991;
    if (by256 <= by128) go(GemmTile<2, 4, 4, 2, 8>{});
    else go(GemmTile<2, 4, 2, 2, 4>{});
    if (metric == kL2) bf_sqnorms(base, n, dp, dim, m.vsq, m.any, s);  // if any query is left over
  }
  bf_one_pass(base, n, dp, queries, nq, k, metric, m.vsq, m.qsq, m.qcand, out_ids, out_d, state.tile,
              state.q, s);
}

void bruteforce_knn(const void* base, int64_t n, uint32_t dim, uint32_t dp, const void* queries, int64_t nq,
                    uint32_t k, int metric, int32_t* out_ids, float* out_d, hipStream_t s) {
  if (k == 0 || nq <= 0) return;
  if (k > (uint32_t)kBfMaxK) throw std::invalid_argument("bruteforce_knn supports k <= 128");
  if (dp % 8 != 0 || dp > kBfMaxDp) throw std::invalid_argument("bruteforce_knn supports padded dim <= 4096");
  if (n <= 0) throw std::invalid_argument("empty base");
  if (n > 0x7FFFFFFFll) throw std::invalid_argument("too many base vectors");
  if (nq > 0x7FFFFFFFll) throw std::invalid_argument("too many queries");
  // Rounds from 16,384 rows on (round 0 alone is 4,096). At small k, bases
  // that the one-pass kernels scan before the rounds' launches and trims are
  // done stay with them: below 65,536 rows of up to 128 values (20,000 x 128,
  // k = 1, 10k queries: 0.36 ms in one pass, 0.47 in rounds; 65,536 rows 0.77
  // and 0.60) and below 262,144 of up to 256 (100,000 x 136, k = 1, 7,000
  // queries: 0.63 and 0.75; 1M x 256, k = 10, 3,750: 5.1 and 3.4). Longer rows
  // (40,000 x 384, k = 10, 2,000 queries: 0.58 and 0.31) and larger k (50,000
  // x 64, k = 32: 3.1 and 0.8), where the scan's buffers are compacted ever
  // more often, do not; nor do they with one to a hundred queries (16,384 x
  // 128, k = 17, 1 query: 0.30 and 0.12; x 384, k = 1, 10 queries: 0.17 and
  // 0.13). At the lines, few queries: 65,536 x 128, k = 1, 300 queries 0.15 and
  // 0.14.
  // At k <= 2 the scan's buffers hardly ever fill, and it keeps two more ranges:
  // up to 64 queries of rows of more than 256 values, where a round leaves most
  // of its 128 query rows empty (x 960, k = 1, by inner product: 16,384 rows, one
  // query 66 us and 93, 50 queries 103 and 129; 65,536 rows, 30 queries 1%
  // apart; 131,072 rows, one query 3%), and 128 to 2,048 queries by inner
  // product of rows of up to 128, where there are no norms to share (131,072 x
  // 128, k = 1, 500 queries: 1.27 times as long in rounds; 262,144 rows 0.86
  // times, 100 queries 1.03, 5,000 0.68).
  int64_t scanned = k > 16 ? 0 : dp > 256 ? 0 : dp > 128 ? 262144 : 65536;
  if (k <= 2 && dp > 256 && nq <= 64) scanned = 98304 - 1024 * nq;
  if (k <= 2 && dp <= 128 && metric == kIP && nq >= 128 && nq <= 2048) scanned = 196608;
  if (n >= std::max<int64_t>(4 * (int64_t)kBfFirst, scanned)) {
    // 16 KB of scratch per query, 268 MB for a block of queries
    const int64_t block = std::min<int64_t>(nq, kBfBlock);
    void* scratch = nullptr;
    hip_check(hipMallocAsync(&scratch, BfScratch::bytes(n, nq, block, k, metric == kL2), s), "alloc round scratch");
    const BfScratch m(scratch, n, nq, block, k, metric == kL2);
    if (metric == kL2 && dp <= 128) bf_sqnorms(base, n, dp, dim, m.vsq, nullptr, s);
    for (int64_t q = 0; q < nq; q += block)
      bf_in_rounds(base, n, dim, dp, (const uint16_t*)queries + (size_t)q * dp, std::min(block, nq - q), k, metric, m,
                   out_ids + (size_t)q * k, out_d + (size_t)q * k, s);
    (void)hipFreeAsync(scratch, s);
    return;
  }
  const size_t list_bytes = BfChunks(n, nq, k).list_bytes;
  void* scratch = nullptr;
  hip_check(hipMallocAsync(&scratch, list_bytes + (metric == kL2 ? (size_t)(n + nq) * 4 : 0), s), "alloc chunk lists");
  float* vsq = metric == kL2 ? (float*)((char*)scratch + list_bytes) : nullptr;
  float* qsq = metric == kL2 ? vsq + n : nullptr;
  if (metric == kL2) {
    bf_sqnorms(base, n, dp, dim, vsq, nullptr, s);
    bf_sqnorms(queries, nq, dp, dim, qsq, nullptr, s);
  }
  bf_one_pass(base, n, dp, queries, nq, k, metric, vsq, qsq, (uint64_t*)scratch, out_ids, out_d, nullptr, nullptr, s);
  (void)hipFreeAsync(scratch, s);
}

}  // namespace jasper_amd
