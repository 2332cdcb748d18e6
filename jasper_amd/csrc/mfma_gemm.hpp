// mfma_gemm.hpp -- the main loop of products of fp16 rows on the matrix
// cores: C[i][j] = sum_k A[i][k] * B[j][k] in fp32, both operands rows of
// whole 16-byte chunks (K contiguous), used where the rows are long enough
// that K has to be read in slices (the ground truth's tile kernel, the
// rotation's GEMM).
//
// A work-group owns TM rows of A and walks tiles of TN rows of B. K runs in
// slices of KC chunks, both operands' slices loaded from global memory
// straight into LDS (no registers in between), double-buffered; the walk is
// one stream of slices over all tiles, so a tile's epilogue runs while the
// next tile's first slice loads. Each wave computes 32*WTM x 32*WTN of the
// tile with v_mfma_f32_32x32x16_f16, K ascending (the order of every other
// kernel that computes these products, so the sums are the same bits).
//
// What bounds it: per K step of 16 a wave reads WTM + WTN fragments (1 KB
// each) for WTM*WTN MFMAs of 32 cycles; at 2 x 4 that is 96 bytes per cycle
// and CU of the 128 that LDS gives. A step's fragments are read before the
// previous step's MFMAs are issued (the scheduling barriers): left alone the
// compiler reads each fragment right before its use and waits for it.
// Measured without an epilogue, 1024 x 262144 x 960: 991 TFLOP/s at WTM x WTN
// = 2 x 4, eight waves (256 x 256), KC = 8 (710 without the early reads); 850
// at 2 x 4, four waves (128 x 256), KC = 4; 805 at 2 x 2, four waves, KC = 8.
//
// LDS rows are KC*16 bytes, without padding because a wave's direct load
// fills 1 KB in lane order; instead chunk c of row r sits at slot c ^ f(r),
// f chosen so that 8 consecutive rows' equal chunks fall on different banks.
// The swizzle is applied to the global address each lane reads.
#pragma once

#include "common.hpp"

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace jasper_amd {

typedef _Float16 gemm_half8 __attribute__((ext_vector_type(8)));
typedef float gemm_acc __attribute__((ext_vector_type(16)));

template <int WTM_, int WTN_, int WAM_, int WAN_, int KC_>
struct GemmTile {
  static constexpr int WTM = WTM_, WTN = WTN_, WAM = WAM_, WAN = WAN_, KC = KC_;
  static constexpr int TM = 32 * WTM * WAM, TN = 32 * WTN * WAN, kWaves = WAM * WAN, kThreads = 64 * kWaves;
  static constexpr int kRowBytes = KC * 16, kBuf = (TM + TN) * kRowBytes;  // one slice of both operands
  static constexpr int kLoadsA = TM * kRowBytes / 1024 / kWaves, kLoadsB = TN * kRowBytes / 1024 / kWaves;
  static constexpr size_t kLds = 2 * (size_t)kBuf;
  static_assert(KC == 4 || KC == 8, "swizzles exist for slices of 4 and 8 chunks");
  static_assert(kLoadsA * 1024 * kWaves == TM * kRowBytes && kLoadsB * 1024 * kWaves == TN * kRowBytes,
                "every wave loads whole kilobytes of each operand");
  // load j of a wave fills kilobyte j * waves + wave of an operand's slice:
  // kRowsPerLoad rows from load_row on, lane l row l / KC, slot l % KC
  static constexpr uint32_t kRowsPerLoad = 64 / KC;
  static __device__ __forceinline__ uint32_t load_row(int j, uint32_t wave) {
    return ((uint32_t)j * kWaves + wave) * kRowsPerLoad;
  }
  static __device__ __forceinline__ uint32_t swizzle(uint32_t r) { return KC == 8 ? (r & 7u) : ((r >> 1) & 3u); }
};

typedef __attribute__((address_space(3))) void gemm_lds_void;
typedef __attribute__((address_space(1))) const void gemm_glb_void;

__device__ __forceinline__ void gemm_load_lds16(const void* g, void* l) {
  __builtin_amdgcn_global_load_lds((gemm_glb_void*)g, (gemm_lds_void*)l, 16, 0, 0);
}

// s plus the squares of 8 values (v_dot2: fp16 subnormals are kept)
__device__ __forceinline__ float gemm_sq_add(gemm_half8 h, float s) {
  typedef _Float16 half2v __attribute__((ext_vector_type(2)));
#pragma unroll
  for (int e = 0; e < 8; e += 2) {
    const half2v p = {h[e], h[e + 1]};
    s = __builtin_amdgcn_fdot2(p, p, s, false);
  }
  return s;
}

// How many parts to cut a walk of `tiles` tiles into, for `groups` rows of
// work-groups each: the count whose last turn of `resident` work-groups is
// fullest (a part's tiles set its turn's time).
inline uint32_t gemm_parts(uint32_t groups, uint32_t tiles, uint32_t resident) {
  uint32_t best = 1;
  uint64_t cost = ~0ull;
  for (uint32_t c = 1; c <= tiles; ++c) {
    const uint64_t turns = ((uint64_t)groups * c + resident - 1) / resident;
    if (turns > 4 && c > 1) break;
    const uint64_t x = turns * ((tiles + c - 1) / c);
    if (x < cost) {
      cost = x;
      best = c;
    }
  }
  return best;
}

// Walks tiles 0 .. n_tiles - 1. `a_row0` / `a_last`: the work-group's first
// row of A and the last valid one (rows past it read that row again);
// tile_row(t, j, r): the B row at row r of tile t, r the first of load j of this
// wave (whose rows follow each other); `b_last` as a_last. a_stride,
// b_stride: 16-byte chunks from row to row; nck: chunks multiplied. zero: 16
// bytes of zeros in global memory, read for chunks past the row in the last
// slice (both operands, so that no value is multiplied by a stray one).
// slice(k, s, y): called with the B fragments of each K step s of slice k;
// epi(t, acc): called with a tile's sums, lane l holding column l % 32 of B tile
// b and rows 8*(i/4) + 4*(l/32) + i%4 of A tile a in acc[a][b][i]. epi may use
// LDS outside [lds, lds + G::kLds).
template <class G, class TileRow, class Slice, class Epi>
__device__ __forceinline__ void gemm_walk(char* lds, const void* A, uint32_t a_stride, int64_t a_row0, int64_t a_last,
                                          const void* B, uint32_t b_stride, int64_t b_last, uint32_t nck,
                                          const void* zero, uint32_t n_tiles, TileRow tile_row, Slice slice, Epi epi) {
  if (n_tiles == 0) return;
  const uint32_t lane = threadIdx.x & 63u, wave = uniform(threadIdx.x >> 6);
  const uint32_t wm = wave % G::WAM, wn = wave / G::WAM;
  const uint32_t ns = (nck + G::KC - 1) / G::KC, rem = nck - (ns - 1) * G::KC;  // chunks in the last slice
  const uint32_t lr = lane / G::KC, slot = lane % G::KC;
  const char* pa[G::kLoadsA];
  const char* pb[G::kLoadsB];
  auto chunk_of = [&](uint32_t r) { return slot ^ G::swizzle(r); };
#pragma unroll
  for (int j = 0; j < G::kLoadsA; ++j) {
    const uint32_t r = G::load_row(j, wave) + lr;
    const int64_t row = min(a_row0 + (int64_t)r, a_last);
    pa[j] = (const char*)A + (size_t)row * a_stride * 16 + chunk_of(r) * 16;
  }
  auto set_tile = [&](uint32_t t) {
#pragma unroll
    for (int j = 0; j < G::kLoadsB; ++j) {
      const uint32_t r = G::load_row(j, wave) + lr;
      const int64_t row = min(tile_row(t, j, G::load_row(j, wave)) + (int64_t)lr, b_last);
      pb[j] = (const char*)B + (size_t)row * b_stride * 16 + chunk_of(r) * 16;
    }
  };
  auto issue = [&](uint32_t k, uint32_t buf) {
    char* la = lds + buf * G::kBuf + wave * 1024;
    char* lb = la + G::TM * G::kRowBytes;
    const size_t ko = (size_t)k * G::kRowBytes;
    if (k + 1 < ns || rem == G::KC) {
#pragma unroll
      for (int j = 0; j < G::kLoadsA; ++j) gemm_load_lds16(pa[j] + ko, la + j * G::kWaves * 1024);
#pragma unroll
      for (int j = 0; j < G::kLoadsB; ++j) gemm_load_lds16(pb[j] + ko, lb + j * G::kWaves * 1024);
    } else {
#pragma unroll
      for (int j = 0; j < G::kLoadsA; ++j) {
        const uint32_t r = G::load_row(j, wave) + lr;
        gemm_load_lds16(chunk_of(r) < rem ? (const void*)(pa[j] + ko) : zero, la + j * G::kWaves * 1024);
      }
#pragma unroll
      for (int j = 0; j < G::kLoadsB; ++j) {
        const uint32_t r = G::load_row(j, wave) + lr;
        gemm_load_lds16(chunk_of(r) < rem ? (const void*)(pb[j] + ko) : zero, lb + j * G::kWaves * 1024);
      }
    }
  };
  const uint32_t am = lane & 31u, ah = lane >> 5, fs = G::swizzle(am);
  gemm_acc acc[G::WTM][G::WTN];
  auto compute = [&](uint32_t k, uint32_t buf) {
    const char* la = lds + buf * G::kBuf + (wm * G::WTM * 32 + am) * G::kRowBytes;
    const char* lb = lds + buf * G::kBuf + (G::TM + wn * G::WTN * 32 + am) * G::kRowBytes;
    gemm_half8 x[2][G::WTM], y[2][G::WTN];
    auto read = [&](int s, gemm_half8 (&xx)[G::WTM], gemm_half8 (&yy)[G::WTN]) {
      const uint32_t o = (((uint32_t)s * 2 + ah) ^ fs) * 16;
#pragma unroll
      for (int a = 0; a < G::WTM; ++a) xx[a] = *reinterpret_cast<const gemm_half8*>(la + a * 32 * G::kRowBytes + o);
#pragma unroll
      for (int b = 0; b < G::WTN; ++b) yy[b] = *reinterpret_cast<const gemm_half8*>(lb + b * 32 * G::kRowBytes + o);
    };
    read(0, x[0], y[0]);
#pragma unroll
    for (int s = 0; s < G::KC / 2; ++s) {
      if (s + 1 < G::KC / 2) read(s + 1, x[(s + 1) & 1], y[(s + 1) & 1]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int a = 0; a < G::WTM; ++a)
#pragma unroll
        for (int b = 0; b < G::WTN; ++b)
          acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(x[s & 1][a], y[s & 1][b], acc[a][b], 0, 0, 0);
      slice(k, s, y[s & 1]);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  uint32_t buf = 0;
  set_tile(0);
  issue(0, 0);
  for (uint32_t t = 0; t < n_tiles; ++t) {
#pragma unroll
    for (int a = 0; a < G::WTM; ++a)
#pragma unroll
      for (int b = 0; b < G::WTN; ++b) acc[a][b] = gemm_acc{};
    for (uint32_t k = 0; k < ns; ++k) {
      // this slice's loads have landed, and every wave is done reading the
      // other buffer, which the next slice's loads may now overwrite
      __builtin_amdgcn_s_waitcnt(0x70);  // vmcnt(0) lgkmcnt(0)
      __syncthreads();
      if (k + 1 < ns) {
        issue(k + 1, buf ^ 1u);
      } else if (t + 1 < n_tiles) {
        set_tile(t + 1);
        issue(0, buf ^ 1u);
      }
      compute(k, buf);
      buf ^= 1u;
    }
    epi(t, acc);
  }
}

}  // namespace jasper_amd
