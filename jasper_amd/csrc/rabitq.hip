// rabitq.hip -- one-bit RaBitQ codes (reference rabitq/quantize.cuh:144-383,
// rabitq/layout.cuh:43-143).
//
// At one bit per dimension the quantizer reduces to a closed form (the
// multi-bit code is clamped to 0, so t_const does not matter): with
// r = P^T x - P c, bit_i = [r_i >= 0] and two fp32 factors per vector
// (f_add, f_rescale). The rotation P^T x is a GEMM. All residuals of a vector
// stay in the registers of the four lanes that hold it; the factor sums are
// reduced across those lanes with two xor shuffles.
//
// fp16 rows (rabitq_split_kernel): x is exact in fp16, and each fp32 entry of
// P is the sum of three fp16 values (times its row's power of two), so the
// fp32 product runs as three v_mfma_f32_16x16x32_f16 chains at 16 times the
// fp32 matrix rate: every product is exact and the sums are fp32. An entry's
// 24 bits split exactly down to 2^-15 of its row's largest; of a smaller one
// less than 2^-39 of the largest is lost, under the sums' own rounding. Where a
// residual lies within the two products' rounding of zero (the bound is
// counted at rabitq_setup_kernel), its tile (16 coordinates of 16 vectors)
// takes the fp32 product instead, so the code bytes are that one's.
// fp32 rows (rabitq_kernel): v_mfma_f32_16x16x4_f32, one wave per 16 vectors:
// the MFMA's M side is 16 output coordinates, its N side 16 vectors, and the
// four K slots of each MFMA take coordinates k = 32b + 8q + s (q = lane/16,
// s = 0..7 across eight MFMAs), so each lane feeds the MFMA from one 32-byte
// run of its vector.
//
// Node layout (rabitq_data_store<float>): code bytes = ceil(dim/8) rounded
// up to 4, bits LSB-first, then f_add and f_rescale.
#include "common.hpp"
#include "graph.hpp"
#include "mfma_gemm.hpp"
#include "rabitq.hpp"

#include <cmath>
#include <limits>
#include <stdexcept>

namespace jasper_amd {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float float4v __attribute__((ext_vector_type(4)));

uint32_t rabitq_code_bytes(uint32_t dim) { return ((dim + 7u) / 8u + 3u) / 4u * 4u; }

// w_s of the bound below.
__device__ __forceinline__ float rabitq_weight(uint32_t steps, uint32_t s) { return (float)(64u * (steps - s) + 4u); }

// Scratch of one call, written by one launch of rabitq_setup_kernel: the
// rotated centroid rc[i] = sum_k P[i + k*dim] c[k] (P times c: the centroid
// goes through CUBLAS_OP_N, rotation.cuh:160-176; zero without a centroid and
// for i >= dim), and Pt[i][k] = P[k + i*dim], zero padded to [mp][kp]. For
// fp16 rows (split) also three fp16 parts [3][mp][kp] of Pt[i][k] * 2^s_i;
// inv[i] = 2^-s_i, where 2^s_i brings row i's largest entry to [2^14, 2^15);
// and tol[i], which times a vector's xw (rabitq_residuals) bounds the difference
// of the two products' sums i. An MFMA is taken to add its products one after
// the other in any order, each sum rounded to nearest. A sum rounded in K step s
// (32 coordinates) is at most A_s, the sum of |P_ik x_k| over the steps to s; the
// fp32 chain rounds 32 of them per step, and so does the fp16 chain of the
// first parts. The two others' sums are 2^-11 of it, so all their roundings
// count as less than one A, and so does what the split lost; the fp32 chain's
// rounded products and joining the two fp16 sums are one each:
//   u (sum_s 64 A_s + 4 A) = u sum_s w_s a_s,  w_s = 64 (steps - s) + 4,
// a_s = A_s - A_{s-1} <= |P_is| |x_s|, which by Cauchy-Schwarz is at most
// u sqrt(sum_s w_s |P_is|^2) sqrt(sum_s w_s |x_s|^2) = tol[i] xw, u = 2^-24 (1%
// on each factor for its own rounding). Rows whose largest entry is outside
// [2^-60, 2^60] are always taken from the fp32 product: nearer the ends of the
// exponent range its products underflow or its sums overflow.
// Block i < mp: row i. Block mp: the centroid.
__global__ __launch_bounds__(256) void rabitq_setup_kernel(const float* __restrict__ P, const float* __restrict__ c,
                                                           uint32_t dim, uint32_t mp, uint32_t kp, bool split,
                                                           float* __restrict__ rc, float* __restrict__ inv,
                                                           float* __restrict__ tol, float* __restrict__ pt,
                                                           _Float16* __restrict__ parts) {
  const uint32_t i = blockIdx.x, t = threadIdx.x;
  if (i == mp) {
    if (t >= mp) return;
    float acc = 0.0f;
    if (c && t < dim)
      for (uint32_t k = 0; k < dim; ++k) acc = __builtin_fmaf(P[(size_t)t + (size_t)k * dim], c[k], acc);
    rc[t] = acc;
    return;
  }
  const float v = i < dim && t < dim ? P[(size_t)t + (size_t)i * dim] : 0.0f;  // kp <= 256
  if (t < kp) pt[(size_t)i * kp + t] = v;
  if (!split) return;
  __shared__ uint32_t top[4];
  __shared__ float sq[4];
  uint32_t m = __builtin_bit_cast(uint32_t, fabsf(v));
#pragma unroll
  for (int x = 32; x >= 1; x >>= 1) m = max(m, (uint32_t)__shfl_xor((int)m, x, 64));
  if ((t & 63u) == 0) top[t >> 6] = m;
  __syncthreads();
  m = max(max(top[0], top[1]), max(top[2], top[3]));
  // the largest entry's exponent; rows of zeros, subnormals, infinities or
  // NaN are taken as they are
  const int e = (int)(m >> 23) - 127;
  const int sh = m >> 23 == 0 || m >> 23 == 255 ? 0 : 14 - e;
  const float w = __builtin_ldexpf(v, sh);
  float s2 = t < kp ? rabitq_weight(kp / 32, t / 32) * w * w : 0.0f;  // (w: no underflow at any scale)
#pragma unroll
  for (int x = 32; x >= 1; x >>= 1) s2 += __shfl_xor(s2, x, 64);
  if ((t & 63u) == 0) sq[t >> 6] = s2;
  const _Float16 p1 = (_Float16)w;
  const bool whole = fabsf((float)p1) < __builtin_inff();
  const float r1 = whole ? w - (float)p1 : 0.0f;  // exact
  const _Float16 p2 = (_Float16)r1;
  const _Float16 p3 = (_Float16)(r1 - (float)p2);
  if (t < kp) {
    const size_t at = (size_t)i * kp + t, part = (size_t)mp * kp;
    parts[at] = p1;
    parts[part + at] = p2;
    parts[2 * part + at] = p3;
  }
  __syncthreads();
  if (t == 0) {
    const float scale = __builtin_ldexpf(1.0f, -sh);
    inv[i] = scale;
    const bool ends = m != 0 && (e < -60 || e > 60);
    tol[i] = ends ? __builtin_inff() : 0x1p-24f * 1.01f * sqrtf((sq[0] + sq[1]) + (sq[2] + sq[3])) * scale;
  }
}

// The factors and the node of one vector, from the four lanes (q = 0..3) that
// hold its residuals r_i at i = 16t + 4q + j in res[t][j] (zero for i >= dim).
// rcv(t, j): the rotated centroid at i.
// |r_i| / ||r|| is rounded as the correctly rounded quotient: y = RN(1/||r||),
// then two residual corrections (five fp32 operations where the f64 division
// took about twenty; it was most of the kernel's time). The corrections are
// exact while nothing is near the exponent range's ends; a wave with a norm
// outside [2^-60, 2^60] (zero, infinite and NaN ones included) divides in f64.
template <int KT, class Rc>
__device__ __forceinline__ void rabitq_emit(float4v (&res)[KT], float l2, uint32_t dim, uint32_t q, Rc rcv, int metric,
                                            bool ok, uint32_t* __restrict__ node) {
  l2 += __shfl_xor(l2, 16, 64);
  l2 += __shfl_xor(l2, 32, 64);
  const float l2_norm = sqrt_rn(l2);
  const float y = (float)(1.0 / (double)l2_norm);
  const bool plain = ballot(!(l2_norm >= 0x1p-60f && l2_norm <= 0x1p60f)) == 0;
  float ipn = 0.0f, s_rx = 0.0f, s_cx = 0.0f, s_rc = 0.0f;
  constexpr int KW = (KT + 1) / 2;
  uint32_t word[KW];
#pragma unroll
  for (int w = 0; w < KW; ++w) word[w] = 0;
#pragma unroll
  for (int t = 0; t < KT; ++t) {
    const float4v cv = rcv(t);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t i = 16u * t + 4u * q + j;
      // only the last tile holds coordinates past dim (dim > 16 (KT - 1))
      if (t < KT - 1 || i < dim) {
        const float r = res[t][j];
        const float c = cv[j];
        float d;
        if (plain) {
          d = r * y;
          d = __builtin_fmaf(__builtin_fmaf(-d, l2_norm, r), y, d);
          d = __builtin_fmaf(__builtin_fmaf(-d, l2_norm, r), y, d);
        } else {
          d = div_rn(r, l2_norm);
        }
        ipn += 0.5f * fabsf(d);
        const bool bit = r >= 0.0f;
        const float xucb = bit ? 0.5f : -0.5f;
        s_rx = __builtin_fmaf(r, xucb, s_rx);
        s_cx = __builtin_fmaf(c, xucb, s_cx);
        s_rc = __builtin_fmaf(r, c, s_rc);
        word[t / 2] |= (bit ? 1u : 0u) << (16 * (t & 1) + j);
      }
    }
  }
#pragma unroll
  for (int m = 16; m <= 32; m <<= 1) {
    ipn += __shfl_xor(ipn, m, 64);
    s_rx += __shfl_xor(s_rx, m, 64);
    s_cx += __shfl_xor(s_cx, m, 64);
    s_rc += __shfl_xor(s_rc, m, 64);
  }
  float ipn_inv = div_rn(1.0f, ipn);
  if (isnan(ipn_inv)) ipn_inv = 1.0f;
  if (s_rx == 0.0f) s_rx = __builtin_inff();
  float f_add, f_rescale;
  if (metric == kL2) {
    f_add = l2 + div_rn(2.0f * l2 * s_cx, s_rx);
    f_rescale = ipn_inv * -2.0f * l2_norm;
  } else {
    f_add = (1.0f - s_rc) + div_rn(l2 * s_cx, s_rx);
    f_rescale = ipn_inv * -l2_norm;
  }
  // this lane's nibbles into their places (4q of each half word), then the
  // four lanes' together; lane q writes dwords q, q + 4, ... of the node
  uint32_t dw[KW + 2 + 3];
#pragma unroll
  for (int w = 0; w < KW; ++w) {
    uint32_t x = word[w] << (4 * q);
    x |= (uint32_t)__shfl_xor((int)x, 16, 64);
    x |= (uint32_t)__shfl_xor((int)x, 32, 64);
    dw[w] = x;
  }
  dw[KW] = __builtin_bit_cast(uint32_t, f_add);
  dw[KW + 1] = __builtin_bit_cast(uint32_t, f_rescale);
#pragma unroll
  for (int w = KW + 2; w < KW + 5; ++w) dw[w] = 0;
  uint32_t pick[4];
#pragma unroll
  for (uint32_t w = 0; w < 4; ++w) pick[w] = q == w ? ~0u : 0u;
  if (ok) {
#pragma unroll
    for (int w = 0; w < KW + 2; w += 4) {
      // (by masks: selects of array elements become an indexed array)
      const uint32_t x = (dw[w] & pick[0]) | (dw[w + 1] & pick[1]) | (dw[w + 2] & pick[2]) | (dw[w + 3] & pick[3]);
      if ((uint32_t)w + q < KW + 2) node[(uint32_t)w + q] = x;
    }
  }
}

// The values of the row chunk at coordinates k .. k + 7 that lie below dim;
// zeros past it, whatever a row's padding holds.
__device__ __forceinline__ uint4 keep_below(uint4 w, uint32_t k, uint32_t dim) {
  uint32_t ws[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
  for (uint32_t j = 0; j < 4; ++j) {
    if (k + 2 * j >= dim) ws[j] = 0;
    else if (k + 2 * j + 1 >= dim) ws[j] &= 0xFFFFu;
  }
  return make_uint4(ws[0], ws[1], ws[2], ws[3]);
}

// What the fp16-row kernels keep in LDS beside P, [mp] each.
struct RqTables {
  const float *rc, *inv, *tol;
};

// One tile of 16 vectors from the split product's sums to its residuals, in
// place; returns sum r^2 over this lane's coordinates. x2: this lane's part of
// sum_s w_s |x_s|^2. An output tile with a residual within its bound of zero is
// taken again from the fp32 product (about one in 50 at 128 dims, one in 17 at
// 256). Redoing the vectors' other output tiles with it cost more: 45 us of
// 1M x 128 when one in 130 was taken again.
template <int KT>
__device__ __forceinline__ float rabitq_residuals(float4v (&acc)[KT], float x2, const uint16_t* __restrict__ x, int64_t v,
                                                  int64_t n, uint32_t stride, uint32_t dim,
                                                  const float* __restrict__ pt, uint32_t col, uint32_t q,
                                                  const RqTables& tab) {
  constexpr uint32_t kp = 32 * ((KT + 1) / 2);
  x2 += __shfl_xor(x2, 16, 64);
  x2 += __shfl_xor(x2, 32, 64);
  const float xw = sqrtf(x2) * 1.01f;
  uint32_t q4 = 4 * q;
  asm volatile("" : "+v"(q4));  // opaque: or the tables are held in registers for all tiles
  uint32_t redo = 0;  // output tiles with a residual within its tolerance
#pragma unroll
  for (int t = 0; t < KT; ++t) {
    const float4v cv = *reinterpret_cast<const float4v*>(tab.rc + 16 * t + q4);
    const float4v iv = *reinterpret_cast<const float4v*>(tab.inv + 16 * t + q4);
    const float4v tv = *reinterpret_cast<const float4v*>(tab.tol + 16 * t + q4);
    bool near = false;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const bool in = t < KT - 1 || 16u * t + 4u * q + j < dim;
      // (the scaling is exact: one rounding, that of the subtraction)
      const float r = in ? __builtin_fmaf(acc[t][j], iv[j], -cv[j]) : 0.0f;
      near = near || (in && !(fabsf(r) > tv[j] * xw));  // NaN included
      acc[t][j] = r;
    }
    if (ballot(near && v < n)) redo |= 1u << t;
  }
  redo = uniform(redo);
  if (redo) {
    // the fp32 product of output tile t, the loads of up to HS K steps issued
    // together: they meet cold caches (1 to 2 us a round trip; Pt is another
    // XCD's write). One step after the other, 10,000 x 256 took 131 us, this way 78;
    // 1M x 256 1.54 -> 1.40 ms. More steps than that spill beside 64 sums.
    constexpr uint32_t KS = kp / 32, HS = KS <= 5 ? KS : 4;
    const uint16_t* row = x + (size_t)(v < n ? v : 0) * stride;
    do {
      const uint32_t t = (uint32_t)__builtin_ctz(redo);
      redo &= redo - 1u;
      const float4* pr = reinterpret_cast<const float4*>(pt + (size_t)(16 * t + col) * kp + 8 * q);
      float4v a = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (uint32_t s0 = 0; s0 < KS; s0 += HS) {
        uint4 w[HS];
        float4 p[2 * HS];
#pragma unroll
        for (uint32_t s = 0; s < HS && s0 + s < KS; ++s) {
          const uint32_t k = 32 * (s0 + s) + 8 * q;
          w[s] = *reinterpret_cast<const uint4*>(row + (k < dim ? k : 0u));
          p[2 * s] = pr[8 * (s0 + s)];
          p[2 * s + 1] = pr[8 * (s0 + s) + 1];
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (uint32_t s = 0; s < HS && s0 + s < KS; ++s) {
          const uint4 y = keep_below(w[s], 32 * (s0 + s) + 8 * q, dim);
          const float xv[8] = {h2f_lo(y.x), h2f_hi(y.x), h2f_lo(y.y), h2f_hi(y.y),
                               h2f_lo(y.z), h2f_hi(y.z), h2f_lo(y.w), h2f_hi(y.w)};
          const float pv[8] = {p[2 * s].x,     p[2 * s].y,     p[2 * s].z,     p[2 * s].w,
                               p[2 * s + 1].x, p[2 * s + 1].y, p[2 * s + 1].z, p[2 * s + 1].w};
#pragma unroll
          for (int e = 0; e < 8; ++e) a = __builtin_amdgcn_mfma_f32_16x16x4f32(pv[e], xv[e], a, 0, 0, 0);
        }
      }
      const float4v cv = *reinterpret_cast<const float4v*>(tab.rc + 16 * t + q4);
#pragma unroll
      for (int j = 0; j < 4; ++j) a[j] = 16u * t + 4u * q + j < dim ? a[j] - cv[j] : 0.0f;
#pragma unroll
      for (int u = 0; u < KT; ++u)
        if (t == (uint32_t)u) acc[u] = a;
    } while (redo);
  }
  float l2 = 0.0f;
#pragma unroll
  for (int t = 0; t < KT; ++t)
#pragma unroll
    for (int j = 0; j < 4; ++j) l2 = __builtin_fmaf(acc[t][j], acc[t][j], l2);
  return l2;
}

// KT = number of 16-wide output tiles (mp = 16 * KT <= 256). Three waves per SIMD
// where that takes at most 30 spilled registers (13 and 14 tiles): 1M x 200
// 2.11 -> 1.87 ms, x 224 2.32 -> 2.06, against two waves; 15 tiles would spill 41
// (2.45 -> 2.56), and 12 lose 11% at 1,000 rows.
template <int KT>
__global__ __launch_bounds__(256, KT == 13 || KT == 14 ? 3 : 2) void rabitq_kernel(
    const float* __restrict__ x, int64_t n, uint32_t stride, uint32_t dim, const float* __restrict__ pt, uint32_t kp,
    const float* __restrict__ rc, int metric, uint32_t* __restrict__ out) {
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t wave = threadIdx.x >> 6;
  const uint32_t col = lane & 15u;  // vector within the tile
  const uint32_t q = lane >> 4;     // K slot / output quarter
  constexpr uint32_t kNode = (KT + 1) / 2 + 2;  // dwords per node
  const int64_t tiles = (n + 15) / 16;
  for (int64_t tile = (int64_t)blockIdx.x * 4 + wave; tile < tiles; tile += (int64_t)gridDim.x * 4) {
    const int64_t v = tile * 16 + col;
    const bool ok = v < n;
    float4v acc[KT];
    const float* xr = x + (size_t)(ok ? v : 0) * stride;
#pragma unroll
    for (int t = 0; t < KT; ++t) acc[t] = {0.0f, 0.0f, 0.0f, 0.0f};
    for (uint32_t b = 0; b < kp; b += 32) {
      float xv[8];
      const uint32_t k = b + 8 * q;
#pragma unroll
      for (int j = 0; j < 8; ++j) xv[j] = (ok && k + j < dim) ? xr[k + j] : 0.0f;
#pragma unroll
      for (int t = 0; t < KT; ++t) {
        const float4* pr = reinterpret_cast<const float4*>(pt + (size_t)(16 * t + col) * kp + k);
        const float4 p0 = pr[0], p1 = pr[1];
        const float pv[8] = {p0.x, p0.y, p0.z, p0.w, p1.x, p1.y, p1.z, p1.w};
#pragma unroll
        for (int s = 0; s < 8; ++s) acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(pv[s], xv[s], acc[t], 0, 0, 0);
      }
    }
    // lane holds r_i for vector v at i = 16t + 4q + j
    float l2 = 0.0f;
#pragma unroll
    for (int t = 0; t < KT; ++t)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t i = 16u * t + 4u * q + j;
        const float r = i < dim ? acc[t][j] - rc[i] : 0.0f;
        acc[t][j] = r;
        l2 = __builtin_fmaf(r, r, l2);
      }
    rabitq_emit<KT>(
        acc, l2, dim, q, [&](int t) { return *reinterpret_cast<const float4v*>(rc + 16 * t + 4 * q); }, metric, ok,
        out + (size_t)v * kNode);
  }
}

// fp16 rows. A block stages the three parts of Pt in LDS once (rows one chunk
// past a multiple of 256 bytes, so that the 16 rows of a fragment fall on
// different banks) and its waves then walk tiles of 16 * NT vectors alone:
// each fragment of P read from LDS serves NT MFMAs (the small parts of P over
// all of K first, as the bound above counts them), and the next tile's rows
// load while this tile's factors are summed. LDS bounds NT = 1 (98 KB per 16
// vectors at 128 dims), so two where the registers hold them (KT <= 8: 128
// VGPRs of sums and rows).
// 1M x 128: 614 us (f32 MFMA, f64 divisions, byte stores) -> 221 us; 1M x 96:
// 378 -> 158 us, 1M x 160: 1.02 -> 0.36 ms.
template <int KT, int NT>
__global__ __launch_bounds__(512, 2) void rabitq_split_kernel(const uint16_t* __restrict__ x, int64_t n,
                                                              uint32_t stride, uint32_t dim,
                                                              const _Float16* __restrict__ parts,
                                                              const float* __restrict__ pt,
                                                              const float* __restrict__ tables, int metric,
                                                              uint32_t* __restrict__ out) {
  constexpr uint32_t KS = (KT + 1) / 2, kp = 32 * KS, mp = 16 * KT;
  constexpr uint32_t kRow = kp / 8 + 1;  // chunks per row of a part
  extern __shared__ uint4 rq_lds[];
  const uint4* pg = reinterpret_cast<const uint4*>(parts);
  float* tabl = reinterpret_cast<float*>(rq_lds + 3 * mp * kRow);  // rc, inv, tol
  const RqTables tab{tabl, tabl + mp, tabl + 2 * mp};
  for (uint32_t e = threadIdx.x; e < 3 * mp * (kp / 8); e += 512) rq_lds[(e / (kp / 8)) * kRow + e % (kp / 8)] = pg[e];
  for (uint32_t e = threadIdx.x; e < 3 * mp; e += 512) tabl[e] = tables[e];
  __syncthreads();
  const uint32_t lane = threadIdx.x & 63u, col = lane & 15u, q = lane >> 4;
  const int64_t tiles = (n + 16 * NT - 1) / (16 * NT);
  const int64_t step = (int64_t)gridDim.x * 8;
  int64_t tile = (int64_t)blockIdx.x * 8 + uniform(threadIdx.x >> 6);
  // lane: coordinates 32s + 8q .. + 7 of vector 16 u + col; zeros past the
  // row's dim, whatever the padding holds
  uint4 xf[NT][KS];
  auto load = [&](int64_t tl) {
#pragma unroll
    for (int u = 0; u < NT; ++u) {
      const int64_t v = tl * (16 * NT) + 16 * u + col;
#pragma unroll
      for (uint32_t s = 0; s < KS; ++s) {
        const uint32_t k = 32 * s + 8 * q;
        xf[u][s] = v < n && k < dim ? *reinterpret_cast<const uint4*>(x + (size_t)v * stride + k)
                                    : make_uint4(0, 0, 0, 0);
      }
    }
  };
  if (tile < tiles) load(tile);
  for (; tile < tiles; tile += step) {
    // opaque per tile: or the compiler reads every fragment of P, the same for
    // all tiles, before the loop, and spills them
    uint32_t frag = col * kRow + q;
    asm volatile("" : "+v"(frag));
    float4v acc[NT][KT];
#pragma unroll
    for (int u = 0; u < NT; ++u)
#pragma unroll
      for (int t = 0; t < KT; ++t) acc[u][t] = {0.0f, 0.0f, 0.0f, 0.0f};
    float x2[NT], l2[NT];
#pragma unroll
    for (int u = 0; u < NT; ++u) x2[u] = 0.0f;
#pragma unroll
    for (int u = 0; u < NT; ++u)
#pragma unroll
      for (uint32_t s = 0; s < KS; ++s) {
        // (stride >= 8-padded dim, so a chunk past dim's own is never read)
        if (s == KS - 1 && dim % 8 != 0) xf[u][s] = keep_below(xf[u][s], 32 * s + 8 * q, dim);
        half8 xh;
        __builtin_memcpy(&xh, &xf[u][s], 16);
        x2[u] = __builtin_fmaf(rabitq_weight(KS, s), gemm_sq_add(xh, 0.0f), x2[u]);
      }
    // the small parts' sums first, then the first parts' on top of them
#pragma unroll
    for (int first = 0; first < 2; ++first) {
#pragma unroll
      for (uint32_t s = 0; s < KS; ++s) {
#pragma unroll
        for (int t = 0; t < KT; ++t) {
#pragma unroll
          for (int part = first ? 0 : 2; part >= (first ? 0 : 1); --part) {
            const uint4 w = rq_lds[frag + ((uint32_t)part * mp + 16 * t) * kRow + 4 * s];
            half8 ph;
            __builtin_memcpy(&ph, &w, 16);
#pragma unroll
            for (int u = 0; u < NT; ++u) {
              half8 xh;
              __builtin_memcpy(&xh, &xf[u][s], 16);
              acc[u][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(ph, xh, acc[u][t], 0, 0, 0);
            }
          }
        }
      }
    }
#pragma unroll
    for (int u = 0; u < NT; ++u)
      l2[u] = rabitq_residuals<KT>(acc[u], x2[u], x, tile * (16 * NT) + 16 * u + col, n, stride, dim, pt, col, q, tab);
    if (tile + step < tiles) load(tile + step);
    uint32_t q4 = 4 * q;
    asm volatile("" : "+v"(q4));
#pragma unroll
    for (int u = 0; u < NT; ++u) {
      const int64_t v = tile * (16 * NT) + 16 * u + col;
      rabitq_emit<KT>(
          acc[u], l2[u], dim, q, [&](int t) { return *reinterpret_cast<const float4v*>(tab.rc + 16 * t + q4); }, metric,
          v < n, out + (size_t)v * (KS + 2));
    }
  }
}

// fp16 rows of more than 160 values: the parts of Pt exceed LDS, so a block
// stages them one K step of 32 at a time (3 * mp * 64 bytes, double-buffered,
// loaded straight into LDS) and its eight waves take the step together, each
// for its own 16 vectors, the first parts' sums beside the two others' (128 per
// lane at 256 values). Read through the caches instead, by each wave, 500k x 256
// took 1.7 times as long. 1M x 256: 2.24 ms on the f32 MFMA, 1.40 this way.
// Chunk q of row r sits at slot q ^ (r / 2 % 4) (mfma_gemm.hpp).
template <int KT>
__global__ __launch_bounds__(512, 2) void rabitq_split_long_kernel(const uint16_t* __restrict__ x, int64_t n,
                                                                   uint32_t stride, uint32_t dim,
                                                                   const _Float16* __restrict__ parts,
                                                                   const float* __restrict__ pt,
                                                                   const float* __restrict__ tables, int metric,
                                                                   uint32_t* __restrict__ out) {
  constexpr uint32_t KS = (KT + 1) / 2, kp = 32 * KS, mp = 16 * KT;
  constexpr uint32_t kLoads = 3 * KT;  // kilobytes per step
  __shared__ uint4 slice[2][3 * mp * 4];
  __shared__ __align__(16) float tabl[3 * mp];  // rc, inv, tol
  for (uint32_t e = threadIdx.x; e < 3 * mp; e += 512) tabl[e] = tables[e];
  const RqTables tab{tabl, tabl + mp, tabl + 2 * mp};
  const uint32_t lane = threadIdx.x & 63u, wave = uniform(threadIdx.x >> 6), col = lane & 15u, q = lane >> 4;
  auto issue = [&](uint32_t s, uint32_t buf) {
#pragma unroll
    for (uint32_t j = 0; j < (kLoads + 7) / 8; ++j) {
      const uint32_t kb = j * 8 + wave;  // 16 rows of 4 chunks
      if (kb < kLoads) {
        const uint32_t r = kb * 16 + (lane >> 2), c = (lane & 3u) ^ ((r >> 1) & 3u);
        gemm_load_lds16(parts + (size_t)r * kp + 32 * s + 8 * c, (char*)slice[buf] + kb * 1024);
      }
    }
  };
  const int64_t tiles = (n + 15) / 16;
  const int64_t turns = (tiles + (int64_t)gridDim.x * 8 - 1) / ((int64_t)gridDim.x * 8);  // the same for every wave
  auto row_chunk = [&](int64_t tl, uint32_t s) {
    const int64_t v = tl * 16 + col;
    const uint32_t k = 32 * s + 8 * q;
    uint4 w = make_uint4(0, 0, 0, 0);
    if (v < n && k < dim) w = *reinterpret_cast<const uint4*>(x + (size_t)v * stride + k);
    if (s == KS - 1 && dim % 8 != 0) w = keep_below(w, k, dim);
    return w;
  };
  issue(0, 0);
  uint32_t buf = 0;
  for (int64_t turn = 0; turn < turns; ++turn) {
    const int64_t tile = (turn * gridDim.x + blockIdx.x) * 8 + wave;  // past the last: no rows
    float4v acc[KT], low[KT];  // sums of the first parts, and of the two others
#pragma unroll
    for (int t = 0; t < KT; ++t) acc[t] = low[t] = {0.0f, 0.0f, 0.0f, 0.0f};
    float x2 = 0.0f;
    uint4 xn = row_chunk(tile, 0);
    for (uint32_t s = 0; s < KS; ++s) {
      half8 xh;
      __builtin_memcpy(&xh, &xn, 16);
      x2 = __builtin_fmaf(rabitq_weight(KS, s), gemm_sq_add(xh, 0.0f), x2);
      __builtin_amdgcn_s_waitcnt(0x70);  // vmcnt(0) lgkmcnt(0): this step's slice and rows are here
      __syncthreads();                   // and every wave is done with the other buffer
      if (s + 1 < KS) {
        issue(s + 1, buf ^ 1u);
        xn = row_chunk(tile, s + 1);
      } else if (turn + 1 < turns) {
        issue(0, buf ^ 1u);
      }
      const char* pl = (const char*)slice[buf] + col * 64 + ((q ^ ((col >> 1) & 3u)) * 16);
#pragma unroll
      for (int t = 0; t < KT; ++t) {
#pragma unroll
        for (int part = 2; part >= 0; --part) {  // smallest part first
          const half8 ph = *reinterpret_cast<const half8*>(pl + (part * mp + 16 * t) * 64);
          float4v& sum = part ? low[t] : acc[t];
          sum = __builtin_amdgcn_mfma_f32_16x16x32_f16(ph, xh, sum, 0, 0, 0);
        }
      }
      buf ^= 1u;
    }
    const int64_t v = tile * 16 + col;
#pragma unroll
    for (int t = 0; t < KT; ++t) acc[t] += low[t];
    const float l2 = rabitq_residuals<KT>(acc, x2, x, v, n, stride, dim, pt, col, q, tab);
    uint32_t q4 = 4 * q;
    asm volatile("" : "+v"(q4));
    rabitq_emit<KT>(
        acc, l2, dim, q, [&](int t) { return *reinterpret_cast<const float4v*>(tab.rc + 16 * t + q4); }, metric,
        v < n, out + (size_t)v * (KS + 2));
  }
}

void rabitq_quantize(const void* x, bool f16, int64_t n, uint32_t dim, uint32_t stride, const float* P,
                     const float* centroid, int metric, void* out, hipStream_t s) {
  if (dim == 0 || dim > 256) throw std::invalid_argument("rabitq_quantize supports 1 <= dim <= 256");
  if (stride < dim) throw std::invalid_argument("row stride below dim");
  if (f16 && (stride % 8 != 0 || ((uintptr_t)x & 15u) != 0))
    throw std::invalid_argument("fp16 rows must be 16-byte aligned with a stride that is a multiple of 8");
  if (n <= 0) return;
  const uint32_t kp = (dim + 31u) & ~31u, mp = (dim + 15u) & ~15u, kt = mp / 16;
  // one allocation: rc, inv and tol [mp], Pt, then its parts
  float* tables = nullptr;
  const size_t ptn = (size_t)mp * kp;
  hip_check(hipMallocAsync((void**)&tables, (size_t)3 * mp * 4 + ptn * (f16 ? 10 : 4), s), "alloc rabitq rotation");
  float* pt = tables + 3 * mp;  // 16-byte aligned: mp is a multiple of 16
  _Float16* parts = (_Float16*)(pt + ptn);
  hipLaunchKernelGGL(rabitq_setup_kernel, dim3(mp + 1), dim3(256), 0, s, P, centroid, dim, mp, kp, f16, tables,
                     tables + mp, tables + 2 * mp, pt, parts);
  hip_check(hipGetLastError(), "launch rabitq set-up");
  auto wide = [&](auto kern) {
    const int64_t tiles = (n + 15) / 16;
    const uint32_t grid = (uint32_t)std::min<int64_t>((tiles + 3) / 4, 16384);
    hipLaunchKernelGGL(kern, dim3(grid), dim3(256), 0, s, (const float*)x, n, stride, dim, (const float*)pt, kp,
                       (const float*)tables, metric, (uint32_t*)out);
  };
  auto split = [&](auto kern, int nt, size_t lds) {
    if (lds > 64 * 1024)
      hip_check(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds),
                "rabitq LDS");
    // one turn of resident blocks (two waves per SIMD are one block of eight)
    const int64_t tiles = (n + 16 * nt - 1) / (16 * nt);
    const uint32_t grid = (uint32_t)std::min<int64_t>((tiles + 7) / 8, 256);
    hipLaunchKernelGGL(kern, dim3(grid), dim3(512), lds, s, (const uint16_t*)x, n, stride, dim, (const _Float16*)parts,
                       (const float*)pt, (const float*)tables, metric, (uint32_t*)out);
  };
  const size_t staged = (size_t)3 * mp * (kp / 8 + 1) * 16 + (size_t)3 * mp * 4;
#define JA_RQ_CASE(K)                                                                   \
  case K:                                                                               \
    if (!f16) wide(rabitq_kernel<K>);                                                   \
    else if constexpr (K <= 10) split(rabitq_split_kernel<K, (K <= 8 ? 2 : 1)>, K <= 8 ? 2 : 1, staged); \
    else split(rabitq_split_long_kernel<K>, 1, 0);                                      \
    break;
  switch (kt) {
    JA_RQ_CASE(1) JA_RQ_CASE(2) JA_RQ_CASE(3) JA_RQ_CASE(4) JA_RQ_CASE(5) JA_RQ_CASE(6) JA_RQ_CASE(7)
    JA_RQ_CASE(8) JA_RQ_CASE(9) JA_RQ_CASE(10) JA_RQ_CASE(11) JA_RQ_CASE(12) JA_RQ_CASE(13) JA_RQ_CASE(14)
    JA_RQ_CASE(15) JA_RQ_CASE(16)
    default: throw std::invalid_argument("rabitq_quantize: unsupported dim");
  }
#undef JA_RQ_CASE
  hip_check(hipGetLastError(), "launch rabitq_kernel");
  (void)hipFreeAsync(tables, s);
}

}  // namespace jasper_amd
