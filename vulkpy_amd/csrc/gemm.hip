// GEMM on CDNA4 matrix cores (F15 matmul, F16 Dense affine).
//
// The reference computes every output with one thread looping over K from
// global memory (vulkpy/shader/matmul.comp:23-33, batch_affine.comp:25-39).
// Here a block computes a BM x BN tile: operand slices are staged through LDS
// ahead of their use, and each wave owns a sub-tile of 32 x 32 or 16 x 16 MFMA
// blocks:
//   FP32    v_mfma_f32_32x32x2_f32, 16x16x4 for few outputs (operands as stored;
//           an FP32 MFMA adds its terms one after the other, each rounded once, as
//           fma does.  Three BF16 parts of an element on the BF16 matrix cores took
//           4.4 ms at 8192^3, 7.9 so, but those round their sums more coarsely: an
//           output of one nonzero term was up to 1.42 ulp off, 0.5 so)
//   BF16    v_mfma_f32_16x16x32_bf16  (operands rounded to nearest-even BF16)
//   BF16X3  the same instruction three times: lo*hi + hi*lo + hi*hi, where
//           x = hi + lo + O(2^-16 |x|) with hi = bf16(x), lo = bf16(x - hi)
// Accumulation is FP32 in every mode.  The epilogue applies alpha, beta*C,
// bias[n] and an activation, and can also emit a BF16 copy of the result.
// Blocks are remapped so that consecutive tiles land on the same XCD (each of
// the 8 XCDs has its own L2) and grouped along M for L2 reuse of B.
#include <type_traits>
#include <utility>

#include "common.h"
#include "fastdiv.h"

namespace vkh {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(16))) float f32x16_t;
// f(integral_constant<int, 0>), ..., f(integral_constant<int, N - 1>): a
// loop unrolled by construction
template <typename F, int... I>
__device__ __forceinline__ void static_for_seq(F& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  static_for_seq(f, std::make_integer_sequence<int, N>{});
}


typedef __attribute__((ext_vector_type(4))) float f32x4_t;
// the same in memory at any 4-byte alignment (global accesses of 16 bytes need
// no more on this hardware)
typedef __attribute__((ext_vector_type(4), aligned(4))) float f32x4u_t;

struct GemmArgs {
  const float* A;
  const float* B;
  float* C;
  const float* bias;
  uint16_t* Cbf;
  uint64_t M, N, K, lda, ldb, ldc;
  float alpha, beta;
  int act;
  const float* aux;  // activation output whose derivative multiplies the result
  uint64_t ldaux;
  int aux_act;
  int vec_c;  // C, bias, aux, Cbf rows allow 16-byte (Cbf: 8-byte) accesses
  uint32_t tiles_m, tiles_n;
  uint16_t* Cbft;  // C^T as BF16: Cbft[n * ldt + m] (optional)
  uint64_t ldt;
  // column sums of the final C over each chunk of CS_ROWS rows, in row order
  // from the chunk's first row: cs[(m / CS_ROWS) * N + n] (optional; waves
  // with 128-row slabs only)
  float* cs;
  int no_c;  // 1: the FP32 C is not stored (only Cbf / Cbft / cs)
  // the aux activation's output as BF16 instead of aux (ReLU' only: the BF16
  // copy has the sign, zero-ness and NaN-ness of the value)
  const uint16_t* aux16;
};
constexpr int CS_ROWS = 128;

// SIG = false: the caller has ruled out the sigmoid (whose FP64 exp is most
// of the code of an unrolled epilogue)
template <bool SIG = true>
__device__ __forceinline__ float act_apply(int act, float v) {
  if (act == VKH_ACT_RELU) return (v >= 0.0f || v != v) ? v : 0.0f;  // np.maximum(v, 0)
  if (SIG && act == VKH_ACT_SIGMOID) return 1.0f / (1.0f + (float)exp((double)(-v)));
  return v;
}

// dy * act'(y) given the activation's output y, in the op order of
// nn/layers.py:207-210 (ReLU) and 264-267 (Sigmoid)
__device__ __forceinline__ float act_deriv_mul(int act, float y, float dy) {
  if (act == VKH_ACT_RELU) {
    // max(sign(y), 0) (np.maximum keeps a NaN): 1 for y > 0, y itself for a
    // NaN, +0 otherwise
    const float d = y > 0.f ? 1.f : (y != y ? y : 0.f);
    return d * dy;
  }
  if (act == VKH_ACT_SIGMOID) {
    float d = 1.0f - y;
    d = d * y;
    return d * dy;
  }
  return dy;
}

// XCD-aware tile order: consecutive remapped ids share an XCD, then tiles are
// grouped by GROUP_M rows of tiles.
__device__ __forceinline__ void tile_coords(const GemmArgs& p, uint32_t& tm, uint32_t& tn) {
  const uint32_t nb = p.tiles_m * p.tiles_n;
  uint32_t b = blockIdx.x;
  if (nb % 8 == 0) b = (b % 8) * (nb / 8) + b / 8;
  constexpr uint32_t GROUP_M = 8;
  const uint32_t width = GROUP_M * p.tiles_n;
  const uint32_t group = b / width;
  const uint32_t first_m = group * GROUP_M;
  const uint32_t gsize = min(p.tiles_m - first_m, GROUP_M);
  tm = first_m + (b % width) % gsize;
  tn = (b % width) / gsize;
}

// ---- packed BF16 path ---------------------------------------------------------------
// BF16 / BF16X3 GEMMs first pack op(A) and op(B)^T into zero-padded, K-major
// BF16 buffers ([Mp][Kp], [Np][Kp]; for BF16X3 also the low parts), so the
// main kernel's inner loop is 16-byte loads, 16-byte LDS stores and MFMAs with
// no conversion and no bounds checks.
constexpr int PK_KALIGN = 64;  // packed K (Kp) is a multiple of every kernel's k slice
constexpr int PK_TR = 128;     // transpose tile (rows r and k) in k_pack_cols (divides every Rp)

// dst[r][k] = bf16(op(src)[r][k]) for r < Rp, k < Kp, zero outside [R, K);
// op(src)[r][k] = src[r*ld + k] (TRANS = false) or src[k*ld + r] (TRANS = true).
// With PARTS > 1 an element is the sum of PARTS BF16 values, each the rounding
// of what the ones before it leave, and a row holds groups of 32 k, the parts
// of a group one after another (so a k slice of a row is contiguous in memory
// in every mode).
template <int PARTS>
__device__ __forceinline__ uint64_t pack_off(uint64_t r, uint64_t k, uint64_t Kp) {
  return PARTS == 1 ? r * Kp + k : r * Kp * PARTS + (k / 32) * (32 * PARTS) + k % 32;
}

// Floats as BF16, two a word.  The conversion instruction rounds as f2bf does
// except for NaNs (f2bf keeps the payload) and denormals (f2bf rounds none of
// them to zero): rows with one of those are converted again by f2bf.
template <int N>
__device__ __forceinline__ void f2bf_pairs(const float (&v)[N], uint32_t (&h)[N / 2]) {
  typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2_t;
  constexpr int SPECIAL = 0x93;  // NaNs and denormals, for v_cmp_class
  bool odd = false;
#pragma unroll
  for (int k = 0; k < N; k += 2) {
    odd |= __builtin_amdgcn_classf(v[k], SPECIAL) | __builtin_amdgcn_classf(v[k + 1], SPECIAL);
    const bf16x2_t t = {(__bf16)v[k], (__bf16)v[k + 1]};
    h[k / 2] = __builtin_bit_cast(uint32_t, t);
  }
  if (__builtin_expect(odd, 0)) {
#pragma unroll
    for (int k = 0; k < N; k += 2) h[k / 2] = f2bf(v[k]) | ((uint32_t)f2bf(v[k + 1]) << 16);
  }
}

// Row-major source: 4 consecutive elements a thread, one thread per 4 of
// the padded [Rp][Kp] (Rp * Kp / 4 < 2^31: the row from one 32-bit
// multiply-high division), so that each load instruction reads one contiguous
// 1 KB run and each store writes 512 B (64-byte runs with PARTS > 1).  HBM-bound:
// 65536 x 1024 in two parts 84 us (96 with the rounding in integer steps).
template <int PARTS>
__global__ void __launch_bounds__(256)
k_pack_rows(const float* src, uint64_t ld, uint64_t R, uint64_t K, uint16_t* dst, uint32_t total4, FastDiv kq,
            uint64_t Kp) {
  const uint32_t t = blockIdx.x * 256 + threadIdx.x;
  if (t >= total4) return;
  const uint32_t r = kq.div(t);
  const uint64_t k = (uint64_t)(t - r * kq.d) * 4;
  float v[4];
  if (r < R && k + 3 < K) {
    const f32x4u_t a = __builtin_nontemporal_load(reinterpret_cast<const f32x4u_t*>(src + r * ld + k));
#pragma unroll
    for (int q = 0; q < 4; ++q) v[q] = a[q];
  } else {
#pragma unroll
    for (int q = 0; q < 4; ++q) v[q] = (r < R && k + q < K) ? src[r * ld + k + q] : 0.f;
  }
  const uint64_t off = pack_off<PARTS>(r, k, Kp);
#pragma unroll
  for (int part = 0; part < PARTS; ++part) {
    uint32_t h[2];
    f2bf_pairs(v, h);
    *reinterpret_cast<uint2*>(dst + off + part * 32) = make_uint2(h[0], h[1]);
#pragma unroll
    for (int q = 0; q < 4; ++q) v[q] = v[q] - __uint_as_float(q & 1 ? h[q / 2] & 0xffff0000u : h[q / 2] << 16);
  }
}

// Transposed source: a T (k) x T (r) tile goes through LDS (BF16
// pairs for the plain pack, rows of T + 1 floats for the split one: the
// column reads of the second phase spread over the banks), so the reads are
// 16-byte loads along r (512-byte row segments) and the writes 16-byte
// stores along k (256-byte row segments of the packed buffer; lengths for T =
// 128).  Rp is a multiple of T; the last k tile may pass Kp.  HBM-bound; with nontemporal
// reads (the source is not needed again, the packed rows are) and the rounding by
// the conversion instruction 4096 x 16384 and its like take 56 us, 69 without.
template <int PARTS, int T>
__global__ void __launch_bounds__(256)
k_pack_cols(const float* src, uint64_t ld, uint64_t R, uint64_t K, uint16_t* dst, uint64_t Rp, uint64_t Kp) {
  const uint64_t r0 = (uint64_t)blockIdx.x * T, k0 = (uint64_t)blockIdx.y * T;
  constexpr int R4 = T / 4;
  constexpr int NL = T * R4 / 256;  // 16-byte loads per thread, all issued before the LDS writes
  vkh_f4v v[NL];
#pragma unroll
  for (int i = 0; i < NL; ++i) {
    const int f = threadIdx.x + i * 256;
    const int kk = f / R4, rr = (f % R4) * 4;
    const uint64_t r = r0 + rr, k = k0 + kk;
    if (k < K && r + 3 < R) {
      v[i] = __builtin_nontemporal_load(reinterpret_cast<const f32x4u_t*>(src + k * ld + r));
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q) v[i][q] = (k < K && r + q < R) ? src[k * ld + r + q] : 0.f;
    }
  }
  if constexpr (PARTS == 1) {
    // BF16 tile: the values are rounded on the way in (the rounding the
    // packed row would apply), so the tile takes 33 KB and four blocks fit
    // a compute unit.  Word w of row kk holds r = 2w (low half) and 2w + 1;
    // a thread of the second phase reads one word of 8 consecutive k and
    // writes the packed rows of both r.
    constexpr int PW = T / 2 + 1;  // words a row: odd, so the column reads spread over banks
    __shared__ uint32_t tb[T][PW];
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int f = threadIdx.x + i * 256;
      const int kk = f / R4, w = (f % R4) * 2;
      const float t[4] = {v[i][0], v[i][1], v[i][2], v[i][3]};
      uint32_t h[2];
      f2bf_pairs(t, h);
      tb[kk][w] = h[0];
      tb[kk][w + 1] = h[1];
    }
    __syncthreads();
    constexpr int KC = T / 8;
    for (int f = threadIdx.x; f < (T / 2) * KC; f += 256) {
      const int rp = f / KC, kc = f % KC;
      const uint64_t k = k0 + kc * 8;
      if (k >= Kp) continue;
      uint32_t wd[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) wd[q] = tb[kc * 8 + q][rp];
      uint4 ev, od;  // rows 2 rp (low halves) and 2 rp + 1 (high halves), k ascending
      ev.x = (wd[0] & 0xffffu) | (wd[1] << 16); od.x = (wd[0] >> 16) | (wd[1] & 0xffff0000u);
      ev.y = (wd[2] & 0xffffu) | (wd[3] << 16); od.y = (wd[2] >> 16) | (wd[3] & 0xffff0000u);
      ev.z = (wd[4] & 0xffffu) | (wd[5] << 16); od.z = (wd[4] >> 16) | (wd[5] & 0xffff0000u);
      ev.w = (wd[6] & 0xffffu) | (wd[7] << 16); od.w = (wd[6] >> 16) | (wd[7] & 0xffff0000u);
      const uint64_t off = (r0 + 2 * rp) * Kp + k;
      *reinterpret_cast<uint4*>(dst + off) = ev;
      *reinterpret_cast<uint4*>(dst + off + Kp) = od;
    }
  } else {  // FP32 tile: the lower parts need the values
    __shared__ float t[T][T + 1];
#pragma unroll
    for (int i = 0; i < NL; ++i) {
      const int f = threadIdx.x + i * 256;
      const int kk = f / R4, rr = (f % R4) * 4;
#pragma unroll
      for (int q = 0; q < 4; ++q) t[kk][rr + q] = v[i][q];
    }
    __syncthreads();
    constexpr int KC = T / 8;  // 8-element chunks per packed row in the tile
    for (int f = threadIdx.x; f < T * KC; f += 256) {
      const int rr = f / KC, kc = f % KC;
      const uint64_t k = k0 + kc * 8;
      if (k >= Kp) continue;
      float v[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) v[q] = t[kc * 8 + q][rr];
      const uint64_t off = pack_off<PARTS>(r0 + rr, k, Kp);
#pragma unroll
      for (int part = 0; part < PARTS; ++part) {
        uint32_t h[4];
        f2bf_pairs(v, h);
        *reinterpret_cast<uint4*>(dst + off + part * 32) = make_uint4(h[0], h[1], h[2], h[3]);
#pragma unroll
        for (int q = 0; q < 8; ++q) v[q] = v[q] - __uint_as_float(q & 1 ? h[q / 2] & 0xffff0000u : h[q / 2] << 16);
      }
    }
  }
}

struct PackedArgs {
  const uint16_t* A;
  const uint16_t* B;
  uint64_t Kp;
  // split k: block (tile, blockIdx.y = s) accumulates k in [s*kc, (s+1)*kc)
  // and writes its raw accumulators to part[s][M][N]; k_splitk_combine then
  // applies the epilogue.  part == nullptr: the whole k range, epilogue here.
  uint64_t kc;
  float* part;
  GemmArgs e;
};

// 4 consecutive floats p[0 .. cnt) (one 16-byte load when `full`), zeros beyond.
__device__ __forceinline__ f32x4_t load4(const float* p, bool full, int cnt) {
  if (full) return *reinterpret_cast<const f32x4_t*>(p);
  f32x4_t v;
  v[0] = cnt > 0 ? p[0] : 0.f;
  v[1] = cnt > 1 ? p[1] : 0.f;
  v[2] = cnt > 2 ? p[2] : 0.f;
  v[3] = cnt > 3 ? p[3] : 0.f;
  return v;
}

// 4 consecutive BF16 values p[0 .. cnt) as floats (one 8-byte load when
// `full`), zeros beyond.
__device__ __forceinline__ f32x4_t load4_bf(const uint16_t* p, bool full, int cnt) {
  f32x4_t v;
  if (full) {
    const uint2 t = *reinterpret_cast<const uint2*>(p);
    v[0] = __uint_as_float(t.x << 16);
    v[1] = __uint_as_float(t.x & 0xffff0000u);
    v[2] = __uint_as_float(t.y << 16);
    v[3] = __uint_as_float(t.y & 0xffff0000u);
    return v;
  }
  v[0] = cnt > 0 ? bf2f(p[0]) : 0.f;
  v[1] = cnt > 1 ? bf2f(p[1]) : 0.f;
  v[2] = cnt > 2 ? bf2f(p[2]) : 0.f;
  v[3] = cnt > 3 ? bf2f(p[3]) : 0.f;
  return v;
}

// the aux activation's outputs at C[m, n..n+3] (FP32 or BF16 aux)
__device__ __forceinline__ f32x4_t aux4(const GemmArgs& e, uint64_t m, uint64_t n, bool full, int cnt) {
  return e.aux16 ? load4_bf(e.aux16 + m * e.ldaux + n, full, cnt) : load4(e.aux + m * e.ldaux + n, full, cnt);
}

// The final values of 4 consecutive outputs C[m, n..n+3] from their
// accumulators, given C's old values (beta != 0), bias[n..n+3] and the aux
// activation's outputs, in the order alpha*acc (+ beta*C) (+ bias[n]),
// activation, times the aux activation's derivative; stored with 16-byte
// accesses when `full` (cnt outputs of the group in range otherwise).  The
// transposed BF16 copy is written here, one element at a time, unless write_t
// is false (the staged epilogue writes it in whole runs).
// D: x holds the derivative factors themselves (ReLU' decoded from codes)
template <bool SIG = true, bool D = false>
__device__ __forceinline__ float4 finish4(const GemmArgs& e, uint64_t m, uint64_t n, float4 acc, bool full,
                                          int cnt, f32x4_t c, f32x4_t b, f32x4_t x, bool write_t) {
  float* cp = e.C + m * e.ldc + n;
  float v[4] = {acc.x, acc.y, acc.z, acc.w};
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    float t = e.alpha * v[q];
    if (e.beta != 0.f) t += e.beta * c[q];
    if (e.bias) t += b[q];
    t = act_apply<SIG>(e.act, t);
    if (e.aux || e.aux16) t = D ? x[q] * t : act_deriv_mul(e.aux_act, x[q], t);
    v[q] = t;
  }
  if (full) {
    if (!e.no_c) *reinterpret_cast<float4*>(cp) = make_float4(v[0], v[1], v[2], v[3]);
    if (e.Cbf) {
      uint2 h;
      h.x = f2bf(v[0]) | ((uint32_t)f2bf(v[1]) << 16);
      h.y = f2bf(v[2]) | ((uint32_t)f2bf(v[3]) << 16);
      *reinterpret_cast<uint2*>(e.Cbf + m * e.ldc + n) = h;
    }
  } else {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if (q < cnt) {
        if (!e.no_c) cp[q] = v[q];
        if (e.Cbf) e.Cbf[m * e.ldc + n + q] = f2bf(v[q]);
      }
    }
  }
  if (e.Cbft && write_t) {
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if (q < cnt) e.Cbft[(n + q) * e.ldt + m] = f2bf(v[q]);
  }
  return make_float4(v[0], v[1], v[2], v[3]);
}

// finish4 with its inputs read here (C's old values, bias, aux).
__device__ __forceinline__ float4 epilogue4(const GemmArgs& e, uint64_t m, uint64_t n, float4 acc,
                                            bool write_t = true) {
  const bool full = e.vec_c && n + 3 < e.N;
  const int cnt = full ? 4 : (int)min<uint64_t>(4, e.N - n);
  const f32x4_t z = {0.f, 0.f, 0.f, 0.f};
  const f32x4_t c = e.beta != 0.f ? load4(e.C + m * e.ldc + n, full, cnt) : z;
  const f32x4_t b = e.bias ? load4(e.bias + n, full, cnt) : z;
  const f32x4_t x = e.aux || e.aux16 ? aux4(e, m, n, full, cnt) : z;
  return finish4(e, m, n, acc, full, cnt, c, b, x, write_t);
}

// Raw accumulators C[m, n..n+3] of one k chunk into part [M][N] (16-byte
// store when the group is whole and rows are 16-byte aligned).
__device__ __forceinline__ void store_part4(float* part, uint64_t N, uint64_t m, uint64_t n, float4 v) {
  float* pp = part + m * N + n;
  if (N % 4 == 0) {
    *reinterpret_cast<float4*>(pp) = v;
  } else {
    const float a[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if (n + q < N) pp[q] = a[q];
  }
}

// Epilogue of a block whose waves each hold TM x TN 32 x 32 accumulator blocks
// of a WM x WN sub-tile at (wm, wn): acc[i][j][r] is C[m, n] with m = m0 + wm*WM +
// i*32 + (r/4)*8 + lhi*4 + r%4 and n = n0 + wn*WN + j*32 + l32 (l32 = lane % 32,
// lhi = lane / 32).  Each wave writes rows i*32 .. i*32+31 of its sub-tile to its
// own 32 x (WN+4) float staging slice of `smem`, then reads them back as 4-float
// row segments (WN/4 lanes per row), so C is accessed in whole row segments.
// With `part` the raw sums go to that k chunk's partial matrix instead.  For
// the transposed BF16 copy (e.Cbft) the row pass puts the final values back
// into the slice and each group of four lanes converts one column of 32 rows
// into a 64-byte run.  The caller's operand tiles in `smem` must be dead (a
// barrier before the call).
template <int WM, int WN, int TM, int TN>
__device__ __forceinline__ void staged_epilogue(float* smem, const f32x16_t (&acc)[TM][TN], const GemmArgs& e,
                                                float* part, uint64_t m0, uint64_t n0, int wm, int wn) {
  static_assert(TM * 32 == WM && TN * 32 == WN, "a pass is 32 rows");
  constexpr int SROW = WN + 4, F4R = WN / 4, RPI = 64 / F4R;
  static_assert(64 % F4R == 0, "whole rows per wave pass");
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int l32 = lane & 31, lhi = lane >> 5;
  float* st = smem + wave * 32 * SROW;
  const uint64_t nb = n0 + wn * WN;
  const bool tr = e.Cbft && !part;
  const bool tr_vec = e.ldt % 8 == 0 && ((uintptr_t)e.Cbft & 15u) == 0;
  // column sums: the wave's WM = 128 rows are one chunk; lane c < WN walks
  // column c down the staged slices in row order, 32 rows per pass
  const bool csum = WM == CS_ROWS && e.cs && !part;
  float csacc = 0.f;
  // A lane's row segments: columns n .. n+3 of rows r0 + k*RPI of each pass.
  // In the common case (a whole 4-column group, every row of the pass in
  // range, no sigmoid) no global load waits between the passes' stores (a
  // wait on a load also waits for every store issued before it): bias is
  // read once; a ReLU' aux is read for every pass before the first store and
  // kept as a 2-bit code per value (positive, NaN, else), which is all ReLU'
  // needs (the BF16 aux); other aux values are in registers before their pass,
  // read during the previous pass where they fit (ITER <= 8), else in groups
  // of PF at its start.  Other segments (and the split-k partial sums) take
  // one loop iteration each, with their own loads.
  constexpr int ITER = 32 / RPI, PF = ITER < 8 ? ITER : 8;
  constexpr bool AHEAD = ITER == PF;
  const int cc = (lane % F4R) * 4, r0 = lane / F4R;
  const uint64_t n = nb + cc;
  const bool ncol = n < e.N;
  const bool lane_fast = !part && e.act != VKH_ACT_SIGMOID && e.vec_c && n + 3 < e.N;
  const f32x4_t z = {0.f, 0.f, 0.f, 0.f};
  const f32x4_t bq = lane_fast && e.bias ? *reinterpret_cast<const f32x4_t*>(e.bias + n) : z;
  const bool aux = lane_fast && (e.aux || e.aux16);
  const bool relu_codes = aux && e.aux16;  // (a BF16 aux is ReLU' only)
  const bool xpre = aux && !relu_codes;
  // codes: 8 bits a row segment (2 a value), four segments a word; read as
  // raw bits, a pass a batch
  constexpr int NSEG = TM * ITER;
  uint32_t cw[(NSEG + 3) / 4];
#pragma unroll
  for (int w = 0; w < (NSEG + 3) / 4; ++w) cw[w] = 0u;
  auto put_code = [&](int seg, uint32_t byte) { cw[seg / 4] |= byte << (8 * (seg % 4)); };
  if (relu_codes) {
    constexpr int BP = 1;
#pragma unroll
    for (int i0 = 0; i0 < TM; i0 += BP) {
      uint2 raw[BP * ITER];
#pragma unroll
      for (int g = 0; g < BP * ITER; ++g) {
        const int i = i0 + g / ITER, k = g % ITER;
        const uint64_t m = m0 + wm * WM + i * 32 + r0 + k * RPI;
        raw[g] = (i < TM && m < e.M) ? *reinterpret_cast<const uint2*>(e.aux16 + m * e.ldaux + n)
                                     : make_uint2(0u, 0u);
      }
#pragma unroll
      for (int g = 0; g < BP * ITER; ++g) {
        if (i0 * ITER + g < NSEG) {
          uint32_t byte = 0u;
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const uint32_t hb = ((q < 2 ? raw[g].x : raw[g].y) >> (16 * (q & 1))) & 0xffffu, mag = hb & 0x7fffu;
            byte |= (mag > 0x7f80u ? 2u : ((hb & 0x8000u) == 0u && mag != 0u ? 1u : 0u)) << (2 * q);
          }
          put_code(i0 * ITER + g, byte);
        }
      }
    }
  }
  // ReLU' of segment seg's aux values, as act_deriv_mul finds it: 1 (positive),
  // NaN (NaN) or 0
  auto relu_x = [&](int seg) {
    const uint32_t byte = (cw[seg / 4] >> (8 * (seg % 4))) & 0xffu;
    f32x4_t xv;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const uint32_t c = (byte >> (2 * q)) & 3u;
      xv[q] = c == 1u ? 1.f : (c == 2u ? __builtin_nanf("") : 0.f);
    }
    return xv;
  };
  f32x4_t xq[PF];
#pragma unroll
  for (int k = 0; k < PF; ++k) xq[k] = z;
  auto load_aux = [&](int i, int k0) {
#pragma unroll
    for (int k = 0; k < PF; ++k) {
      const uint64_t m = m0 + wm * WM + i * 32 + r0 + (k0 + k) * RPI;
      xq[k] = m < e.M ? aux4(e, m, n, true, 4) : z;
    }
  };
  if (xpre && AHEAD) load_aux(0, 0);
  // pass i: rows i*32 .. i*32+31 of the sub-tile (a constant i: the registers of
  // its accumulators need constant indices)
  auto pass = [&](auto ic) __attribute__((always_inline)) {
    constexpr int i = decltype(ic)::value;
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) st[((r / 4) * 8 + lhi * 4 + (r % 4)) * SROW + j * 32 + l32] = acc[i][j][r];
    __syncthreads();
    const uint64_t mb = m0 + wm * WM + i * 32;
    if (lane_fast && mb + 31 < e.M) {
#pragma unroll
      for (int k0 = 0; k0 < ITER; k0 += PF) {
        if (xpre && !AHEAD) load_aux(i, k0);
#pragma unroll
        for (int k = 0; k < PF; ++k) {
          const int rr = r0 + (k0 + k) * RPI;
          const float4 v = *reinterpret_cast<const float4*>(st + rr * SROW + cc);
          const f32x4_t c = e.beta != 0.f ? *reinterpret_cast<const f32x4_t*>(e.C + (mb + rr) * e.ldc + n) : z;
          const float4 f = relu_codes
                               ? finish4<false, true>(e, mb + rr, n, v, true, 4, c, bq, relu_x(i * ITER + k0 + k), false)
                               : finish4<false>(e, mb + rr, n, v, true, 4, c, bq, xq[k], false);
          if (csum || tr) *reinterpret_cast<float4*>(st + rr * SROW + cc) = f;
        }
      }
    } else {
      for (int rr = r0; rr < 32; rr += RPI) {
        const uint64_t m = mb + rr;
        if (m < e.M && ncol) {
          const float4 v = *reinterpret_cast<const float4*>(st + rr * SROW + cc);
          if (part) {
            store_part4(part, e.N, m, n, v);
          } else {
            const float4 f = epilogue4(e, m, n, v, false);
            if (csum || tr) *reinterpret_cast<float4*>(st + rr * SROW + cc) = f;
          }
        }
      }
    }
    if (xpre && AHEAD && i + 1 < TM) load_aux(i + 1, 0);
    __syncthreads();
    if (csum && lane < WN) {
      if (mb + 31 < e.M) {
        // the sum stays a chain in row order; its reads go out 8 at a time
#pragma unroll
        for (int r8 = 0; r8 < 32; r8 += 8) {
          float v[8];
#pragma unroll
          for (int q = 0; q < 8; ++q) v[q] = st[(r8 + q) * SROW + lane];
#pragma unroll
          for (int q = 0; q < 8; ++q) csacc = (i == 0 && r8 + q == 0) ? v[q] : csacc + v[q];
        }
      } else {
        for (int rr = 0; rr < 32; ++rr) {
          if (mb + rr >= e.M) break;
          const float v = st[rr * SROW + lane];
          csacc = (i == 0 && rr == 0) ? v : csacc + v;
        }
      }
    }
    if (csum && !tr) __syncthreads();  // st is read before the next pass writes it
    if (tr) {
      // four lanes per column, 8 rows (16 bytes) each: one store covers 16
      // columns in whole 64-byte runs
      const int q = lane & 3;
      for (int c = lane >> 2; c < WN; c += 16) {
        const uint64_t nt = nb + c;
        if (nt >= e.N) continue;
        uint16_t* dst = e.Cbft + nt * e.ldt + mb + q * 8;
        const float* col = st + q * 8 * SROW + c;
        if (tr_vec && mb + 31 < e.M) {
          uint32_t w[4];
#pragma unroll
          for (int t = 0; t < 4; ++t)
            w[t] = f2bf(col[(2 * t) * SROW]) | ((uint32_t)f2bf(col[(2 * t + 1) * SROW]) << 16);
          *reinterpret_cast<uint4*>(dst) = make_uint4(w[0], w[1], w[2], w[3]);
        } else {
          for (int r = 0; r < 8; ++r)
            if (mb + q * 8 + r < e.M) dst[r] = f2bf(col[r * SROW]);
        }
      }
      __syncthreads();
    }
  };
  // A copy of the code for each pass, whose accumulators die with it: a loop over
  // the passes of a 256 x 256 tile spills 104 registers (16384 x 4096 x 256 in such
  // tiles 364 us, 351 so; x 4096 4045 and 4023), over those of a 128 x 128 tile it
  // costs 2% at 2500^3 and saves 1.7% with B transposed.
  static_for<TM>([&](auto ic) __attribute__((always_inline)) { pass(ic); });
  if (csum && lane < WN) {
    const uint64_t m = m0 + wm * WM, nc = nb + lane;
    if (m < e.M && nc < e.N) e.cs[(m / CS_ROWS) * e.N + nc] = csacc;
  }
}

// Epilogue straight from the accumulators, for kernels that multiply with the
// operands exchanged (each block of the accumulators is then C^T's, so a lane
// holds 4 consecutive columns of a row): no LDS, 16-byte accesses, 64-byte runs
// of a row an instruction.  For alpha, beta, bias and ReLU (and the split-k
// partial sums); anything else takes copies_epilogue (small FP32 tiles: the
// 128 x 128 one's staged epilogue).  acc[i][j] is the
// 16 x 16 block (i, j) of the wave's sub-tile: row l16 = lane % 16, columns
// 4 (lane / 16) .. + 3.  65536 x 1024 x 1024 151 us against 200 us staged.
static bool direct_ok(const GemmArgs& e) {
  return !e.Cbft && !e.cs && !e.Cbf && !e.no_c && !e.aux && !e.aux16 && e.act != VKH_ACT_SIGMOID;
}

template <int TM, int TN>
__device__ __forceinline__ void direct_epilogue(const f32x4_t (&acc)[TM][TN], const GemmArgs& e, float* part,
                                                uint64_t mw, uint64_t nw) {
  const int lane = threadIdx.x & 63, l16 = lane & 15, lq = lane >> 4;
  const uint64_t m0 = mw + l16, n0 = nw + lq * 4;
  const uint64_t ld = part ? e.N : e.ldc;
  float* cp = (part ? part : e.C) + m0 * ld + n0;
  // raw sums (a partial, or nothing to apply)
  const bool raw = part || (e.alpha == 1.f && e.beta == 0.f && !e.bias && e.act == VKH_ACT_NONE);
  auto apply = [&](float acc1, float c, float b) {
    float t = e.alpha * acc1;
    if (e.beta != 0.f) t += e.beta * c;
    if (e.bias) t += b;
    return act_apply<false>(e.act, t);
  };
  // whole groups of 4 columns: 16-byte accesses at any 4-byte alignment
  const bool inm = mw + TM * 16 <= e.M;  // every row in range
  if (raw) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
      if (inm || m0 + i * 16 < e.M) {
#pragma unroll
        for (int j = 0; j < TN; ++j)
          if (n0 + j * 16 + 3 < e.N) *reinterpret_cast<f32x4u_t*>(cp + i * 16 * ld + j * 16) = acc[i][j];
      }
  } else {
    f32x4_t b[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j)
      b[j] = e.bias && n0 + j * 16 + 3 < e.N ? *reinterpret_cast<const f32x4u_t*>(e.bias + n0 + j * 16)
                                             : f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < TM; ++i)
      if (inm || m0 + i * 16 < e.M) {
        f32x4_t c[TN];
        if (e.beta != 0.f)  // a block row's old values before its first store
#pragma unroll
          for (int j = 0; j < TN; ++j)
            if (n0 + j * 16 + 3 < e.N) c[j] = *reinterpret_cast<const f32x4u_t*>(cp + i * 16 * ld + j * 16);
#pragma unroll
        for (int j = 0; j < TN; ++j)
          if (n0 + j * 16 + 3 < e.N) {
            f32x4_t v;
#pragma unroll
            for (int q = 0; q < 4; ++q) v[q] = apply(acc[i][j][q], c[j][q], b[j][q]);
            *reinterpret_cast<f32x4u_t*>(cp + i * 16 * ld + j * 16) = v;
          }
      }
  }
  // the group that straddles the last column: 1 to 3 elements
  if (e.N % 4 != 0 && nw < e.N && e.N < nw + TN * 16) {
    const int jt = (int)((e.N - nw) / 16);
    f32x4_t v[TM];
    static_for<TN>([&](auto jc) __attribute__((always_inline)) {
      if (jt == decltype(jc)::value)
#pragma unroll
        for (int i = 0; i < TM; ++i) v[i] = acc[i][decltype(jc)::value];
    });
    const uint64_t n = n0 + jt * 16;
    if (n < e.N && n + 3 >= e.N) {
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int q = 0; q < 3; ++q)
          if (m0 + i * 16 < e.M && n + q < e.N) {
            float* d = cp + i * 16 * ld + jt * 16 + q;
            *d = raw ? v[i][q] : apply(v[i][q], e.beta != 0.f ? *d : 0.f, e.bias ? e.bias[n + q] : 0.f);
          }
    }
  }
}

// ---- register epilogue of the pipelined kernel, with BF16 copies and column sums ----
// For what direct_epilogue leaves: BF16 copies of C (Cbf) and of C^T (Cbft),
// column sums, aux derivatives, sigmoid.  The operands are exchanged as there,
// so a lane holds 4 consecutive columns of a row and the values become final
// where they are.  Only the copies pass through LDS, each wave in its own
// area, so no block barrier is needed: a block row's 16 x WN BF16 values for
// whole runs of a row, 64 rows' transposed values for 128-byte runs of C^T,
// and (column sums) a block row's floats, which a lane per column adds in row
// order.  What bounds it is the count of vector instructions, about 10 an
// element (a quarter of them the rounding to BF16), and the stores.
template <int TM, int TN>
struct CopyArea {
  static constexpr int WM = TM * 16, WN = TN * 16;
  static constexpr int TR = WM < 64 ? WM : 64;   // rows of a transposed tile
  static constexpr int TP = TR + 8, RP = WN + 8, FP = WN + 4;
  static constexpr bool CSUM = WM == CS_ROWS && WN == 64;
  static constexpr int T_BYTES = WN * TP * 2, R_BYTES = 16 * RP * 2, F_BYTES = CSUM ? 16 * FP * 4 : 0;
  static constexpr int BYTES = T_BYTES + R_BYTES + F_BYTES + WN * 4;  // of a wave
  static_assert(T_BYTES % 16 == 0 && R_BYTES % 16 == 0, "16-byte accesses");
};

// LDS of this wave written by other lanes of it is read after this (and the
// other way round): the hardware keeps a wave's LDS accesses in order
__device__ __forceinline__ void wave_order() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// AUX: 0 none, 1 e.aux16, 2 e.aux
template <int AUX, int TM, int TN>
__device__ __forceinline__ void copies_epilogue(char* area, const f32x4_t (&acc)[TM][TN], const GemmArgs& e,
                                                uint64_t mw, uint64_t nw) {
  using L = CopyArea<TM, TN>;
  constexpr int WN = L::WN;
  static_assert(TM % 2 == 0, "block rows in pairs");
  uint16_t* tt = reinterpret_cast<uint16_t*>(area);
  uint16_t* rt = reinterpret_cast<uint16_t*>(area + L::T_BYTES);
  float* ft = reinterpret_cast<float*>(area + L::T_BYTES + L::R_BYTES);
  float* bt = reinterpret_cast<float*>(area + L::T_BYTES + L::R_BYTES + L::F_BYTES);
  int lane = threadIdx.x & 63, l16 = lane & 15, lq = lane >> 4;
  // the lane's number anew, so that no address made from it is kept in a
  // register from one block row to the next (the accumulators leave too few)
  auto fresh = [&]() __attribute__((always_inline)) {
    asm volatile("" : "+v"(lane));
    l16 = lane & 15;
    lq = lane >> 4;
  };
  // every column in range: groups of 4 at any 4-byte alignment, with the
  // lane's place within 16 rows in 32 bits next to a wave-uniform address
  const bool whole = nw + WN <= e.N && e.ldc < (1u << 26) && e.ldaux < (1u << 26);
  // (no bias: -0, which changes no value)
  if (lane < WN) bt[lane] = e.bias ? e.bias[nw + lane < e.N ? nw + lane : e.N - 1] : -0.f;
  wave_order();
  // Row m0 + l16 of a matrix, TN groups of 4 columns.  Rows and columns beyond
  // the matrix read its last ones; what is made of them is not stored.
  auto load_row = [&](float(&d)[TN * 4], const float* base, uint64_t ld, uint64_t m0) __attribute__((always_inline)) {
    if (whole && m0 + 15 < e.M) {
      const float* p = base + m0 * ld + nw;
      const uint32_t off = l16 * (uint32_t)ld + lq * 4;
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const f32x4_t t = *reinterpret_cast<const f32x4u_t*>(p + j * 16 + off);
#pragma unroll
        for (int q = 0; q < 4; ++q) d[j * 4 + q] = t[q];
      }
    } else {
      const float* p = base + min(m0 + l16, e.M - 1) * ld;
#pragma unroll
      for (int k = 0; k < TN * 4; ++k) d[k] = p[min(nw + lq * 4 + (k / 4) * 16 + k % 4, e.N - 1)];
    }
  };
  // the aux activation's outputs, two block rows ahead (a BF16 aux as raw
  // bits, two columns a register)
  constexpr int NX = AUX == 2 ? TN * 4 : TN * 2;
  float ring[2][NX];
  const bool aux8 = whole && ((uintptr_t)e.aux16 & 7u) == 0 && e.ldaux % 4 == 0;
  auto load_aux = [&](float(&d)[NX], int i) __attribute__((always_inline)) {
    const uint64_t m0 = mw + i * 16;
    if constexpr (AUX == 2) {
      load_row(d, e.aux, e.ldaux, m0);
    } else if constexpr (AUX == 1) {
      if (aux8 && m0 + 15 < e.M) {
        const uint16_t* p = e.aux16 + m0 * e.ldaux + nw;
        const uint32_t off = l16 * (uint32_t)e.ldaux + lq * 4;
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          const uint2 t = *reinterpret_cast<const uint2*>(p + j * 16 + off);
          d[2 * j] = __uint_as_float(t.x);
          d[2 * j + 1] = __uint_as_float(t.y);
        }
      } else {
        const uint16_t* p = e.aux16 + min(m0 + l16, e.M - 1) * e.ldaux;
        auto at = [&](int k) { return (uint32_t)p[min(nw + lq * 4 + (k / 4) * 16 + k % 4, e.N - 1)]; };
#pragma unroll
        for (int k = 0; k < TN * 4; k += 2) d[k / 2] = __uint_as_float(at(k) | (at(k + 1) << 16));
      }
    }
  };
  if constexpr (AUX != 0) {
    load_aux(ring[0], 0);
    load_aux(ring[1], 1);
  }
  const bool row16 = ((uintptr_t)e.Cbf & 15u) == 0 && e.ldc % 8 == 0 && nw + WN <= e.N;
  const bool col16 = ((uintptr_t)e.Cbft & 15u) == 0 && e.ldt % 8 == 0;
  const bool csum = L::CSUM && e.cs;
  // ReLU: what is less than this becomes 0 (nothing without it)
  const float floor_v = e.act == VKH_ACT_RELU ? 0.f : -__builtin_inff();
  float csacc = 0.f;
  // one copy of the code for every two block rows (the ring's registers);
  // only the choice of the accumulators, whose indices are constants, is
  // unrolled further
#pragma unroll 1
  for (int i2 = 0; i2 < TM; i2 += 2) {
    static_for<2>([&](auto hc) __attribute__((always_inline)) {
      constexpr int H = decltype(hc)::value;
      const int i = i2 + H;
      const uint64_t m0 = mw + i * 16;
      if (m0 >= e.M) return;
      fresh();
      float v[TN * 4];
      static_for<TM / 2>([&](auto ic) __attribute__((always_inline)) {
        if (i2 == 2 * decltype(ic)::value)
#pragma unroll
          for (int k = 0; k < TN * 4; ++k) v[k] = acc[2 * decltype(ic)::value + H][k / 4][k % 4];
      });
#pragma unroll
      for (int k = 0; k < TN * 4; ++k) v[k] = e.alpha * v[k];
      if (e.beta != 0.f) {
        float c[TN * 4];
        load_row(c, e.C, e.ldc, m0);
#pragma unroll
        for (int k = 0; k < TN * 4; ++k) v[k] += e.beta * c[k];
      }
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const f32x4_t b = *reinterpret_cast<const f32x4_t*>(bt + j * 16 + lq * 4);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const float t = v[j * 4 + q] + b[q];
          v[j * 4 + q] = t < floor_v ? 0.f : t;
        }
      }
      if (__builtin_expect(e.act == VKH_ACT_SIGMOID, 0)) {
        // one copy of its FP64 code: the values move past it in turn
#pragma unroll 1
        for (int t = 0; t < TN * 4; ++t) {
          const float y = act_apply(VKH_ACT_SIGMOID, v[0]);
#pragma unroll
          for (int k = 0; k + 1 < TN * 4; ++k) v[k] = v[k + 1];
          v[TN * 4 - 1] = y;
        }
      }
      if constexpr (AUX == 1) {
        // (ReLU' only)
#pragma unroll
        for (int k = 0; k < TN * 4; ++k) {
          const uint32_t w = __float_as_uint(ring[H][k / 2]);
          v[k] = act_deriv_mul(VKH_ACT_RELU, __uint_as_float(k & 1 ? w & 0xffff0000u : w << 16), v[k]);
        }
      } else if constexpr (AUX == 2) {
#pragma unroll
        for (int k = 0; k < TN * 4; ++k) v[k] = act_deriv_mul(e.aux_act, ring[H][k], v[k]);
      }
      if (AUX != 0 && i + 2 < TM) load_aux(ring[H], i + 2);
      if (!e.no_c) {
        if (whole && m0 + 15 < e.M) {
          float* p = e.C + m0 * e.ldc + nw;
          const uint32_t off = l16 * (uint32_t)e.ldc + lq * 4;
#pragma unroll
          for (int j = 0; j < TN; ++j)
            *reinterpret_cast<f32x4u_t*>(p + j * 16 + off) = f32x4_t{v[j * 4], v[j * 4 + 1], v[j * 4 + 2], v[j * 4 + 3]};
        } else if (m0 + l16 < e.M) {
          const uint64_t n = nw + lq * 4;
          float* p = e.C + (m0 + l16) * e.ldc + n;
#pragma unroll
          for (int k = 0; k < TN * 4; ++k)
            if (n + (k / 4) * 16 + k % 4 < e.N) p[(k / 4) * 16 + k % 4] = v[k];
        }
      }
      wave_order();  // (the previous block row's reads come before these writes)
      if (csum) {
#pragma unroll
        for (int j = 0; j < TN; ++j)
          *reinterpret_cast<f32x4_t*>(ft + l16 * L::FP + j * 16 + lq * 4) =
              f32x4_t{v[j * 4], v[j * 4 + 1], v[j * 4 + 2], v[j * 4 + 3]};
      }
      if (e.Cbf || e.Cbft) {
        uint32_t h[TN * 2];
        f2bf_pairs(v, h);
        if (e.Cbf) {
#pragma unroll
          for (int j = 0; j < TN; ++j)
            *reinterpret_cast<uint2*>(rt + l16 * L::RP + j * 16 + lq * 4) = make_uint2(h[2 * j], h[2 * j + 1]);
        }
        if (e.Cbft) {
          uint16_t* d = tt + lq * 4 * L::TP + (i * 16) % L::TR + l16;
#pragma unroll
          for (int k = 0; k < TN * 4; ++k)
            d[((k / 4) * 16 + k % 4) * L::TP] = (uint16_t)(k & 1 ? h[k / 2] >> 16 : h[k / 2]);
        }
      }
      wave_order();
      if (e.Cbf) {
        constexpr int LPR = WN / 8, RPI = 64 / LPR;  // lanes of a row, rows an instruction
        const int c = (lane % LPR) * 8, r0 = lane / LPR;
        uint16_t* dst = e.Cbf + (m0 + r0) * e.ldc + nw + c;
        const uint16_t* src = rt + r0 * L::RP + c;
        if (row16 && m0 + 15 < e.M) {
#pragma unroll
          for (int r = 0; r < 16 / RPI; ++r)
            *reinterpret_cast<uint4*>(dst + r * RPI * e.ldc) = *reinterpret_cast<const uint4*>(src + r * RPI * L::RP);
        } else {
#pragma unroll 1
          for (int r = r0; r < 16 && m0 + r < e.M; r += RPI, dst += RPI * e.ldc, src += RPI * L::RP)
            for (int q = 0; q < 8 && nw + c + q < e.N; ++q) dst[q] = src[q];
        }
      }
      if (csum) {
        // a chain in row order from the slab's first row (every lane a column)
        float f[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) f[r] = ft[r * L::FP + lane];
        csacc = i == 0 ? f[0] : csacc + f[0];
        if (m0 + 15 < e.M) {
#pragma unroll
          for (int r = 1; r < 16; ++r) csacc = csacc + f[r];
        } else {
#pragma unroll
          for (int r = 1; r < 16; ++r) csacc = m0 + r < e.M ? csacc + f[r] : csacc;
        }
      }
      if (e.Cbft && ((i + 1) * 16 % L::TR == 0 || m0 + 16 >= e.M)) {
        const uint64_t mt = mw + (i * 16) / L::TR * L::TR;   // first row of the tile
        constexpr int LPC = L::TR / 8, CPI = 64 / LPC;       // lanes of a column, columns an instruction
        const int r = (lane % LPC) * 8, c0 = lane / LPC;
        uint16_t* dst = e.Cbft + (nw + c0) * e.ldt + mt + r;
        const uint16_t* src = tt + c0 * L::TP + r;
        if (col16 && nw + WN <= e.N && mt + L::TR <= e.M) {
#pragma unroll
          for (int c = 0; c < WN / CPI; ++c)
            *reinterpret_cast<uint4*>(dst + c * CPI * e.ldt) = *reinterpret_cast<const uint4*>(src + c * CPI * L::TP);
        } else {
#pragma unroll 1
          for (int c = c0; c < WN && nw + c < e.N; c += CPI, dst += CPI * e.ldt, src += CPI * L::TP)
            for (int q = 0; q < 8 && mt + r + q < e.M; ++q) dst[q] = src[q];
        }
      }
    });
  }
  if (csum && nw + lane < e.N) e.cs[(mw / CS_ROWS) * e.N + nw + lane] = csacc;
}

// ---- FP32 path ----------------------------------------------------------------------
// FP32 products on v_mfma_f32_32x32x2_f32 with the operands read as stored
// (no packing pass).  A BM x BN tile per block, WGM x WGN waves of
// (BM/WGM) x (BN/WGN); 32-deep k slices go through registers into
// double-buffered LDS with one barrier per slice, the next slice's global
// loads in flight while the current one is multiplied.  Each operand keeps
// its global layout in LDS:
//   * K-major (A row-major [M][K], B stored [N][K]): rows of 32 floats
//     (128 B) whose 16-byte chunks are XOR-swizzled by row (chunk c of row r
//     sits at position c ^ (r & 7)), so 8 consecutive rows read at one chunk
//     touch 8 distinct bank groups;
//   * otherwise (A stored [K][M], B row-major [K][N]): 32 k rows of the tile
//     width plus 8 floats, so the two half-waves of a fragment read (k rows 4
//     apart) fall on different banks.
// The MFMA takes one float of A and one of B per lane: lane (r, h), r =
// lane % 32, h = lane / 32, supplies row (column) r at its k.  In the 8-deep
// k group g of a slice, MFMA t = 0..3 takes k = 8g + 4h + t, so a K-major
// operand feeds the whole group with one 16-byte read per 32-row block.
// Every output sums its k in this fixed order; slices beyond K are zeros,
// so K needs no padding.
//
// Operand loads never branch per lane: a lane whose element is out of range
// loads from a block of zeros instead, so the compiler issues every load of
// a slice back to back and waits for them only at the LDS store.  (With
// per-lane guarded loads it waits for each load before issuing the next.)
constexpr int F32_BK = 32;

static __device__ __attribute__((aligned(16))) float k_f32_zeros[4];

//
// VEC: the operand's contiguous extent is a multiple of 4, so a run of 4 is
// wholly in or out of range.  Otherwise a run that crosses the end is read from
// 4 elements before the end (the extent is more than 4) and shifted into place
// at the LDS store.  16-byte loads need 4-byte alignment only.
template <int ROWS, bool KMAJ, int THREADS, bool VEC, int BK = F32_BK>
struct F32Stager {
  static constexpr int NV = ROWS * BK / 4 / THREADS;  // float4 per thread
  static_assert(NV * 4 * THREADS == ROWS * BK, "whole float4 per thread");
  static constexpr int R4 = KMAJ ? BK / 4 : ROWS / 4;  // runs of a row
  // LDS row (floats); tiles of up to 64 rows are read by 16-row fragments, four
  // k rows (0, 4, 1, 5 apart) at a time, which 36 more floats keep apart
  static constexpr int LD = KMAJ ? BK : ROWS > 64 ? ROWS + 8 : ROWS == 64 ? 100 : 36;
  static constexpr int FLOATS = KMAJ ? ROWS * BK : BK * LD;
  f32x4_t r[NV];

  // Rows row0.. (K-major: the operand's rows; otherwise its columns) at k0,
  // as runs of 4 elements along the contiguous dimension.
  __device__ __forceinline__ void load(const float* P, uint64_t ld, uint64_t row0, uint64_t nrows,
                                       uint64_t k0, uint64_t K) {
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int idx = threadIdx.x + i * THREADS;
      uint64_t gr, gc, rlim, clim;  // run row, first column, and their limits
      if constexpr (KMAJ) {
        gr = row0 + idx / R4; gc = k0 + (idx % R4) * 4; rlim = nrows; clim = K;
      } else {
        gr = k0 + idx / R4; gc = row0 + (idx % R4) * 4; rlim = K; clim = nrows;
      }
      const bool ok = gr < rlim && gc < clim;
      if constexpr (!VEC) gc = min(gc, clim - 4);
      r[i] = *reinterpret_cast<const f32x4u_t*>(ok ? P + (gr * ld + gc) : k_f32_zeros);
    }
  }

  // into LDS; row0, nrows, k0, K as given to load
  __device__ __forceinline__ void store(float* s, uint64_t row0, uint64_t nrows, uint64_t k0, uint64_t K) const {
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int idx = threadIdx.x + i * THREADS;
      int off;
      if constexpr (KMAJ) {
        const int row = idx / R4, c = idx % R4;
        off = row * BK + ((c ^ (row & 7)) << 2);
      } else {
        off = (idx / R4) * LD + (idx % R4) * 4;
      }
      f32x4_t v = r[i];
      if constexpr (!VEC) {
        const uint64_t gc = (KMAJ ? k0 : row0) + (idx % R4) * 4, last = (KMAJ ? K : nrows) - 4;
        if (gc > last) {  // shifted down by the elements before the run (or out of range: zeros)
          const uint64_t sh = gc - last;
          v[0] = sh == 1 ? v[1] : sh == 2 ? v[2] : sh == 3 ? v[3] : 0.f;
          v[1] = sh == 1 ? v[2] : sh == 2 ? v[3] : 0.f;
          v[2] = sh == 1 ? v[3] : 0.f;
          v[3] = 0.f;
        }
      }
      *reinterpret_cast<f32x4_t*>(s + off) = v;
    }
  }

  // values of tile row `row` for the MFMAs t = 0..3 of k group g, half-wave h
  __device__ __forceinline__ static f32x4_t frag(const float* s, int row, int g, int h) {
    if constexpr (KMAJ) {
      const int c = 2 * g + h;
      return *reinterpret_cast<const f32x4_t*>(s + row * BK + ((c ^ (row & 7)) << 2));
    } else {
      const float* q = s + (8 * g + 4 * h) * LD + row;
      return f32x4_t{q[0], q[LD], q[2 * LD], q[3 * LD]};
    }
  }

  // values of tile row `row` for the two 16 x 16 x 4 MFMAs of k group g: lanes
  // 16 q .. 16 q + 15 supply k = 0, 4, 1, 5 [q] of the group, then 2, 6, 3, 7,
  // the order in which four 32 x 32 x 2 MFMAs add them
  __device__ __forceinline__ static void frag16(const float* s, int row, int g, int q, float (&v)[2]) {
    if constexpr (KMAJ) {
      const f32x4_t f = frag(s, row, g, q & 1);
      v[0] = q & 2 ? f[1] : f[0];
      v[1] = q & 2 ? f[3] : f[2];
    } else {
      const float* p = s + (8 * g + 4 * (q & 1) + (q >> 1)) * LD + row;
      v[0] = p[0];
      v[1] = p[2 * LD];
    }
  }
};

template <bool AK, bool BKM, bool VEC, int BM, int BN, int WGM, int WGN>
__global__ void __launch_bounds__(64 * WGM * WGN, 2)
k_gemm_f32(GemmArgs p, float* part, uint64_t kc) {
  constexpr int THREADS = 64 * WGM * WGN, WAVES = WGM * WGN;
  constexpr int WM = BM / WGM, WN = BN / WGN;
  static_assert(WM % 32 == 0 && WN % 32 == 0, "32 x 32 MFMA blocks per wave");
  constexpr int TM = WM / 32, TN = WN / 32;
  using SA = F32Stager<BM, AK, THREADS, VEC>;
  using SB = F32Stager<BN, BKM, THREADS, VEC>;
  constexpr int MAIN = 2 * (SA::FLOATS + SB::FLOATS), STAGE = WAVES * 32 * (WN + 4);
  constexpr int SMEM_FLOATS = MAIN > STAGE ? MAIN : STAGE;
  __shared__ __attribute__((aligned(16))) float smem[SMEM_FLOATS];
  auto As = [&](int b) { return smem + b * SA::FLOATS; };
  auto Bs = [&](int b) { return smem + 2 * SA::FLOATS + b * SB::FLOATS; };

  uint32_t tm, tn;
  tile_coords(p, tm, tn);
  const uint64_t m0 = (uint64_t)tm * BM, n0 = (uint64_t)tn * BN;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = wave / WGN, wn = wave % WGN;
  const int l32 = lane & 31, lhi = lane >> 5;
  const int arow = wm * WM + l32, brow = wn * WN + l32;

  SA sa;
  SB sb;
  f32x16_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

  // fragments of one k group, double-buffered: group g+1 is read while the
  // MFMAs of group g issue
  constexpr int G = F32_BK / 8;                                // k groups per slice
  constexpr int NM = 4 * TM * TN;                              // MFMAs per group
  constexpr int NDS = (AK ? TM : 2 * TM) + (BKM ? TN : 2 * TN);  // LDS reads per group
  constexpr int WPM = (SA::NV + SB::NV + NM - 1) / NM;         // LDS stores per MFMA
  static_assert(NDS <= NM, "fragment reads fit between the MFMAs of a group");
  f32x4_t fa[2][TM], fb[2][TN];
  auto frags = [&](int buf, int fi, int g) {
#pragma unroll
    for (int i = 0; i < TM; ++i) fa[fi][i] = SA::frag(As(buf), arow + i * 32, g, lhi);
#pragma unroll
    for (int j = 0; j < TN; ++j) fb[fi][j] = SB::frag(Bs(buf), brow + j * 32, g, lhi);
  };

  // k range of this block: all of k, or chunk blockIdx.y of kc (a multiple of
  // F32_BK, so the slices tile the chunk) when k is split
  const uint64_t K = p.K;
  const uint64_t kb = part ? (uint64_t)blockIdx.y * kc : 0;
  const uint64_t ke = part ? min(kb + kc, K) : K;
  const uint64_t nk = (ke - kb + F32_BK - 1) / F32_BK;
  sa.load(p.A, p.lda, m0, p.M, kb, K);
  sb.load(p.B, p.ldb, n0, p.N, kb, K);
  sa.store(As(0), m0, p.M, kb, K);
  sb.store(Bs(0), n0, p.N, kb, K);
  __syncthreads();
  frags(0, 0, 0);
  int cur = 0;
  for (uint64_t kt = 0; kt < nk; ++kt) {
    // the next slice (past K: zeros) into registers
    // (the prefetch after a chunk's last slice is stored but never used)
    sa.load(p.A, p.lda, m0, p.M, kb + (kt + 1) * F32_BK, K);
    sb.load(p.B, p.ldb, n0, p.N, kb + (kt + 1) * F32_BK, K);
    // keep the loads here: left to itself the scheduler sinks them to the
    // LDS store at the end of the slice, where their latency is exposed
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const int c = g & 1;
      if (g + 1 < G) frags(cur, c ^ 1, g + 1);
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[c][i][t], fb[c][j][t], acc[i][j], 0, 0, 0);
      // every group but the last alternates one MFMA with one fragment read
      // of the next group, so LDS latency hides behind matrix-core work
      if (g + 1 < G) {
#pragma unroll
        for (int q = 0; q < NDS; ++q) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // MFMA
          __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // DS read
        }
        __builtin_amdgcn_sched_group_barrier(0x008, NM - NDS, 0);
      }
    }
    // the last group's MFMAs alternate with the LDS stores of the next slice
    sa.store(As(cur ^ 1), m0, p.M, kb + (kt + 1) * F32_BK, K);
    sb.store(Bs(cur ^ 1), n0, p.N, kb + (kt + 1) * F32_BK, K);
#pragma unroll
    for (int q = 0; q < NM; ++q) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);    // MFMA
      __builtin_amdgcn_sched_group_barrier(0x200, WPM, 0);  // DS write
    }
    __syncthreads();
    cur ^= 1;
    frags(cur, 0, 0);
  }
  __syncthreads();  // every wave is done with the operand tiles before staging
  staged_epilogue<WM, WN>(smem, acc, p, part ? part + (uint64_t)blockIdx.y * p.M * p.N : nullptr,
                          m0, n0, wm, wn);
}

// Small FP32 tiles (T x T, four waves of T/2 x T/2) for products with few
// outputs, on 16 x 16 x 4 MFMAs: an FP32 MFMA adds its k terms one after the
// other, so in the k order of frag16 every output has the bits of the larger
// tiles.  A 128 x 128 tile takes 128 matrix-core cycles a k on its CU however
// few tiles there are (512^3: 16 CUs busy, 43 us); 64 x 64 takes 32 and 32 x 32
// takes 8 (9.6 us), bound by the latency of a slice's loads.  Slices are 32 and
// 64 deep: 64 and 128 are no faster alone (9.1-9.5 us) and leave one block a CU
// (5137 x 586 x 270 52 against 35 us).  The code is small and the accumulators
// are stored without staging (direct_epilogue): 150 x 32 x 32 3.3 against 12 us.
template <bool AK, bool BKM, bool VEC, int T, int BK>
__global__ void __launch_bounds__(256)
k_gemm_f32_small(GemmArgs p, float* part, uint64_t kc) {
  constexpr int W = T / 2, TM = W / 16;
  using SA = F32Stager<T, AK, 256, VEC, BK>;
  using SB = F32Stager<T, BKM, 256, VEC, BK>;
  __shared__ __attribute__((aligned(16))) float smem[2 * (SA::FLOATS + SB::FLOATS)];
  auto As = [&](int b) { return smem + b * SA::FLOATS; };
  auto Bs = [&](int b) { return smem + 2 * SA::FLOATS + b * SB::FLOATS; };
  uint32_t tm, tn;
  tile_coords(p, tm, tn);
  const uint64_t m0 = (uint64_t)tm * T, n0 = (uint64_t)tn * T;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, wm = wave >> 1, wn = wave & 1;
  const int l16 = lane & 15, lq = lane >> 4;
  f32x4_t acc[TM][TM];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  const uint64_t K = p.K;
  const uint64_t kb = part ? (uint64_t)blockIdx.y * kc : 0;
  const uint64_t ke = part ? min(kb + kc, K) : K;
  const uint64_t nk = (ke - kb + BK - 1) / BK;
  SA sa;
  SB sb;
  sa.load(p.A, p.lda, m0, p.M, kb, ke);
  sb.load(p.B, p.ldb, n0, p.N, kb, ke);
  sa.store(As(0), m0, p.M, kb, ke);
  sb.store(Bs(0), n0, p.N, kb, ke);
  __syncthreads();
  for (uint64_t kt = 0; kt < nk; ++kt) {
    const int cur = (int)(kt & 1);
    const uint64_t k1 = kb + (kt + 1) * BK;
    const bool more = kt + 1 < nk;
    if (more) {
      sa.load(p.A, p.lda, m0, p.M, k1, ke);
      sb.load(p.B, p.ldb, n0, p.N, k1, ke);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int g = 0; g < BK / 8; ++g) {
      float fa[TM][2], fb[TM][2];
#pragma unroll
      for (int i = 0; i < TM; ++i) SA::frag16(As(cur), wm * W + i * 16 + l16, g, lq, fa[i]);
#pragma unroll
      for (int j = 0; j < TM; ++j) SB::frag16(Bs(cur), wn * W + j * 16 + l16, g, lq, fb[j]);
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TM; ++j)  // (operands exchanged, for direct_epilogue)
            acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(fb[j][u], fa[i][u], acc[i][j], 0, 0, 0);
    }
    if (more) {
      sa.store(As(cur ^ 1), m0, p.M, k1, ke);
      sb.store(Bs(cur ^ 1), n0, p.N, k1, ke);
    }
    __syncthreads();
  }
  direct_epilogue(acc, p, part ? part + (uint64_t)blockIdx.y * p.M * p.N : nullptr, m0 + wm * W, n0 + wn * W);
}

// Kernel configurations of the FP32 path (tile and wave grid).  They differ
// in how the output is tiled only: every output sums its k in the same order,
// so the choice never changes a result.
typedef void (*F32Launch)(dim3, hipStream_t, const GemmArgs&, bool ta, bool tb, bool vec, float* part,
                          uint64_t kc);
#define VKH_F32_LAYOUTS(LAUNCH)                  \
  do { /* A is K-major unless transposed, B when transposed */ \
    if (!ta && !tb) LAUNCH(true, false);         \
    else if (!ta && tb) LAUNCH(true, true);      \
    else if (ta && !tb) LAUNCH(false, false);    \
    else LAUNCH(false, true);                    \
  } while (0)
template <int BM, int BN, int WGM, int WGN>
static void launch_f32(dim3 grid, hipStream_t s, const GemmArgs& a, bool ta, bool tb, bool vec, float* part,
                       uint64_t kc) {
  const dim3 block(64 * WGM * WGN);
#define VKH_F32_LAUNCH(AK, BKM)                                                                   \
  do {                                                                                            \
    if (vec)                                                                                      \
      hipLaunchKernelGGL((k_gemm_f32<AK, BKM, true, BM, BN, WGM, WGN>), grid, block, 0, s, a, part, kc); \
    else                                                                                          \
      hipLaunchKernelGGL((k_gemm_f32<AK, BKM, false, BM, BN, WGM, WGN>), grid, block, 0, s, a, part, kc); \
  } while (0)
  VKH_F32_LAYOUTS(VKH_F32_LAUNCH);
#undef VKH_F32_LAUNCH
}
template <int T, int BK>
static void launch_f32_small(dim3 grid, hipStream_t s, const GemmArgs& a, bool ta, bool tb, bool vec, float* part,
                             uint64_t kc) {
#define VKH_F32_LAUNCH(AK, BKM)                                                                  \
  do {                                                                                           \
    if (vec)                                                                                     \
      hipLaunchKernelGGL((k_gemm_f32_small<AK, BKM, true, T, BK>), grid, dim3(256), 0, s, a, part, kc); \
    else                                                                                         \
      hipLaunchKernelGGL((k_gemm_f32_small<AK, BKM, false, T, BK>), grid, dim3(256), 0, s, a, part, kc); \
  } while (0)
  VKH_F32_LAYOUTS(VKH_F32_LAUNCH);
#undef VKH_F32_LAUNCH
}
#undef VKH_F32_LAYOUTS
struct F32Cfg {
  int bm, bn, waves, wm;  // wm: rows of a wave's slab (BM / WGM)
  F32Launch launch;
};
static const F32Cfg F32_CFGS[] = {
    {128, 128, 4, 64, launch_f32<128, 128, 2, 2>},
    {256, 256, 8, 128, launch_f32<256, 256, 2, 4>},
    {64, 64, 4, 32, launch_f32_small<64, 32>},
    {32, 32, 4, 16, launch_f32_small<32, 64>},
};
constexpr int F32_NCFG = sizeof(F32_CFGS) / sizeof(F32_CFGS[0]), F32_CFG_256 = 1;

// Sums the S k-chunk partials of each output in chunk order and applies the
// GEMM epilogue (alpha, beta * C, bias, activation, aux derivative, BF16 copy).
__global__ void __launch_bounds__(256)
k_splitk_combine(const float* part, uint64_t S, GemmArgs e) {
  const uint64_t gpr = (e.N + 3) / 4, total = e.M * gpr, MN = e.M * e.N;
  const uint64_t stride = (uint64_t)gridDim.x * 256;
  for (uint64_t t = (uint64_t)blockIdx.x * 256 + threadIdx.x; t < total; t += stride) {
    const uint64_t m = t / gpr, n = (t - m * gpr) * 4;
    const float* pp = part + m * e.N + n;
    float4 acc;
    if (e.N % 4 == 0) {
      acc = *reinterpret_cast<const float4*>(pp);
      for (uint64_t s = 1; s < S; ++s) {
        const float4 v = *reinterpret_cast<const float4*>(pp + s * MN);
        acc.x += v.x; acc.y += v.y; acc.z += v.z; acc.w += v.w;
      }
    } else {
      float a[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        if (n + q < e.N) {
          float x = pp[q];
          for (uint64_t s = 1; s < S; ++s) x += pp[s * MN + q];
          a[q] = x;
        }
      }
      acc = make_float4(a[0], a[1], a[2], a[3]);
    }
    epilogue4(e, m, n, acc);
  }
}

// ---- pipelined BF16 products ----------------------------------------------------
// C from packed operands on v_mfma_f32_16x16x32_bf16.  PARTS BF16 values stand
// for each operand element (1: BF16 mode, 2: split mode); a packed row holds its
// k in groups of KG, the parts of a group one after another, so a slice of every row is ROWB
// contiguous bytes in every mode.
//
// What bounds a loop that fills LDS, waits at a barrier and multiplies is the
// wait: with the next slice requested at the start of a slice and awaited at
// its end, 8192^3 ran at 1.04-1.19 PFLOP/s (matrix cores 58% busy).  Here:
//  * slices go from global memory straight into LDS (no staging registers), a
//    slice and a half ahead: a wave reads its sub-tile in quarters (halves of
//    its rows and of its columns), and each half's LDS is refilled with the
//    slice after next as soon as every wave has read it, so a load has six
//    phases (about 3000 cycles) to arrive.  Waits count the loads still in
//    flight (vmcnt) instead of draining them;
//  * the two waves of a SIMD run half a phase apart (one extra barrier at the
//    start for the second half of the block): while one reads fragments, the
//    other multiplies;
//  * 16-byte chunks of an LDS row sit XOR-swizzled by row so that the 16 rows
//    of a fragment read fall on 16 different 16-byte banks.
// Measured on the loop alone (same operands, interleaved): 8192^3 761-790 us
// against 928-1062 us for the loop it replaces (1.45 PFLOP/s; 864 us with the
// staggered waves but loads one slice ahead, 855 us without the stagger, 955 us
// with 32 x 32 x 16 instructions), 16384 x 4096 x 4096 405-430 against 490-583 us.
// One 16 x 16 x 32 instruction gives the bits of the two 32 x 32 x 16 ones it
// replaces.
__device__ __forceinline__ void load_lds16(const char* src, char* dst) {
#ifdef __HIP_DEVICE_COMPILE__  // (the host pass would drop the launch stub of a template that uses the builtin)
  __builtin_amdgcn_global_load_lds(src, dst, 16, 0, 0);
#endif
}

// waits until at most N global loads are in flight / a block barrier, neither
// of which the scheduler moves anything across
template <int N>
__device__ __forceinline__ void wait_loads() {
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | 0x0f70);
  __builtin_amdgcn_sched_barrier(0);
}
__device__ __forceinline__ void phase_barrier() {
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
}

template <int PARTS>
struct PipeSlice {
  static constexpr int KG = PARTS == 1 ? 64 : 32;  // k of a slice
  static constexpr int ROWB = KG * 2 * PARTS;      // bytes of a slice row
  static constexpr int NF = ROWB / 64;             // 64-byte fragments of a row: k steps, or parts
  static constexpr int CPR = ROWB / 16;            // 16-byte chunks of a row
  // LDS position of chunk c of row r: rows of 128 bytes alternate between the
  // halves of the 256-byte bank line, so 8 row pairs permute 8 positions
  __device__ __forceinline__ static int pos(int r, int c) { return c ^ ((r >> 1) & 7); }
};

// The operands are exchanged (each block of the accumulators is C^T's).
// DIRECT: direct_epilogue, else copies_epilogue
template <int BM, int BN, int WGM, int WGN, int PARTS, bool DIRECT>
__global__ void __launch_bounds__(64 * WGM * WGN, 2)
k_gemm_pipe(PackedArgs p) {
  using S = PipeSlice<PARTS>;
  constexpr int ROWB = S::ROWB, NF = S::NF, WAVES = WGM * WGN;
  constexpr bool STAGGER = WAVES == 8;  // two waves a SIMD
  constexpr int WM = BM / WGM, WN = BN / WGN;
  constexpr int HM = WM / 2, HN = WN / 2;  // rows / columns of a half
  static_assert(HM % 16 == 0 && HN % 16 == 0, "16 x 16 MFMA blocks per quarter");
  constexpr int TMH = HM / 16, TNH = HN / 16;
  // 1 KB loads (one wave instruction) of one wave row's half, and per wave
  constexpr int GA = HM * ROWB / 1024, GB = HN * ROWB / 1024;
  constexpr int LA = WGM * GA / WAVES, LB = WGN * GB / WAVES;
  static_assert(LA * WAVES == WGM * GA && LB * WAVES == WGN * GB, "whole loads per wave and half");
  constexpr int A_BYTES = BM * ROWB, B_BYTES = BN * ROWB;
  constexpr int MAIN_BYTES = 2 * (A_BYTES + B_BYTES);
  constexpr int EPI_BYTES = DIRECT ? 0 : WAVES * CopyArea<2 * TMH, 2 * TNH>::BYTES;
  constexpr int SMEM_BYTES = MAIN_BYTES > EPI_BYTES ? MAIN_BYTES : EPI_BYTES;
  __shared__ __attribute__((aligned(16))) char smem[SMEM_BYTES];

  const GemmArgs& e = p.e;
  uint32_t tm, tn;
  tile_coords(e, tm, tn);
  const uint64_t m0 = (uint64_t)tm * BM, n0 = (uint64_t)tn * BN;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave / WGN, wn = wave % WGN;

  // Slice kt of this block's k range starts kt * ROWB bytes into each row.
  const uint64_t rowp = p.Kp * 2 * PARTS;  // bytes of a packed row
  const uint64_t kb = p.part ? (uint64_t)blockIdx.y * p.kc : 0;
  const uint64_t nk = ((p.part ? min(kb + p.kc, p.Kp) : p.Kp) - kb) / S::KG;
  const char* ga = reinterpret_cast<const char*>(p.A) + m0 * rowp + kb * 2 * PARTS;
  const char* gb = reinterpret_cast<const char*>(p.B) + n0 * rowp + kb * 2 * PARTS;

  // 1 KB load q of a wave for half h of A (B): LDS offset within the operand's
  // slice (wave-uniform) and this lane's source offset in 16-byte chunks
  auto half_off = [&](int q, int g, int h, int wrows, int hrows) {
    const int idx = q * WAVES + wave;
    return (idx / g) * wrows * ROWB + h * hrows * ROWB + (idx % g) * 1024;
  };
  auto src_off = [&](int lds_off) {
    const int c = (lds_off >> 4) + lane, r = c / S::CPR;
    return (uint32_t)r * (uint32_t)(rowp >> 4) + S::pos(r, c % S::CPR);
  };
  uint32_t oa[2][LA], ob[2][LB];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
#pragma unroll
    for (int q = 0; q < LA; ++q) oa[h][q] = src_off(half_off(q, GA, h, WM, HM));
#pragma unroll
    for (int q = 0; q < LB; ++q) ob[h][q] = src_off(half_off(q, GB, h, WN, HN));
  }
  // slices past the end load the last one again (in range, never read)
  auto slice = [&](uint64_t kt) { return (kt < nk ? kt : nk - 1) * ROWB; };
  auto load_a = [&](int b, uint64_t ks, int h) {
#pragma unroll
    for (int q = 0; q < LA; ++q) load_lds16(ga + ks + ((uint64_t)oa[h][q] << 4), smem + b * A_BYTES + half_off(q, GA, h, WM, HM));
  };
  auto load_b = [&](int b, uint64_t ks, int h) {
#pragma unroll
    for (int q = 0; q < LB; ++q)
      load_lds16(gb + ks + ((uint64_t)ob[h][q] << 4), smem + 2 * A_BYTES + b * B_BYTES + half_off(q, GB, h, WN, HN));
  };

  f32x4_t acc[2 * TMH][2 * TNH];
#pragma unroll
  for (int i = 0; i < 2 * TMH; ++i)
#pragma unroll
    for (int j = 0; j < 2 * TNH; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  // fragment f (64 bytes: 32 k of one part) of 16 rows: lane l holds row
  // l % 16, 16-byte chunk l / 16
  const int l16 = lane & 15, lq = lane >> 4;
  auto frag = [&](const char* buf, int row, int f) {
    return *reinterpret_cast<const bf16x8_t*>(buf + row * ROWB + S::pos(row, 4 * f + lq) * 16);
  };
  bf16x8_t fa[TMH][NF], fb[2][TNH][NF];
  auto read_a = [&](int b, int h) {
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
      for (int i = 0; i < TMH; ++i) fa[i][f] = frag(smem + b * A_BYTES, wm * WM + h * HM + i * 16 + l16, f);
  };
  auto read_b = [&](int b, int h) {
#pragma unroll
    for (int f = 0; f < NF; ++f)
#pragma unroll
      for (int j = 0; j < TNH; ++j)
        fb[h][j][f] = frag(smem + 2 * A_BYTES + b * B_BYTES, wn * WN + h * HN + j * 16 + l16, f);
  };
  auto mul = [&](int h, int g, int f, int q) {
#pragma unroll
    for (int i = 0; i < TMH; ++i)
#pragma unroll
      for (int j = 0; j < TNH; ++j)
        acc[h * TMH + i][g * TNH + j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            fb[g][j][q], fa[i][f], acc[h * TMH + i][g * TNH + j], 0, 0, 0);
  };
  // quarter (h, g): every product of its fragments, k in order (split mode:
  // lo * hi, hi * lo, hi * hi of 32 k at a time)
  auto quarter = [&](int h, int g) {
    phase_barrier();
    if constexpr (PARTS == 1) {
      mul(h, g, 0, 0);
      mul(h, g, 1, 1);
    } else {
      mul(h, g, 1, 0);
      mul(h, g, 0, 1);
      mul(h, g, 0, 0);
    }
    // (without the stagger every wave has read a half before any wave passes
    // the next phase's barrier, which is before its refill is requested)
    if constexpr (STAGGER) phase_barrier();
    else __builtin_amdgcn_sched_barrier(0);
  };

  load_a(0, slice(0), 0);
  load_b(0, slice(0), 0);
  load_b(0, slice(0), 1);
  load_a(0, slice(0), 1);
  load_a(1, slice(1), 0);
  load_b(1, slice(1), 0);
  load_b(1, slice(1), 1);
  wait_loads<2 * LA + 3 * LB>();
  phase_barrier();
  if (STAGGER && wave >= WAVES / 2) phase_barrier();
  for (uint64_t kt = 0; kt < nk; ++kt) {
    const int cur = (int)(kt & 1);
    const uint64_t k1 = slice(kt + 1), k2 = slice(kt + 2);
    read_b(cur, 0);
    read_a(cur, 0);
    load_a(cur ^ 1, k1, 1);
    wait_loads<3 * LA + 2 * LB>();  // this slice's second half of B has landed
    quarter(0, 0);
    read_b(cur, 1);
    wait_loads<2 * LA + 2 * LB>();  // this slice's second half of A has landed
    quarter(0, 1);
    read_a(cur, 1);
    load_a(cur, k2, 0);
    load_b(cur, k2, 0);
    quarter(1, 1);
    load_b(cur, k2, 1);
    wait_loads<2 * LA + 3 * LB>();  // the next slice's first halves have landed
    quarter(1, 0);
  }
  if (STAGGER && wave < WAVES / 2) phase_barrier();
  wait_loads<0>();  // the last loads no longer write LDS
  float* part = p.part ? p.part + (uint64_t)blockIdx.y * e.M * e.N : nullptr;
  if constexpr (DIRECT) {
    direct_epilogue(acc, e, part, m0 + wm * WM, n0 + wn * WN);
  } else {
    __syncthreads();  // (the waves' areas lie over every wave's operands)
    const uint64_t mw = m0 + wm * WM, nw = n0 + wn * WN;
    char* area = smem + wave * CopyArea<2 * TMH, 2 * TNH>::BYTES;
    if (mw >= e.M || nw >= e.N) return;
    if (e.aux16) copies_epilogue<1>(area, acc, e, mw, nw);
    else if (e.aux) copies_epilogue<2>(area, acc, e, mw, nw);
    else copies_epilogue<0>(area, acc, e, mw, nw);
  }
}

// Kernel configurations of the packed path: tile, k slice, waves and the rows
// of a wave's slab.  Split mode has two parts in a slice row, so half the k.
typedef void (*PackedLaunch)(dim3, hipStream_t, const PackedArgs&);
template <int BM, int BN, int WGM, int WGN, int PARTS>
static void launch_pipe(dim3 grid, hipStream_t s, const PackedArgs& pa) {
  if (pa.part || direct_ok(pa.e))
    hipLaunchKernelGGL((k_gemm_pipe<BM, BN, WGM, WGN, PARTS, true>), grid, dim3(64 * WGM * WGN), 0, s, pa);
  else
    hipLaunchKernelGGL((k_gemm_pipe<BM, BN, WGM, WGN, PARTS, false>), grid, dim3(64 * WGM * WGN), 0, s, pa);
}
struct PackedCfg {
  int bm, bn, bk, waves, wm;  // wm: rows of a wave's slab (BM / WGM)
  PackedLaunch launch;
};
static const PackedCfg BF16_CFGS[] = {
    {256, 256, 64, 8, 128, launch_pipe<256, 256, 2, 4, 1>},
    {128, 128, 64, 4, 64, launch_pipe<128, 128, 2, 2, 1>},
    {64, 64, 64, 4, 32, launch_pipe<64, 64, 2, 2, 1>},
    // (256 x 128 and 128 x 256 with 8 waves were fastest on none of 16 shapes)
};
static const PackedCfg SPLIT_CFGS[] = {
    {256, 256, 32, 8, 128, launch_pipe<256, 256, 2, 4, 2>},
    {128, 128, 32, 4, 64, launch_pipe<128, 128, 2, 2, 2>},
    {64, 64, 32, 4, 32, launch_pipe<64, 64, 2, 2, 2>},
};
constexpr int PK_MAXTILE = 256;  // largest bm / bn of any configuration

static const PackedCfg* packed_cfgs(int mode, int& count) {
  if (mode == VKH_GEMM_BF16) { count = (int)(sizeof(BF16_CFGS) / sizeof(BF16_CFGS[0])); return BF16_CFGS; }
  count = (int)(sizeof(SPLIT_CFGS) / sizeof(SPLIT_CFGS[0]));
  return SPLIT_CFGS;
}

// Configuration without tuning, from measurements on MI355X.  The pipelined
// kernels: the tile with the least estimated time, blocks of a CU times the
// measured time of a tile per k (ns; alone on its CU / sharing it) plus a
// fixed part (us).  Measured us for the tiles 256 / 128 / 64: 512^3 19 / 8.5 /
// 5.2, 1024^3 28 / 12.7 / 7.6, 4096 x 1024 x 1024 30 / 15.2 / 16.3,
// 3000^3 72 / 69 / 127, 16384 x 4096 x 4096 402 / 504 / 792, 65536 x 1024 x
// 1024 150 / 212 / 288.
// Split mode, packing included: 1024^3 68 / 36 / 26, 4096 x 1024 x 1024 75 /
// 46 / 47, 3000^3 194 / 195 / 284, 8192^3 2172 / 2697 / 3508.
// FP32 tiles likewise (the 256 x 256 tile for long k, where its blocks, whose
// epilogue is not hidden by another block of the CU, fill the chip evenly), us for
// 128 / 64 / 32: 150 x 32 x 32 12.2 / 3.9 / 3.3, 512^3 43 / 19 / 9.6, 1024^3 33 / 36 /
// 41, 5137 x 586 x 270 44 / 35 / 35, 2048 x 2048 x 512 50 / 54 / 63, 4096 x 1024 x 1024
// 92 / 102 / 123; for 256 / 128: 16384 x 4096 x 256 351 / 317, 65536 x 1024 x 1024 1092 /
// 1090, 8192 x 8192 x 2048 2064 / 2118, 16384 x 4096 x 4096 4023 / 4174, 8192^3 7935 / 8350.
static uint64_t splitk_chunk(uint64_t M, uint64_t N, uint64_t Kp);
static uint64_t f32_splitk_chunk(uint64_t M, uint64_t N, uint64_t K);

struct TileCost {
  int cfg;
  uint64_t tile;
  // us once, and a block; ns a k of a block: alone on its CU, and sharing it
  double fixed_us, block_us, alone_ns, shared_ns;
};
static const TileCost F32_COST[] = {{0, 128, 5.0, 3.0, 76.0, 61.0}, {2, 64, 3.0, 0.0, 32.0, 25.0},
                                    {3, 32, 2.5, 0.0, 14.0, 9.0}, {1, 256, 8.0, 28.0, 233.0, 233.0}};
static const TileCost BF16_COST[] = {{0, 256, 4.0, 0.0, 22.9, 22.9}, {1, 128, 3.5, 0.0, 8.2, 7.5},
                                     {2, 64, 2.5, 0.0, 4.7, 3.5}};
static const TileCost SPLIT_COST[] = {{0, 256, 4.0, 0.0, 59.5, 59.5}, {1, 128, 3.5, 0.0, 22.0, 18.9},
                                      {2, 64, 2.5, 0.0, 11.0, 6.3}};

// the configuration with the least estimated time (us)
static int default_cfg(int mode, uint64_t M, uint64_t N, uint64_t K) {
  const bool f32 = mode == VKH_GEMM_FP32;
  const TileCost* T = f32 ? F32_COST : mode == VKH_GEMM_BF16 ? BF16_COST : SPLIT_COST;
  const uint64_t k = std::max<uint64_t>(K, 1), Kp = f32 ? k : ceil_div(k, (uint64_t)PK_KALIGN) * PK_KALIGN;
  const uint64_t kc = f32 ? f32_splitk_chunk(M, N, Kp) : splitk_chunk(M, N, Kp), S = ceil_div(Kp, kc);
  int cfg = 0;
  double bt = 0;
  for (int i = 0; i < (f32 ? 4 : 3); ++i) {
    const double n = (double)ceil_div(ceil_div(M, T[i].tile) * ceil_div(N, T[i].tile) * S, (uint64_t)256);
    const double t = T[i].fixed_us + n * T[i].block_us +
                     1e-3 * (double)kc * std::max(T[i].alone_ns, T[i].shared_ns * n);
    if (i == 0 || t < bt) { cfg = T[i].cfg; bt = t; }
  }
  return cfg;
}

// number of kernel configurations of a mode
static int mode_cfgs(int mode) {
  if (mode == VKH_GEMM_FP32) return F32_NCFG;
  int n = 0;
  packed_cfgs(mode, n);
  return n;
}

static std::array<uint64_t, 6> cfg_key(int mode, int ta, int tb, uint64_t M, uint64_t N, uint64_t K) {
  return {(uint64_t)mode, (uint64_t)(ta != 0), (uint64_t)(tb != 0), M, N, K};
}

// The configuration of a product on a context: the one chosen for it, else the
// default.  With column sums, which need waves of 128-row slabs, large FP32
// products default to their 256 x 256 tile whatever is faster without.
static int product_cfg(const vkh_gpu* g, int mode, int ta, int tb, uint64_t M, uint64_t N, uint64_t K, bool colsum) {
  auto it = g->gemm_cfg.find(cfg_key(mode, ta, tb, M, N, K));
  if (it != g->gemm_cfg.end()) return it->second;
  if (colsum && mode == VKH_GEMM_FP32 && ceil_div(M, (uint64_t)256) * ceil_div(N, (uint64_t)256) >= 512)
    return F32_CFG_256;
  return default_cfg(mode, M, N, K);
}

// Fills p[0..n) with values in [-0.5, 0.5) from a hash of the index (operands
// of the autotuning runs: data-dependent power draw makes zero operands an
// unrepresentative benchmark).
__global__ void __launch_bounds__(256) k_fill_noise(float* p, uint64_t n, uint32_t seed) {
  const uint64_t stride = (uint64_t)gridDim.x * 256;
  for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += stride) {
    uint32_t h = (uint32_t)i * 0x9e3779b1u ^ (uint32_t)(i >> 32) ^ seed;
    h ^= h >> 16; h *= 0x85ebca6bu; h ^= h >> 13; h *= 0xc2b2ae35u; h ^= h >> 16;
    p[i] = (float)(h >> 8) * (1.0f / 16777216.0f) - 0.5f;
  }
}

// Split k.  A product with few output tiles and a long k leaves most CUs
// idle (4096 x 256 x 16384: 16 tiles of 256 x 256), so k is split into S
// chunks that run as separate blocks; k_splitk_combine sums the chunk
// partials in chunk order.  S and the chunk bounds depend on (M, N, K) only,
// never on the kernel configuration, so every configuration accumulates each
// chunk in the same order and configurations still never change results.
constexpr uint64_t SPLITK_MIN_KP = 4096;    // shorter k: no split
constexpr uint64_t SPLITK_MIN_CHUNK = 1024;  // k per chunk at least
constexpr uint64_t SPLITK_REF_BLOCKS = 256;  // blocks to aim for (one per CU of MI355X)

static uint64_t splitk_chunk(uint64_t M, uint64_t N, uint64_t Kp) {
  const uint64_t tiles = ceil_div(M, 256) * ceil_div(N, 256);
  if (Kp < SPLITK_MIN_KP || tiles * 2 > SPLITK_REF_BLOCKS) return Kp;
  const uint64_t S = std::min(ceil_div(SPLITK_REF_BLOCKS, tiles), Kp / SPLITK_MIN_CHUNK);
  if (S < 2) return Kp;
  return ceil_div(Kp / PK_KALIGN, S) * PK_KALIGN;
}

static size_t operand_bytes(int mode, uint64_t M, uint64_t N, uint64_t Kp) {
  const uint64_t Mp = ceil_div(M, PK_MAXTILE) * PK_MAXTILE, Np = ceil_div(N, PK_MAXTILE) * PK_MAXTILE;
  const uint64_t parts = mode == VKH_GEMM_BF16X3 ? 2 : 1;
  return (size_t)ceil_div((Mp + Np) * Kp * 2 * parts, 256) * 256;
}

// Packing area of an M x N x K product: operands with rows padded to
// PK_MAXTILE, which covers every configuration (so a reservation never
// depends on tuning), then the split-k partials [S][M][N] when k is split.
static size_t packed_bytes(int mode, uint64_t M, uint64_t N, uint64_t K) {
  const uint64_t Kp = ceil_div(std::max<uint64_t>(K, 1), PK_KALIGN) * PK_KALIGN;
  const uint64_t kc = splitk_chunk(M, N, Kp);
  const uint64_t S = ceil_div(Kp, kc);
  return operand_bytes(mode, M, N, Kp) + (S > 1 ? (size_t)(S * M * N * 4) : 0);
}

// Packing area.  Eager calls share a per-context grow-only area: stream order
// keeps uses apart, and the caller holds pack_mu until the last kernel that
// uses the area is launched.  A captured GEMM uses its graph's packing region, which
// the graph owns for as long as it can be replayed; it is sized when the
// capture begins from what vkh_gemm_reserve recorded, and a capture that
// needs more fails and records the size for the next capture.
static uint16_t* pack_area(vkh_gpu* g, size_t bytes) {
  if (g->capturing) {
    if (bytes <= g->graph_pack_bytes) return (uint16_t*)g->graph_pack;
    g->graph_pack_hint = std::max(g->graph_pack_hint, bytes);
    fail(VKH_OUT_OF_MEMORY, "graph GEMM packing region too small (" + std::to_string(g->graph_pack_bytes) +
                                " < " + std::to_string(bytes) +
                                " bytes); call vkh_gemm_reserve before the capture, or capture again");
  }
  if (bytes <= g->pack_bytes) return (uint16_t*)g->pack;
  VKH_REQUIRE(g->alloc, "GEMM packing needs a context with its own allocator");
  if (g->pack) g->alloc->release(g->pack);
  g->pack = nullptr;
  g->pack_bytes = 0;
  const size_t want = bytes + bytes / 4;
  g->pack = g->alloc->allocate(want);
  g->pack_bytes = want;
  return (uint16_t*)g->pack;
}

template <int PARTS>
static void pack_operand(vkh_gpu* g, const float* src, uint64_t ld, bool trans, uint64_t R,
                         uint64_t K, uint16_t* dst, uint64_t Rp, uint64_t Kp) {
  if (!trans) {
    const uint64_t total4 = Rp * (Kp / 4);
    VKH_REQUIRE(total4 < (uint64_t(1) << 31), "gemm pack: operand too large");
    hipLaunchKernelGGL((k_pack_rows<PARTS>), dim3((unsigned)ceil_div(total4, 256)), dim3(256), 0, g->stream,
                       src, ld, R, K, dst, (uint32_t)total4, FastDiv((uint32_t)(Kp / 4)), Kp);
  } else {
    VKH_REQUIRE(Rp % PK_TR == 0, "gemm pack: padded rows not a multiple of the tile");
    // Tiles of 64 x 64 where 128 x 128 ones are fewer than two a compute unit: 573 x
    // 1301 and its like in two parts 4.7 us against 9.4, 500 x 500 2.9 against 6.0, 4000 x 1000
    // 7.2 against 8.6; at four a unit (4096 x 2048) 9.4 against 10.2 in one part.
    const bool small = (Rp / PK_TR) * ceil_div(Kp, PK_TR) < 2 * (uint64_t)(g->num_cus > 0 ? g->num_cus : 256);
    const unsigned t = small ? PK_TR / 2 : PK_TR;
    const dim3 grid((unsigned)(Rp / t), (unsigned)ceil_div(Kp, (uint64_t)t));
    auto kernel = small ? k_pack_cols<PARTS, PK_TR / 2> : k_pack_cols<PARTS, PK_TR>;
    hipLaunchKernelGGL(kernel, grid, dim3(256), 0, g->stream, src, ld, R, K, dst, Rp, Kp);
  }
  check_launch("gemm pack");
}

// a_pre / b_pre (BF16 mode, K % PK_KALIGN == 0): op(A) / op(B)^T already in
// the packed layout -- BF16 rows of K elements, M / N rounded up to
// PK_MAXTILE rows -- so that operand's packing pass is skipped (the bits are
// the ones it would write)
static void gemm_packed(vkh_gpu* g, int mode, bool ta, bool tb, GemmArgs& a, int cfg,
                        const uint16_t* a_pre = nullptr, const uint16_t* b_pre = nullptr) {
  const bool split = mode == VKH_GEMM_BF16X3;
  int ncfg = 0;
  const PackedCfg* cfgs = packed_cfgs(mode, ncfg);
  VKH_REQUIRE(cfg >= 0 && cfg < ncfg, "gemm: configuration index out of range");
  const PackedCfg& s = cfgs[cfg];
  // rows padded to the tile, and to the transposing pack's
  const uint64_t pm = std::max(s.bm, PK_TR), pn = std::max(s.bn, PK_TR);
  const uint64_t Mp = ceil_div(a.M, pm) * pm, Np = ceil_div(a.N, pn) * pn;
  const uint64_t Kp = ceil_div(std::max<uint64_t>(a.K, 1), PK_KALIGN) * PK_KALIGN;
  std::lock_guard<std::mutex> lock(g->pack_mu);
  uint16_t* base = pack_area(g, packed_bytes(mode, a.M, a.N, a.K));
  const int parts = split ? 2 : 1;
  uint16_t* Bp = base + Mp * Kp * parts;
  // op(A)[m][k] and op(B)^T[n][k] = op(B)[k][n]
  if (split) {
    pack_operand<2>(g, a.A, a.lda, ta, a.M, a.K, base, Mp, Kp);
    pack_operand<2>(g, a.B, a.ldb, !tb, a.N, a.K, Bp, Np, Kp);
  } else {
    if (!a_pre) pack_operand<1>(g, a.A, a.lda, ta, a.M, a.K, base, Mp, Kp);
    if (!b_pre) pack_operand<1>(g, a.B, a.ldb, !tb, a.N, a.K, Bp, Np, Kp);
  }
  a.tiles_m = (uint32_t)ceil_div(a.M, (uint64_t)s.bm);
  a.tiles_n = (uint32_t)ceil_div(a.N, (uint64_t)s.bn);
  const uint64_t nb = (uint64_t)a.tiles_m * a.tiles_n;
  VKH_REQUIRE(nb < (uint64_t(1) << 31), "GEMM too large");
  const uint64_t kc = splitk_chunk(a.M, a.N, Kp);
  const uint64_t S = ceil_div(Kp, kc);
  float* part = nullptr;
  if (S > 1) part = reinterpret_cast<float*>(reinterpret_cast<char*>(base) + operand_bytes(mode, a.M, a.N, Kp));
  PackedArgs pa{a_pre ? a_pre : base, b_pre ? b_pre : Bp, Kp, kc, part, a};
  s.launch(dim3((unsigned)nb, (unsigned)S), g->stream, pa);
  check_launch("gemm (packed)");
  if (S > 1) {
    const uint64_t groups = a.M * ceil_div(a.N, 4);
    hipLaunchKernelGGL(k_splitk_combine, dim3(stream_grid(g, groups, 256, 8)), dim3(256), 0, g->stream,
                       (const float*)part, S, a);
    check_launch("gemm split-k combine");
  }
}

// FP32 split k: as above, for fewer than 256 tiles of 128 x 128 (the
// smallest FP32 tile, 2 blocks per CU) and K >= 1024, in chunks of at least
// 256 that are multiples of the 32-deep slice, aiming at 512 blocks.  The
// chunk bounds depend on (M, N, K) only.  4096 x 256 x 16384 (a weight
// gradient over a batch of 16384): 8 chunks, 31 -> 121-126 TFLOP/s.
constexpr uint64_t F32_SPLITK_MIN_K = 1024, F32_SPLITK_MIN_CHUNK = 256, F32_SPLITK_BLOCKS = 512;

static uint64_t f32_splitk_chunk(uint64_t M, uint64_t N, uint64_t K) {
  const uint64_t tiles = ceil_div(M, 128) * ceil_div(N, 128);
  if (K < F32_SPLITK_MIN_K || tiles * 2 > F32_SPLITK_BLOCKS) return K;
  const uint64_t S = std::min(ceil_div(F32_SPLITK_BLOCKS, tiles), K / F32_SPLITK_MIN_CHUNK);
  if (S < 2) return K;
  return ceil_div(ceil_div(K, (uint64_t)F32_BK), S) * F32_BK;
}

// split-k partials [S][M][N] of an FP32 product (0 when k is not split)
static size_t f32_split_bytes(uint64_t M, uint64_t N, uint64_t K) {
  const uint64_t S = ceil_div(K, f32_splitk_chunk(M, N, K));
  return S > 1 ? (size_t)(S * M * N * 4) : 0;
}

static void gemm_f32(vkh_gpu* g, bool ta, bool tb, GemmArgs& a, int cfg) {
  VKH_REQUIRE(cfg >= 0 && cfg < F32_NCFG, "gemm: configuration index out of range");
  // (a small tile stores what direct_epilogue can; its partial sums always)
  const uint64_t kc = f32_splitk_chunk(a.M, a.N, a.K);
  const uint64_t S = ceil_div(a.K, kc);
  if (F32_CFGS[cfg].bm < 128 && S == 1 && !direct_ok(a)) cfg = 0;
  const F32Cfg& c = F32_CFGS[cfg];
  a.tiles_m = (uint32_t)ceil_div(a.M, (uint64_t)c.bm);
  a.tiles_n = (uint32_t)ceil_div(a.N, (uint64_t)c.bn);
  const uint64_t nb = (uint64_t)a.tiles_m * a.tiles_n;
  VKH_REQUIRE(nb < (uint64_t(1) << 31), "GEMM too large");
  // whole 4-element runs: contiguous extents (A: K unless transposed, else M;
  // B: N unless transposed, else K) that are multiples of 4
  const bool vec = (ta ? a.M : a.K) % 4 == 0 && (tb ? a.K : a.N) % 4 == 0;
  std::unique_lock<std::mutex> lock(g->pack_mu, std::defer_lock);
  if (S > 1) lock.lock();
  float* part = S > 1 ? reinterpret_cast<float*>(pack_area(g, f32_split_bytes(a.M, a.N, a.K))) : nullptr;
  c.launch(dim3((unsigned)nb, (unsigned)S), g->stream, a, ta, tb, vec, part, kc);
  check_launch("gemm");
  if (S > 1) {
    const uint64_t groups = a.M * ceil_div(a.N, 4);
    hipLaunchKernelGGL(k_splitk_combine, dim3(stream_grid(g, groups, 256, 8)), dim3(256), 0, g->stream,
                       (const float*)part, S, a);
    check_launch("gemm split-k combine");
  }
}

// ---- skinny products: min(M, N) <= 16 ------------------------------------------------
// C = op(A) op(B) with one small output dimension Q is a pass over the large
// operand (the Dense layer with one or ten outputs, its weight gradient):
// memory-bound, so it runs in FP32 on the vector units in every mode.  The
// problem is restated as out[p, q] = sum_k X[p, k] Y[k, q] with P the long
// output dimension; X is read once, Y (Q x K) stays in the caches.
//   row-dot      X K-contiguous: one wave per p, lanes along k, wave sums
//   column-walk  X p-contiguous: one thread per p, k chunks, partial sums
//                combined in chunk order by a second kernel
struct SkinnyArgs {
  const float* X;
  const float* Y;
  uint64_t sxp, sxk, syk, syq, P, K;
  int Q;
  int swap;  // 1: p indexes columns n of C and q rows m
  GemmArgs e;
};

__device__ __forceinline__ void skinny_store(const SkinnyArgs& a, uint64_t p, int q, float acc) {
  const GemmArgs& e = a.e;
  const uint64_t m = a.swap ? (uint64_t)q : p, n = a.swap ? p : (uint64_t)q;
  float* cp = e.C + m * e.ldc + n;
  float v = e.alpha * acc;
  if (e.beta != 0.f) v += e.beta * *cp;
  if (e.bias) v += e.bias[n];
  v = act_apply(e.act, v);
  if (e.aux) v = act_deriv_mul(e.aux_act, e.aux[m * e.ldaux + n], v);
  if (e.aux16) v = act_deriv_mul(e.aux_act, bf2f(e.aux16[m * e.ldaux + n]), v);
  if (!e.no_c) *cp = v;
  if (e.Cbf) e.Cbf[m * e.ldc + n] = f2bf(v);
  if (e.Cbft) e.Cbft[n * e.ldt + m] = f2bf(v);
}

__device__ __forceinline__ float wave_sum64(float v) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

template <int QB>
__global__ void __launch_bounds__(256) k_skinny_rowdot(SkinnyArgs a, int vec) {
  const uint64_t p = (uint64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (p >= a.P) return;  // uniform per wave
  float acc[QB];
#pragma unroll
  for (int q = 0; q < QB; ++q) acc[q] = 0.f;
  const float* xr = a.X + p * a.sxp;
  if (vec) {  // X rows and Y columns 16-byte aligned, K % 4 == 0, Y K-contiguous
    for (uint64_t k = (uint64_t)lane * 4; k < a.K; k += 256) {
      const float4 x = *reinterpret_cast<const float4*>(xr + k);
#pragma unroll
      for (int q = 0; q < QB; ++q) {
        if (q < a.Q) {
          const float4 y = *reinterpret_cast<const float4*>(a.Y + q * a.syq + k);
          acc[q] += x.x * y.x;
          acc[q] += x.y * y.y;
          acc[q] += x.z * y.z;
          acc[q] += x.w * y.w;
        }
      }
    }
  } else {
    for (uint64_t k = lane; k < a.K; k += 64) {
      const float x = xr[k];
#pragma unroll
      for (int q = 0; q < QB; ++q)
        if (q < a.Q) acc[q] += x * a.Y[k * a.syk + q * a.syq];
    }
  }
  float mine = 0.f;
#pragma unroll
  for (int q = 0; q < QB; ++q) {
    const float s = wave_sum64(acc[q]);
    if (lane == q) mine = s;
  }
  if (lane < a.Q) skinny_store(a, p, lane, mine);
}

// k_skinny_rowdot for Q = 1 with 16-byte operands and K = 256 * NK: the
// column of op(B) (K floats) is loaded into registers once per wave and a
// wave takes RW rows, so that only X is streamed; every row sums its k in the
// order of k_skinny_rowdot (lane-strided float4 steps, then the wave's
// butterfly)
constexpr int ROWDOT_RW = 4;
template <int NK>
__global__ void __launch_bounds__(256) k_skinny_rowdot1(SkinnyArgs a) {
  const int lane = threadIdx.x & 63;
  const uint64_t p0 = ((uint64_t)blockIdx.x * 4 + (threadIdx.x >> 6)) * ROWDOT_RW;
  if (p0 >= a.P) return;  // uniform per wave
  float4 y[NK];
#pragma unroll
  for (int i = 0; i < NK; ++i) y[i] = *reinterpret_cast<const float4*>(a.Y + lane * 4 + i * 256);
  for (int rw = 0; rw < ROWDOT_RW; ++rw) {
    const uint64_t p = p0 + rw;
    if (p >= a.P) break;
    const float* xr = a.X + p * a.sxp;
    float4 x[NK];
#pragma unroll
    for (int i = 0; i < NK; ++i) x[i] = ld_stream(reinterpret_cast<const float4*>(xr + lane * 4 + i * 256));
    float acc = 0.f;
#pragma unroll
    for (int i = 0; i < NK; ++i) {
      acc += x[i].x * y[i].x;
      acc += x[i].y * y[i].y;
      acc += x[i].z * y[i].z;
      acc += x[i].w * y[i].w;
    }
    const float s = wave_sum64(acc);
    if (lane == 0) skinny_store(a, p, 0, s);
  }
}

// partial sums part[chunk][q][p] over k in [chunk*kchunk, (chunk+1)*kchunk);
// VW consecutive p per thread (VW = 4: 16-byte loads, P % 4 == 0 and X rows
// 16-byte aligned)
template <int QB, int VW>
__global__ void __launch_bounds__(256)
k_skinny_colwalk(SkinnyArgs a, uint64_t kchunk, float* part) {
  const uint64_t p = ((uint64_t)blockIdx.x * 256 + threadIdx.x) * VW;
  const uint64_t chunk = blockIdx.y;
  const bool in = p < a.P;
  const uint64_t k0 = chunk * kchunk, k1 = min(a.K, k0 + kchunk);
  float acc[QB][VW];
#pragma unroll
  for (int q = 0; q < QB; ++q)
#pragma unroll
    for (int w = 0; w < VW; ++w) acc[q][w] = 0.f;
  auto load_x = [&](uint64_t k, float (&x)[VW]) {
    if constexpr (VW == 4) {
      const float4 t = *reinterpret_cast<const float4*>(a.X + k * a.sxk + p);
      x[0] = t.x; x[1] = t.y; x[2] = t.z; x[3] = t.w;
    } else {
      x[0] = a.X[k * a.sxk + p];
    }
  };
  constexpr int U = 8;  // terms of X requested at a time, before the first sum
  if constexpr (QB == 1) {
    if (!in) return;
    uint64_t k = k0;
    for (; k + U <= k1; k += U) {
      float x[U][VW], y[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        load_x(k + u, x[u]);
        y[u] = a.Y[(k + u) * a.syk];
      }
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int w = 0; w < VW; ++w) acc[0][w] += x[u][w] * y[u];
    }
    for (; k < k1; ++k) {
      float x[VW];
      load_x(k, x);
      const float y = a.Y[k * a.syk];
#pragma unroll
      for (int w = 0; w < VW; ++w) acc[0][w] += x[w] * y;
    }
  } else {
    // Segments of KS terms, Y's read into LDS by the whole block.  (With Y read by
    // every thread itself, a scalar load for each term and output, 4096 x 16
    // outputs over 4096 terms took 79 us, 35 now; one output is faster without
    // LDS: 4096 x 1 over 1024 terms 9.8 against 13.6.)
    constexpr int KS = 64;
    __shared__ __attribute__((aligned(16))) float ys[KS * QB];
    for (uint64_t s0 = k0; s0 < k1; s0 += KS) {
      const int n = (int)min<uint64_t>(KS, k1 - s0);
      float r[(KS * QB + 255) / 256];
#pragma unroll
      for (int u = 0; u < (KS * QB + 255) / 256; ++u) {
        const int t = min((int)threadIdx.x + u * 256, n * QB - 1);
        r[u] = a.Y[(s0 + t / QB) * a.syk + min(t % QB, a.Q - 1) * a.syq];
      }
      if (s0 > k0) __syncthreads();
#pragma unroll
      for (int u = 0; u < (KS * QB + 255) / 256; ++u)
        if ((int)threadIdx.x + u * 256 < KS * QB) ys[threadIdx.x + u * 256] = r[u];
      __syncthreads();
      if (!in) continue;
      for (int i = 0; i < n; i += U) {
        float x[U][VW];
#pragma unroll
        for (int u = 0; u < U; ++u) load_x(s0 + min(i + u, n - 1), x[u]);
#pragma unroll
        for (int u = 0; u < U; ++u)
          if (i + u < n)
#pragma unroll
            for (int q = 0; q < QB; ++q)
#pragma unroll
              for (int w = 0; w < VW; ++w) acc[q][w] += x[u][w] * ys[(i + u) * QB + q];
      }
    }
  }
  if (!in) return;
#pragma unroll
  for (int q = 0; q < QB; ++q)
    if (q < a.Q)
#pragma unroll
      for (int w = 0; w < VW; ++w) part[(chunk * a.Q + q) * a.P + p + w] = acc[q][w];
}

__global__ void __launch_bounds__(256)
k_skinny_combine(SkinnyArgs a, const float* part, uint64_t nchunk) {
  const uint64_t total = a.P * (uint64_t)a.Q;
  const uint64_t stride = (uint64_t)gridDim.x * 256;
  for (uint64_t t = (uint64_t)blockIdx.x * 256 + threadIdx.x; t < total; t += stride) {
    const int q = (int)(t / a.P);
    const uint64_t p = t - (uint64_t)q * a.P;
    const uint64_t step = (uint64_t)a.Q * a.P;
    const float* pp = part + (uint64_t)q * a.P + p;
    float s = 0.f;
    uint64_t c = 0;
    for (; c + 8 <= nchunk; c += 8) {  // eight loads in flight, summed in chunk order
      float v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = pp[(c + u) * step];
#pragma unroll
      for (int u = 0; u < 8; ++u) s += v[u];
    }
    for (; c < nchunk; ++c) s += pp[c * step];
    skinny_store(a, p, q, s);
  }
}

// Column walk of few outputs over few chunks (the weight gradient of a narrow
// layer) in one launch: a block takes 64 p and up to 4 q, a wave a chunk (its
// terms added in k order from 0; X requested 32 terms at once, Y's columns read
// into LDS by the whole block first), then the chunks' sums, kept in LDS, are added
// in order from 0 as k_skinny_combine adds them: the same bits. What bounds it
// is the latency of the loads. 32 x 3 outputs over 150 terms 6.5 us (column walk
// and combine 15), 1024 x 16 over 1024 terms 10 (73), over 2048 terms 15.5 (73).
constexpr uint64_t WALK_P = 2048, WALK_CHUNKS = 32, WALK_TERMS = 64;
constexpr int WALK_Q = 4, WALK_U = 32;
__global__ void __launch_bounds__(1024)
k_skinny_walk(SkinnyArgs a, uint32_t kchunk, uint32_t nchunk) {
  extern __shared__ __attribute__((aligned(16))) float walk_lds[];
  float* parts = walk_lds;                         // [nchunk][WALK_Q][64]
  float* ys = walk_lds + nchunk * WALK_Q * 64;     // [K][WALK_Q]
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int waves = blockDim.x >> 6, q0 = blockIdx.y * WALK_Q;
  const uint32_t K = (uint32_t)a.K;
  const uint64_t p0 = (uint64_t)blockIdx.x * 64, pl = min(p0 + lane, a.P - 1);
  // (columns beyond Q read the last one)
  for (uint32_t t0 = threadIdx.x; t0 < K * WALK_Q; t0 += 8 * blockDim.x) {
    float r[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const uint32_t t = min(t0 + u * blockDim.x, K * WALK_Q - 1);
      r[u] = a.Y[(t / WALK_Q) * a.syk + min(q0 + (int)(t % WALK_Q), a.Q - 1) * a.syq];
    }
#pragma unroll
    for (int u = 0; u < 8; ++u)
      if (t0 + u * blockDim.x < K * WALK_Q) ys[t0 + u * blockDim.x] = r[u];
  }
  __syncthreads();
  for (uint32_t c = wave; c < nchunk; c += waves) {
    const uint32_t k0 = c * kchunk, k1 = min(K, k0 + kchunk);
    float acc[WALK_Q] = {0.f, 0.f, 0.f, 0.f};
    for (uint32_t k = k0; k < k1; k += WALK_U) {
      float x[WALK_U];
#pragma unroll
      for (int u = 0; u < WALK_U; ++u) x[u] = a.X[min(k + u, k1 - 1) * a.sxk + pl];  // (past the chunk: its last term)
#pragma unroll
      for (int u = 0; u < WALK_U; ++u)
        if (k + u < k1) {
          const f32x4_t y = *reinterpret_cast<const f32x4_t*>(ys + (k + u) * WALK_Q);
#pragma unroll
          for (int q = 0; q < WALK_Q; ++q) acc[q] += x[u] * y[q];
        }
    }
#pragma unroll
    for (int q = 0; q < WALK_Q; ++q) parts[(c * WALK_Q + q) * 64 + lane] = acc[q];
  }
  __syncthreads();
  for (int t = threadIdx.x; t < WALK_Q * 64; t += blockDim.x) {
    const int q = t >> 6;
    const uint64_t p = p0 + (t & 63);
    float s = 0.f;
#pragma unroll 8
    for (uint32_t c = 0; c < nchunk; ++c) s += parts[c * WALK_Q * 64 + t];
    if (p < a.P && q0 + q < a.Q) skinny_store(a, p, q0 + q, s);
  }
}

constexpr uint64_t SKINNY_MAX = 16;  // largest small dimension of the skinny path

// k per chunk (and the chunk count) of the column walk over P outputs and K
// terms: about 1024 threads per compute unit, at least 64 k per chunk; v4:
// four outputs per thread.  The chunks fix the summation order.
static uint64_t colwalk_chunk(vkh_gpu* g, uint64_t P, uint64_t K, bool v4, uint64_t& nchunk_out) {
  const uint64_t pthreads = v4 ? P / 4 : P;
  const uint64_t target = (uint64_t)(g->num_cus > 0 ? g->num_cus : 256) * 1024;
  uint64_t nchunk = std::max<uint64_t>(1, std::min<uint64_t>(ceil_div(target, pthreads), ceil_div(K, 64)));
  nchunk = std::min<uint64_t>(nchunk, 65535);
  const uint64_t kchunk = ceil_div(std::max<uint64_t>(K, 1), nchunk);
  nchunk_out = ceil_div(std::max<uint64_t>(K, 1), kchunk);
  return kchunk;
}

static void gemm_skinny(vkh_gpu* g, bool ta, bool tb, const GemmArgs& e) {
  SkinnyArgs a{};
  a.e = e;
  if (e.N <= e.M) {  // q = n, p = m: X = op(A), Y = op(B)
    a.swap = 0;
    a.P = e.M;
    a.Q = (int)e.N;
    a.X = e.A;
    a.sxp = ta ? 1 : e.lda;
    a.sxk = ta ? e.lda : 1;
    a.Y = e.B;
    a.syk = tb ? 1 : e.ldb;
    a.syq = tb ? e.ldb : 1;
  } else {  // q = m, p = n: X = op(B)^T, Y = op(A)^T
    a.swap = 1;
    a.P = e.N;
    a.Q = (int)e.M;
    a.X = e.B;
    a.sxp = tb ? e.ldb : 1;
    a.sxk = tb ? 1 : e.ldb;
    a.Y = e.A;
    a.syk = ta ? e.lda : 1;
    a.syq = ta ? 1 : e.lda;
  }
  a.K = e.K;
  const int qb = a.Q <= 1 ? 1 : a.Q <= 2 ? 2 : a.Q <= 4 ? 4 : a.Q <= 8 ? 8 : 16;
  if (a.sxk == 1) {
    const int vec = ((uintptr_t)a.X & 15u) == 0 && a.sxp % 4 == 0 && a.K % 4 == 0 && a.syk == 1 &&
                    ((uintptr_t)a.Y & 15u) == 0 && a.syq % 4 == 0;
    if (qb == 1 && vec && a.K % 256 == 0 && a.K >= 1024 && a.K <= 4096) {
      const unsigned blocks1 = (unsigned)ceil_div(a.P, (uint64_t)4 * ROWDOT_RW);
      switch (a.K / 256) {
#define VKH_ROWDOT1(NKV) case NKV: hipLaunchKernelGGL(k_skinny_rowdot1<NKV>, dim3(blocks1), dim3(256), 0, g->stream, a); break;
        VKH_ROWDOT1(4) VKH_ROWDOT1(5) VKH_ROWDOT1(6) VKH_ROWDOT1(7) VKH_ROWDOT1(8) VKH_ROWDOT1(9) VKH_ROWDOT1(10)
        VKH_ROWDOT1(11) VKH_ROWDOT1(12) VKH_ROWDOT1(13) VKH_ROWDOT1(14) VKH_ROWDOT1(15) VKH_ROWDOT1(16)
#undef VKH_ROWDOT1
      }
      check_launch("gemm (skinny row-dot)");
      return;
    }
    const uint64_t blocks = ceil_div(a.P, 4);
    VKH_REQUIRE(blocks < (uint64_t(1) << 31), "GEMM too large");
    dim3 grid((unsigned)blocks), block(256);
    switch (qb) {
      case 1: hipLaunchKernelGGL(k_skinny_rowdot<1>, grid, block, 0, g->stream, a, vec); break;
      case 2: hipLaunchKernelGGL(k_skinny_rowdot<2>, grid, block, 0, g->stream, a, vec); break;
      case 4: hipLaunchKernelGGL(k_skinny_rowdot<4>, grid, block, 0, g->stream, a, vec); break;
      case 8: hipLaunchKernelGGL(k_skinny_rowdot<8>, grid, block, 0, g->stream, a, vec); break;
      default: hipLaunchKernelGGL(k_skinny_rowdot<16>, grid, block, 0, g->stream, a, vec); break;
    }
    check_launch("gemm (skinny row-dot)");
    return;
  }
  const bool v4 = a.P % 4 == 0 && ((uintptr_t)a.X & 15u) == 0 && a.sxk % 4 == 0;
  const uint64_t pthreads = v4 ? a.P / 4 : a.P;
  uint64_t nchunk = 0;
  const uint64_t kchunk = colwalk_chunk(g, a.P, a.K, v4, nchunk);
  // Few outputs, few short chunks: one launch.  Us of k_skinny_walk / column walk
  // and combine: 2048 x 4 over 512 terms 8.9 / 19, 64 x 4 over 2048 15 / 14, 64 x
  // 16 over 2048 15 / 30; one output 150 terms 6.5 / 7.7, 512 8.3 / 7.6, 2048
  // 15 / 8.8.  Past 32 chunks a block would walk them in turn.
  if (a.P <= WALK_P && nchunk <= WALK_CHUNKS && kchunk <= WALK_TERMS && (a.Q > 1 || nchunk <= 4)) {
    const unsigned waves = (unsigned)std::max<uint64_t>(4, std::min<uint64_t>(16, nchunk));
    hipLaunchKernelGGL(k_skinny_walk, dim3((unsigned)ceil_div(a.P, 64), (unsigned)ceil_div(a.Q, WALK_Q)), dim3(64 * waves),
                       sizeof(float) * WALK_Q * (nchunk * 64 + a.K), g->stream, a, (uint32_t)kchunk, (uint32_t)nchunk);
    check_launch("gemm (skinny walk)");
    return;
  }
  Workspace ws(g, sizeof(float) * nchunk * (uint64_t)a.Q * a.P);
  float* part = (float*)ws.get();
  const uint64_t bx = ceil_div(pthreads, 256);
  VKH_REQUIRE(bx < (uint64_t(1) << 31), "GEMM too large");
  dim3 grid((unsigned)bx, (unsigned)nchunk), block(256);
#define VKH_COLWALK(QB)                                                                                 \
  do {                                                                                                  \
    if (v4) hipLaunchKernelGGL((k_skinny_colwalk<QB, 4>), grid, block, 0, g->stream, a, kchunk, part); \
    else hipLaunchKernelGGL((k_skinny_colwalk<QB, 1>), grid, block, 0, g->stream, a, kchunk, part);    \
  } while (0)
  switch (qb) {
    case 1: VKH_COLWALK(1); break;
    case 2: VKH_COLWALK(2); break;
    case 4: VKH_COLWALK(4); break;
    case 8: VKH_COLWALK(8); break;
    default: VKH_COLWALK(16); break;
  }
#undef VKH_COLWALK
  check_launch("gemm (skinny column walk)");
  const uint64_t total = a.P * (uint64_t)a.Q;
  hipLaunchKernelGGL(k_skinny_combine, dim3(full_grid(total, 256)), dim3(256), 0, g->stream, a,
                     (const float*)part, nchunk);
  check_launch("gemm (skinny combine)");
}

// ---- helpers for the nn path -------------------------------------------------------------
__global__ void __launch_bounds__(256) k_to_bf16(const float* src, uint16_t* dst, uint64_t n) {
  const uint64_t stride = (uint64_t)gridDim.x * 256;
  for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += stride) dst[i] = f2bf(src[i]);
}

}  // namespace vkh

using namespace vkh;

extern "C" {

// ---- products with a short k: K <= SMALLK_MAX --------------------------------------
// C = op(A) op(B) with K of a few elements (the input gradient of a Dense
// layer with one or ten outputs) is a pass that writes C (and reads aux or
// beta * C): memory-bound, so like the skinny products it runs in FP32 on the
// vector units in every mode.  Thread (row m, columns n..n+3) sums
// op(A)[m, k] op(B)[k, n + q] over k in order and applies the GEMM epilogue.
constexpr uint64_t SMALLK_MAX = 16;

__global__ void __launch_bounds__(256)
k_gemm_smallk(GemmArgs e, uint64_t sam, uint64_t sak, uint64_t sbk, uint64_t sbn, int vb) {
  const uint64_t n = ((uint64_t)blockIdx.x * 256 + threadIdx.x) * 4;
  if (n >= e.N) return;
  const int K = (int)e.K;
  for (uint64_t m = blockIdx.y; m < e.M; m += gridDim.y) {
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
    for (int k = 0; k < K; ++k) {
      const float av = e.A[m * sam + k * sak];
      float bv[4];
      if (vb && n + 3 < e.N) {
        const float4 t = *reinterpret_cast<const float4*>(e.B + k * sbk + n);
        bv[0] = t.x; bv[1] = t.y; bv[2] = t.z; bv[3] = t.w;
      } else {
#pragma unroll
        for (int q = 0; q < 4; ++q) bv[q] = n + q < e.N ? e.B[k * sbk + (n + q) * sbn] : 0.f;
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) acc[q] = k == 0 ? av * bv[q] : acc[q] + av * bv[q];
    }
    epilogue4(e, m, n, make_float4(acc[0], acc[1], acc[2], acc[3]));
  }
}

static void gemm_smallk(vkh_gpu* g, bool ta, bool tb, const GemmArgs& a) {
  const uint64_t sam = ta ? 1 : a.lda, sak = ta ? a.lda : 1;
  const uint64_t sbk = tb ? 1 : a.ldb, sbn = tb ? a.ldb : 1;
  const int vb = !tb && ((uintptr_t)a.B & 15u) == 0 && a.ldb % 4 == 0;
  const uint64_t groups = ceil_div(a.N, 4);
  VKH_REQUIRE(ceil_div(groups, 256) < (uint64_t(1) << 31), "gemm: N too large");
  dim3 grid((unsigned)ceil_div(groups, 256), (unsigned)std::min<uint64_t>(a.M, 65535));
  hipLaunchKernelGGL(k_gemm_smallk, grid, dim3(256), 0, g->stream, a, sam, sak, sbk, sbn, vb);
  check_launch("gemm (small k)");
}

// ---- backward of a one-output Dense layer after an activation ---------------------
// For a last layer y = h w^T + b with w [1, N] and h = act(z) [B, N], one pass
// over h produces everything its backward and the previous layer's bias
// gradient need, with the bits of the separate steps:
//   dx[b, n] = act'(h[b, n]) * (dy[b] * w[n])    (vkh_gemm, K = 1, aux = h)
//   dx_bf, dx_bft: dx as BF16, row-major and transposed (the next products'
//                  packed operands); the FP32 dx is not stored when dx is null
//   dw[n]    = sum_b h[b, n] * dy[b]             (the column walk of vkh_gemm
//                  for dY^T h: 0 + products in k order per chunk of kc_dw rows,
//                  chunks summed in order from 0)
//   db[n]    = sum_b dx[b, n]                    (vkh_bias_grad: per chunk of
//                  kc_db rows in row order from its first element, chunks
//                  summed in order)
// A block stages a 128-row x 32-column tile of dx and of h in LDS (33 KB, four
// blocks a compute unit); the chunk sums walk its columns and the transposed
// copy leaves in 256-byte runs (16 bytes a lane).  kc_dw and kc_db divide 128.
// Each block takes a column of tiles in turn, with the next tile's loads in
// flight during the current tile's column walks and stores.
constexpr int D1_TR = 128, D1_TC = 32, D1_PITCH = D1_TC + 1;  // odd pitch: column walks conflict-free
constexpr int D1_LOADS = D1_TR * D1_TC / 4 / 256;                 // float4 loads of h a thread

__global__ void __launch_bounds__(256)
k_dense1_backward(const float* __restrict__ dy, const float* __restrict__ w, const float* __restrict__ h,
                  int act, uint64_t N, uint64_t row_tiles, float* __restrict__ dx,
                  uint16_t* __restrict__ dx_bf, uint16_t* __restrict__ dx_bft, uint64_t ldt,
                  float* __restrict__ part_dw, int kc_dw, float* __restrict__ part_db, int kc_db) {
  __shared__ float D[D1_TR * D1_PITCH], H[D1_TR * D1_PITCH], Y[D1_TR];
  const uint64_t n0 = (uint64_t)blockIdx.x * D1_TC;
  const int t = threadIdx.x, c4 = t % (D1_TC / 4), r0 = t / (D1_TC / 4);
  const uint64_t n = n0 + c4 * 4;
  const float4 wv = *reinterpret_cast<const float4*>(w + n);
  const float wq[4] = {wv.x, wv.y, wv.z, wv.w};
  const int ndb = part_db ? D1_TR / kc_db : 0, ndw = part_dw ? D1_TR / kc_dw : 0;
  // the block walks row tiles blockIdx.y, + gridDim.y, ...; each tile's
  // loads are issued before the previous tile's column walks and
  // transposed stores, so they are in flight meanwhile
  float4 hv[D1_LOADS];
  float d[D1_LOADS], yv = 0.f;
  auto load_tile = [&](uint64_t tile) {
    const uint64_t b0 = tile * D1_TR;
#pragma unroll
    for (int it = 0; it < D1_LOADS; ++it) {
      const uint64_t b = b0 + r0 + it * (256 / (D1_TC / 4));
      hv[it] = ld_stream(reinterpret_cast<const float4*>(h + b * N + n));
      d[it] = dy[b];
    }
    if (t < D1_TR) yv = dy[b0 + t];
  };
  uint64_t tile = blockIdx.y;
  if (tile < row_tiles) load_tile(tile);
  for (; tile < row_tiles; tile += gridDim.y) {
    const uint64_t b0 = tile * D1_TR;
    if (t < D1_TR) Y[t] = yv;
#pragma unroll
    for (int it = 0; it < D1_LOADS; ++it) {
      const int r = r0 + it * (256 / (D1_TC / 4));
      const uint64_t b = b0 + r;
      const float hq[4] = {hv[it].x, hv[it].y, hv[it].z, hv[it].w};
      float o[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        o[q] = act_deriv_mul(act, hq[q], d[it] * wq[q]);
        D[r * D1_PITCH + c4 * 4 + q] = o[q];
        H[r * D1_PITCH + c4 * 4 + q] = hq[q];
      }
      if (dx) st_stream(reinterpret_cast<float4*>(dx + b * N + n), make_float4(o[0], o[1], o[2], o[3]));
      if (dx_bf) {
        uint2 hb;
        hb.x = f2bf(o[0]) | ((uint32_t)f2bf(o[1]) << 16);
        hb.y = f2bf(o[2]) | ((uint32_t)f2bf(o[3]) << 16);
        *reinterpret_cast<uint2*>(dx_bf + b * N + n) = hb;
      }
    }
    __syncthreads();
    if (tile + gridDim.y < row_tiles) load_tile(tile + gridDim.y);
    // chunk sums: one thread per (chunk, column), rows in order (each sum a
    // chain of dependent adds; its LDS reads go out 8 at a time)
    for (int item = t; item < (ndb + ndw) * D1_TC; item += 256) {
      const int col = item % D1_TC, j = item / D1_TC;
      if (j < ndb) {
        const int rs = j * kc_db;
        float acc = D[rs * D1_PITCH + col];
        int r = 1;
        for (; r + 8 <= kc_db; r += 8) {
          float v[8];
#pragma unroll
          for (int q = 0; q < 8; ++q) v[q] = D[(rs + r + q) * D1_PITCH + col];
#pragma unroll
          for (int q = 0; q < 8; ++q) acc = acc + v[q];
        }
        for (; r < kc_db; ++r) acc = acc + D[(rs + r) * D1_PITCH + col];
        part_db[(b0 / kc_db + j) * N + n0 + col] = acc;
      } else {
        const int rs = (j - ndb) * kc_dw;
        float acc = 0.f;
        int r = 0;
        for (; r + 8 <= kc_dw; r += 8) {
          float v[8];
#pragma unroll
          for (int q = 0; q < 8; ++q) v[q] = H[(rs + r + q) * D1_PITCH + col] * Y[rs + r + q];
#pragma unroll
          for (int q = 0; q < 8; ++q) acc += v[q];
        }
        for (; r < kc_dw; ++r) acc += H[(rs + r) * D1_PITCH + col] * Y[rs + r];
        part_dw[(b0 / kc_dw + j - ndb) * N + n0 + col] = acc;
      }
    }
    if (dx_bft) {
      // D1_TC columns x 16 runs of 8 rows; 16 consecutive lanes continue one column
      for (int item = t; item < D1_TC * (D1_TR / 8); item += 256) {
        const int col = item / (D1_TR / 8), seg = item % (D1_TR / 8);
        uint32_t wd[4];
#pragma unroll
        for (int q = 0; q < 4; ++q)
          wd[q] = f2bf(D[(seg * 8 + 2 * q) * D1_PITCH + col]) |
                  ((uint32_t)f2bf(D[(seg * 8 + 2 * q + 1) * D1_PITCH + col]) << 16);
        *reinterpret_cast<uint4*>(dx_bft + (n0 + col) * ldt + b0 + seg * 8) =
            make_uint4(wd[0], wd[1], wd[2], wd[3]);
      }
    }
    __syncthreads();  // D, H and Y are read before the next tile writes them
  }
}

// chunk lengths of the separate steps (dw: the column walk over N outputs and
// B terms; db: vkh_bias_grad's column sums); false where they do not tile the
// kernel's 128 rows
static bool dense1_chunks(vkh_gpu* g, uint64_t B, uint64_t N, uint64_t& kc_dw, uint64_t& ndw, uint64_t& kc_db) {
  if (B == 0 || B % D1_TR != 0 || N % D1_TC != 0 || B / D1_TR >= 65536 || N / D1_TC >= (uint64_t(1) << 31))
    return false;
  kc_dw = colwalk_chunk(g, N, B, true, ndw);
  kc_db = bias_grad_chunk(g, B, N);
  return kc_db > 0 && kc_dw <= (uint64_t)D1_TR && D1_TR % kc_dw == 0 && kc_db <= (uint64_t)D1_TR && D1_TR % kc_db == 0;
}

static void gemm_impl(vkh_gpu* g, int mode, int trans_a, int trans_b, uint64_t M, uint64_t N,
                      uint64_t K, float alpha, const float* A, uint64_t lda, const float* B,
                      uint64_t ldb, float beta, float* Cp, uint64_t ldc, const float* bias, int act,
                      uint16_t* c_bf16, const float* aux, uint64_t ldaux, int aux_act,
                      const uint16_t* a_bf16 = nullptr, const uint16_t* b_bf16 = nullptr,
                      uint16_t* c_bf16t = nullptr, uint64_t ldt = 0, float* cs = nullptr,
                      int no_c = 0, const uint16_t* aux16 = nullptr) {
  use(g);
  if (M == 0 || N == 0) return;
  VKH_REQUIRE(Cp || no_c, "gemm: null C");
  VKH_REQUIRE(!(aux && aux16), "gemm: aux given twice");
  VKH_REQUIRE(!aux16 || aux_act == VKH_ACT_RELU, "gemm: a BF16 aux is for ReLU' only");
  VKH_REQUIRE(K == 0 || (A && B), "gemm: null operand");
  VKH_REQUIRE(ldc >= N, "gemm: ldc < N");
  VKH_REQUIRE(trans_a ? lda >= M : lda >= K, "gemm: lda too small");
  VKH_REQUIRE(trans_b ? ldb >= K : ldb >= N, "gemm: ldb too small");
  VKH_REQUIRE(act >= VKH_ACT_NONE && act <= VKH_ACT_SIGMOID, "gemm: unknown activation");
  VKH_REQUIRE(aux_act >= VKH_ACT_NONE && aux_act <= VKH_ACT_SIGMOID, "gemm: unknown aux activation");
  VKH_REQUIRE(!(aux || aux16) || ldaux >= N, "gemm: ldaux < N");
  VKH_REQUIRE(!c_bf16t || ldt >= M, "gemm: ldt < M");
  VKH_REQUIRE(!c_bf16t || ((uintptr_t)c_bf16t & 1u) == 0, "gemm: c_bf16t not 2-byte aligned");
  VKH_REQUIRE(!a_bf16 || ((uintptr_t)a_bf16 & 15u) == 0, "gemm: a_bf16 not 16-byte aligned");
  VKH_REQUIRE(!b_bf16 || ((uintptr_t)b_bf16 & 15u) == 0, "gemm: b_bf16 not 16-byte aligned");
  GemmArgs a{};
  a.A = A; a.B = B; a.C = Cp; a.bias = bias; a.Cbf = c_bf16;
  a.M = M; a.N = N; a.K = K; a.lda = lda; a.ldb = ldb; a.ldc = ldc;
  a.alpha = alpha; a.beta = beta; a.act = act;
  a.aux = aux; a.ldaux = ldaux; a.aux_act = aux_act;
  a.Cbft = c_bf16t; a.ldt = ldt;
  a.cs = cs; a.no_c = no_c; a.aux16 = aux16;
  VKH_REQUIRE(!no_c || beta == 0.0f, "gemm: beta * C needs C");
  a.vec_c = ((uintptr_t)Cp & 15u) == 0 && ldc % 4 == 0 && (!bias || ((uintptr_t)bias & 15u) == 0) &&
            (!aux || (((uintptr_t)aux & 15u) == 0 && ldaux % 4 == 0)) &&
            (!aux16 || (((uintptr_t)aux16 & 7u) == 0 && ldaux % 4 == 0)) &&
            (!c_bf16 || ((uintptr_t)c_bf16 & 7u) == 0);
  VKH_REQUIRE(mode >= VKH_GEMM_FP32 && mode <= VKH_GEMM_BF16X3, "gemm: unknown mode");
  if (std::min(M, N) <= SKINNY_MAX && K > 0) {
    gemm_skinny(g, trans_a, trans_b, a);
    return;
  }
  if (K <= SMALLK_MAX) {
    gemm_smallk(g, trans_a, trans_b, a);
    return;
  }
  switch (mode) {
    case VKH_GEMM_FP32: {
      gemm_f32(g, trans_a, trans_b, a, product_cfg(g, mode, trans_a, trans_b, M, N, K, cs != nullptr));
      break;
    }
    case VKH_GEMM_BF16:
    case VKH_GEMM_BF16X3: {
      const bool pre = mode == VKH_GEMM_BF16 && K % PK_KALIGN == 0;
      gemm_packed(g, mode, trans_a, trans_b, a, product_cfg(g, mode, trans_a, trans_b, M, N, K, cs != nullptr),
                  pre ? a_bf16 : nullptr, pre ? b_bf16 : nullptr);
      break;
    }
    default: fail(VKH_INVALID, "gemm: unknown mode");
  }
}

int vkh_gemm_configs(int mode, int* count) {
  return guarded([&] {
    VKH_REQUIRE(count, "null out");
    VKH_REQUIRE(mode >= VKH_GEMM_FP32 && mode <= VKH_GEMM_BF16X3, "unknown mode");
    *count = mode_cfgs(mode);
  });
}

int vkh_gemm_config_info(int mode, int index, int* bm, int* bn, int* bk, int* waves, int* direct) {
  return guarded([&] {
    VKH_REQUIRE(bm && bn && bk && waves, "null out");
    VKH_REQUIRE(mode >= VKH_GEMM_FP32 && mode <= VKH_GEMM_BF16X3, "unknown mode");
    if (mode == VKH_GEMM_FP32) {
      VKH_REQUIRE(index >= 0 && index < F32_NCFG, "configuration index out of range");
      const F32Cfg& c = F32_CFGS[index];
      *bm = c.bm; *bn = c.bn; *bk = F32_BK; *waves = c.waves;
      if (direct) *direct = 0;
      return;
    }
    int n = 0;
    const PackedCfg* c = packed_cfgs(mode, n);
    VKH_REQUIRE(index >= 0 && index < n, "configuration index out of range");
    *bm = c[index].bm; *bn = c[index].bn; *bk = c[index].bk; *waves = c[index].waves;
    if (direct) *direct = 1;  // (operand slices from global memory straight into LDS)
  });
}

int vkh_gemm_get_config(vkh_gpu* g, int mode, int trans_a, int trans_b, uint64_t M, uint64_t N,
                        uint64_t K, int* index, int* tuned) {
  return guarded([&] {
    VKH_REQUIRE(g && index, "null argument");
    VKH_REQUIRE(mode >= VKH_GEMM_FP32 && mode <= VKH_GEMM_BF16X3, "unknown mode");
    auto it = g->gemm_cfg.find(cfg_key(mode, trans_a, trans_b, M, N, K));
    const bool have = it != g->gemm_cfg.end();
    *index = have ? it->second : default_cfg(mode, M, N, K);
    if (tuned) *tuned = have ? 1 : 0;
  });
}

int vkh_gemm_set_config(vkh_gpu* g, int mode, int trans_a, int trans_b, uint64_t M, uint64_t N,
                        uint64_t K, int index) {
  return guarded([&] {
    VKH_REQUIRE(g, "null GPU handle");
    VKH_REQUIRE(mode >= VKH_GEMM_FP32 && mode <= VKH_GEMM_BF16X3, "unknown mode");
    const int n = mode_cfgs(mode);
    const auto key = cfg_key(mode, trans_a, trans_b, M, N, K);
    if (index < 0) { g->gemm_cfg.erase(key); return; }
    VKH_REQUIRE(index < n, "configuration index out of range");
    g->gemm_cfg[key] = index;
  });
}

int vkh_gemm_autotune(vkh_gpu* g, int mode, int trans_a, int trans_b, uint64_t M, uint64_t N,
                      uint64_t K, int reps, int* best, float* ms_per_config) {
  return guarded([&] {
    use(g);
    VKH_REQUIRE(mode >= VKH_GEMM_FP32 && mode <= VKH_GEMM_BF16X3, "unknown mode");
    VKH_REQUIRE(!g->capturing, "gemm_autotune: not allowed during graph capture");
    VKH_REQUIRE(M > 0 && N > 0 && K > 0, "gemm_autotune: empty product");
    VKH_REQUIRE(g->alloc, "gemm_autotune needs a context with its own allocator");
    if (reps < 1) reps = 3;
    const int n = mode_cfgs(mode);
    const bool skinny = std::min(M, N) <= SKINNY_MAX || K <= SMALLK_MAX;
    if (skinny) {  // a single kernel choice
      if (ms_per_config)
        for (int i = 0; i < n; ++i) ms_per_config[i] = -1.0f;
      if (best) *best = default_cfg(mode, M, N, K);
      return;
    }
    // scratch operands in the product's own layout
    const uint64_t na = M * K, nbv = K * N, nc = M * N;
    Workspace wa(g, sizeof(float) * na), wb(g, sizeof(float) * nbv), wc(g, sizeof(float) * nc);
    float* A = (float*)wa.get();
    float* B = (float*)wb.get();
    float* C = (float*)wc.get();
    hipLaunchKernelGGL(k_fill_noise, dim3(full_grid(na, 256)), dim3(256), 0, g->stream, A, na, 1u);
    hipLaunchKernelGGL(k_fill_noise, dim3(full_grid(nbv, 256)), dim3(256), 0, g->stream, B, nbv, 2u);
    check_launch("gemm_autotune fill");
    GemmArgs a{};
    a.A = A; a.B = B; a.C = C;
    a.M = M; a.N = N; a.K = K;
    a.lda = trans_a ? M : K; a.ldb = trans_b ? K : N; a.ldc = N;
    a.alpha = 1.0f; a.beta = 0.0f; a.act = VKH_ACT_NONE; a.aux_act = VKH_ACT_NONE;
    a.vec_c = 1;
    // BF16: the operands packed once, padded for the largest tile (which
    // every configuration accepts), so that only the product is timed (the
    // packing passes are the same for every configuration)
    const bool pre = mode == VKH_GEMM_BF16;
    const uint64_t Kp = ceil_div(K, PK_KALIGN) * PK_KALIGN;
    const uint64_t Mp = ceil_div(M, PK_MAXTILE) * PK_MAXTILE, Np = ceil_div(N, PK_MAXTILE) * PK_MAXTILE;
    Workspace wpa(g, pre ? sizeof(uint16_t) * Mp * Kp : 1), wpb(g, pre ? sizeof(uint16_t) * Np * Kp : 1);
    uint16_t* pa = pre ? (uint16_t*)wpa.get() : nullptr;
    uint16_t* pb = pre ? (uint16_t*)wpb.get() : nullptr;
    if (pre) {
      pack_operand<1>(g, A, a.lda, trans_a, M, K, pa, Mp, Kp);
      pack_operand<1>(g, B, a.ldb, !trans_b, N, K, pb, Np, Kp);
    }
    hipEvent_t e0, e1;
    VKH_HIP(hipEventCreate(&e0));
    VKH_HIP(hipEventCreate(&e1));
    int bi = -1;
    float bt = 0.0f;
    try {
      auto run = [&](int i) {
        GemmArgs t = a;
        if (mode == VKH_GEMM_FP32) gemm_f32(g, trans_a, trans_b, t, i);
        else gemm_packed(g, mode, trans_a, trans_b, t, i, pa, pb);
      };
      for (int i = 0; i < n; ++i) {
        run(i);  // warm-up (and packing-area growth)
        VKH_HIP(hipEventRecord(e0, g->stream));
        for (int r = 0; r < reps; ++r) run(i);
        VKH_HIP(hipEventRecord(e1, g->stream));
        VKH_HIP(hipEventSynchronize(e1));
        float ms = 0.0f;
        VKH_HIP(hipEventElapsedTime(&ms, e0, e1));
        ms /= (float)reps;
        if (ms_per_config) ms_per_config[i] = ms;
        if (bi < 0 || ms < bt) { bi = i; bt = ms; }
      }
    } catch (...) {
      (void)hipEventDestroy(e0);
      (void)hipEventDestroy(e1);
      throw;
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    g->gemm_cfg[cfg_key(mode, trans_a, trans_b, M, N, K)] = bi;
    if (best) *best = bi;
  });
}

int vkh_gemm_autotune_ext(vkh_gpu* g, int mode, int trans_a, int trans_b, uint64_t M, uint64_t N, uint64_t K,
                          float alpha, const float* A, uint64_t lda, const float* B, uint64_t ldb, float beta,
                          float* Cp, uint64_t ldc, const float* bias, int act, uint16_t* c_bf16,
                          const float* aux, const uint16_t* aux_bf16, uint64_t ldaux, int aux_act,
                          const uint16_t* a_bf16, const uint16_t* b_bf16, uint16_t* c_bf16t, uint64_t ldt,
                          float* db, int store_c, int reps, int* best, float* ms_per_config) {
  return guarded([&] {
    use(g);
    VKH_REQUIRE(mode >= VKH_GEMM_FP32 && mode <= VKH_GEMM_BF16X3, "unknown mode");
    VKH_REQUIRE(!g->capturing, "gemm_autotune: not allowed during graph capture");
    VKH_REQUIRE(M > 0 && N > 0 && K > 0, "gemm_autotune: empty product");
    if (reps < 1) reps = 3;
    (void)db;  // the column sums are not part of the timing
    const int n = mode_cfgs(mode);
    const auto key = cfg_key(mode, trans_a, trans_b, M, N, K);
    // the call's own epilogue; without its column sums an unstored C would
    // leave no output, so then C is stored
    const int no_c = (store_c || !(c_bf16 || c_bf16t)) ? 0 : 1;
    auto run = [&] {
      gemm_impl(g, mode, trans_a, trans_b, M, N, K, alpha, A, lda, B, ldb, beta, Cp, ldc, bias, act, c_bf16, aux,
                ldaux, aux_act, a_bf16, b_bf16, c_bf16t, ldt, nullptr, no_c, aux_bf16);
    };
    if (std::min(M, N) <= SKINNY_MAX || K <= SMALLK_MAX) {  // a single kernel choice
      if (ms_per_config)
        for (int i = 0; i < n; ++i) ms_per_config[i] = -1.0f;
      if (best) *best = default_cfg(mode, M, N, K);
      return;
    }
    hipEvent_t e0, e1;
    VKH_HIP(hipEventCreate(&e0));
    VKH_HIP(hipEventCreate(&e1));
    int bi = -1;
    float bt = 0.0f;
    try {
      for (int i = 0; i < n; ++i) {
        g->gemm_cfg[key] = i;
        run();  // warm-up (and packing-area growth)
        VKH_HIP(hipEventRecord(e0, g->stream));
        for (int r = 0; r < reps; ++r) run();
        VKH_HIP(hipEventRecord(e1, g->stream));
        VKH_HIP(hipEventSynchronize(e1));
        float ms = 0.0f;
        VKH_HIP(hipEventElapsedTime(&ms, e0, e1));
        ms /= (float)reps;
        if (ms_per_config) ms_per_config[i] = ms;
        if (bi < 0 || ms < bt) { bi = i; bt = ms; }
      }
    } catch (...) {
      g->gemm_cfg.erase(key);
      (void)hipEventDestroy(e0);
      (void)hipEventDestroy(e1);
      throw;
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    g->gemm_cfg[key] = bi;
    if (best) *best = bi;
  });
}

int vkh_gemm_reserve(vkh_gpu* g, int mode, uint64_t M, uint64_t N, uint64_t K) {
  return guarded([&] {
    use(g);
    VKH_REQUIRE(mode >= VKH_GEMM_FP32 && mode <= VKH_GEMM_BF16X3, "gemm_reserve: unknown mode");
    VKH_REQUIRE(!g->capturing, "gemm_reserve: not allowed during graph capture");
    // skinny and short-k products pack nothing; FP32 needs room only for
    // split-k partials
    if (M == 0 || N == 0 || std::min(M, N) <= SKINNY_MAX || K <= SMALLK_MAX) return;
    const size_t bytes = mode == VKH_GEMM_FP32 ? f32_split_bytes(M, N, K) : packed_bytes(mode, M, N, K);
    if (bytes == 0) return;
    std::lock_guard<std::mutex> lock(g->pack_mu);
    g->graph_pack_hint = std::max(g->graph_pack_hint, bytes);
    pack_area(g, bytes);
  });
}

int vkh_gemm(vkh_gpu* g, int mode, int trans_a, int trans_b, uint64_t M, uint64_t N, uint64_t K,
             float alpha, const float* A, uint64_t lda, const float* B, uint64_t ldb, float beta,
             float* Cp, uint64_t ldc, const float* bias, int act, uint16_t* c_bf16) {
  return guarded([&] {
    gemm_impl(g, mode, trans_a, trans_b, M, N, K, alpha, A, lda, B, ldb, beta, Cp, ldc, bias, act,
              c_bf16, nullptr, 0, VKH_ACT_NONE);
  });
}

int vkh_gemm_ex(vkh_gpu* g, int mode, int trans_a, int trans_b, uint64_t M, uint64_t N, uint64_t K,
                float alpha, const float* A, uint64_t lda, const float* B, uint64_t ldb, float beta,
                float* Cp, uint64_t ldc, const float* bias, int act, uint16_t* c_bf16,
                const float* aux, uint64_t ldaux, int aux_act) {
  return guarded([&] {
    gemm_impl(g, mode, trans_a, trans_b, M, N, K, alpha, A, lda, B, ldb, beta, Cp, ldc, bias, act,
              c_bf16, aux, ldaux, aux_act);
  });
}

int vkh_gemm_bf16a(vkh_gpu* g, int mode, int trans_a, int trans_b, uint64_t M, uint64_t N, uint64_t K,
                   float alpha, const float* A, uint64_t lda, const float* B, uint64_t ldb, float beta,
                   float* Cp, uint64_t ldc, const float* bias, int act, uint16_t* c_bf16,
                   const float* aux, uint64_t ldaux, int aux_act, const uint16_t* a_bf16) {
  return guarded([&] {
    gemm_impl(g, mode, trans_a, trans_b, M, N, K, alpha, A, lda, B, ldb, beta, Cp, ldc, bias, act,
              c_bf16, aux, ldaux, aux_act, a_bf16);
  });
}

int vkh_gemm_bf16io(vkh_gpu* g, int mode, int trans_a, int trans_b, uint64_t M, uint64_t N, uint64_t K,
                    float alpha, const float* A, uint64_t lda, const float* B, uint64_t ldb, float beta,
                    float* Cp, uint64_t ldc, const float* bias, int act, uint16_t* c_bf16,
                    const float* aux, uint64_t ldaux, int aux_act, const uint16_t* a_bf16,
                    const uint16_t* b_bf16, uint16_t* c_bf16t, uint64_t ldt) {
  return guarded([&] {
    gemm_impl(g, mode, trans_a, trans_b, M, N, K, alpha, A, lda, B, ldb, beta, Cp, ldc, bias, act,
              c_bf16, aux, ldaux, aux_act, a_bf16, b_bf16, c_bf16t, ldt);
  });
}

// Whether an M x N x K product takes C's column sums in its epilogue with
// vkh_bias_grad's bits: the matrix-core path, a configuration (tuned or
// default) whose waves hold 128-row slabs, no split k, and bias_grad's column
// sums chunked by 128 rows for [M, N].
static bool colsum_ok(vkh_gpu* g, int mode, int ta, int tb, uint64_t M, uint64_t N, uint64_t K) {
  if (std::min(M, N) <= SKINNY_MAX || K <= SMALLK_MAX) return false;
  if (mode < VKH_GEMM_FP32 || mode > VKH_GEMM_BF16X3) return false;
  if (bias_grad_chunk(g, M, N) != (uint64_t)CS_ROWS) return false;
  const int cfg = product_cfg(g, mode, ta, tb, M, N, K, true);
  if (mode == VKH_GEMM_FP32)
    return F32_CFGS[cfg].wm == CS_ROWS && ceil_div(K, f32_splitk_chunk(M, N, K)) == 1;
  int n = 0;
  const PackedCfg* c = packed_cfgs(mode, n);
  const uint64_t Kp = ceil_div(K, (uint64_t)PK_KALIGN) * PK_KALIGN;
  return c[cfg].wm == CS_ROWS && ceil_div(Kp, splitk_chunk(M, N, Kp)) == 1;
}

int vkh_gemm_colsum_supported(vkh_gpu* g, int mode, int trans_a, int trans_b, uint64_t M, uint64_t N,
                              uint64_t K, int* ok) {
  return guarded([&] {
    VKH_REQUIRE(g && ok, "gemm_colsum_supported: null argument");
    *ok = colsum_ok(g, mode, trans_a, trans_b, M, N, K) ? 1 : 0;
  });
}

// vkh_gemm_bf16io with the column sums of C (db, optional), the FP32 C
// optional (store_c) and the aux activation's output as BF16 (aux_bf16)
static void gemm_ext(vkh_gpu* g, int mode, int trans_a, int trans_b, uint64_t M, uint64_t N, uint64_t K,
                     float alpha, const float* A, uint64_t lda, const float* B, uint64_t ldb, float beta, float* Cp,
                     uint64_t ldc, const float* bias, int act, uint16_t* c_bf16, const float* aux,
                     const uint16_t* aux_bf16, uint64_t ldaux, int aux_act, const uint16_t* a_bf16,
                     const uint16_t* b_bf16, uint16_t* c_bf16t, uint64_t ldt, float* db, int store_c) {
  use(g);
  VKH_REQUIRE(store_c || c_bf16 || c_bf16t || db, "gemm: no output");
  if (!db) {
    gemm_impl(g, mode, trans_a, trans_b, M, N, K, alpha, A, lda, B, ldb, beta, Cp, ldc, bias, act, c_bf16, aux,
              ldaux, aux_act, a_bf16, b_bf16, c_bf16t, ldt, nullptr, store_c ? 0 : 1, aux_bf16);
    return;
  }
  VKH_REQUIRE(colsum_ok(g, mode, trans_a, trans_b, M, N, K), "gemm_colsum: shape or configuration not supported");
  const uint64_t nchunk = ceil_div(M, (uint64_t)CS_ROWS);
  Workspace ws(g, sizeof(float) * nchunk * N);
  gemm_impl(g, mode, trans_a, trans_b, M, N, K, alpha, A, lda, B, ldb, beta, Cp, ldc, bias, act, c_bf16, aux,
            ldaux, aux_act, a_bf16, b_bf16, c_bf16t, ldt, (float*)ws.get(), store_c ? 0 : 1, aux_bf16);
  sum_chunks(g, (const float*)ws.get(), db, N, nchunk);
}

int vkh_gemm_bf16io_colsum(vkh_gpu* g, int mode, int trans_a, int trans_b, uint64_t M, uint64_t N,
                           uint64_t K, float alpha, const float* A, uint64_t lda, const float* B, uint64_t ldb,
                           float beta, float* Cp, uint64_t ldc, const float* bias, int act, uint16_t* c_bf16,
                           const float* aux, uint64_t ldaux, int aux_act, const uint16_t* a_bf16,
                           const uint16_t* b_bf16, uint16_t* c_bf16t, uint64_t ldt, float* db, int store_c) {
  return guarded([&] {
    VKH_REQUIRE(db, "gemm_colsum: null db");
    gemm_ext(g, mode, trans_a, trans_b, M, N, K, alpha, A, lda, B, ldb, beta, Cp, ldc, bias, act, c_bf16, aux,
             nullptr, ldaux, aux_act, a_bf16, b_bf16, c_bf16t, ldt, db, store_c);
  });
}

int vkh_gemm_bf16io_ext(vkh_gpu* g, int mode, int trans_a, int trans_b, uint64_t M, uint64_t N, uint64_t K,
                        float alpha, const float* A, uint64_t lda, const float* B, uint64_t ldb, float beta,
                        float* Cp, uint64_t ldc, const float* bias, int act, uint16_t* c_bf16, const float* aux,
                        const uint16_t* aux_bf16, uint64_t ldaux, int aux_act, const uint16_t* a_bf16,
                        const uint16_t* b_bf16, uint16_t* c_bf16t, uint64_t ldt, float* db, int store_c) {
  return guarded([&] {
    gemm_ext(g, mode, trans_a, trans_b, M, N, K, alpha, A, lda, B, ldb, beta, Cp, ldc, bias, act, c_bf16, aux,
             aux_bf16, ldaux, aux_act, a_bf16, b_bf16, c_bf16t, ldt, db, store_c);
  });
}

int vkh_dense1_backward_supported(vkh_gpu* g, uint64_t B, uint64_t N, int* ok) {
  return guarded([&] {
    VKH_REQUIRE(g && ok, "dense1_backward_supported: null argument");
    uint64_t kc_dw = 0, ndw = 0, kc_db = 0;
    *ok = dense1_chunks(g, B, N, kc_dw, ndw, kc_db) ? 1 : 0;
  });
}

int vkh_dense1_backward(vkh_gpu* g, const float* dy, const float* w, const float* h, int act, uint64_t B,
                        uint64_t N, float* dx, uint16_t* dx_bf, uint16_t* dx_bft, uint64_t ldt, float* dw,
                        float* db) {
  return guarded([&] {
    use(g);
    VKH_REQUIRE(dy && w && h, "dense1_backward: null pointer");
    VKH_REQUIRE(act >= VKH_ACT_NONE && act <= VKH_ACT_SIGMOID, "dense1_backward: unknown activation");
    auto a16 = [](const void* p) { return ((uintptr_t)p & 15u) == 0; };
    VKH_REQUIRE(a16(w) && a16(h) && (!dx || a16(dx)), "dense1_backward: operands not 16-byte aligned");
    VKH_REQUIRE(!dx_bf || ((uintptr_t)dx_bf & 7u) == 0, "dense1_backward: dx_bf not 8-byte aligned");
    VKH_REQUIRE(!dx_bft || (a16(dx_bft) && ldt % 8 == 0 && ldt >= B), "dense1_backward: dx_bft layout");
    uint64_t kc_dw = 0, ndw = 0, kc_db = 0;
    VKH_REQUIRE(dense1_chunks(g, B, N, kc_dw, ndw, kc_db), "dense1_backward: shape not supported");
    const uint64_t ndb = B / kc_db;
    Workspace wdw(g, dw ? sizeof(float) * ndw * N : 1), wdb(g, db ? sizeof(float) * ndb * N : 1);
    float* pdw = dw ? (float*)wdw.get() : nullptr;
    float* pdb = db ? (float*)wdb.get() : nullptr;
    // about four blocks a compute unit, each walking B / 128 / gy row tiles
    const uint64_t col_tiles = N / D1_TC, row_tiles = B / D1_TR;
    const uint64_t gy = std::min<uint64_t>(row_tiles, std::max<uint64_t>(1, ceil_div(4 * (uint64_t)g->num_cus,
                                                                                      col_tiles)));
    dim3 grid((unsigned)col_tiles, (unsigned)gy);
    hipLaunchKernelGGL(k_dense1_backward, grid, dim3(256), 0, g->stream, dy, w, h, act, N, row_tiles, dx, dx_bf,
                       dx_bft, ldt, pdw, (int)kc_dw, pdb, (int)kc_db);
    check_launch("dense1_backward");
    // dw: the column walk's combine (0 + chunks in order; its 1 * sum is the sum)
    if (dw) sum_chunks_from_zero(g, (const float*)pdw, dw, N, ndw);
    if (db) sum_chunks(g, (const float*)pdb, db, N, ndb);
  });
}

int vkh_to_bf16(vkh_gpu* g, const float* src, uint16_t* dst, uint64_t n) {
  return guarded([&] {
    use(g);
    if (n == 0) return;
    VKH_REQUIRE(src && dst, "to_bf16: null pointer");
    unsigned grid = stream_grid(g, n, 256, 8);
    hipLaunchKernelGGL(k_to_bf16, dim3(grid), dim3(256), 0, g->stream, src, dst, n);
    check_launch("to_bf16");
  });
}

}  // extern "C"
