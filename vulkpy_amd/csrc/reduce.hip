// Reductions: full (F11/F12), axis (F13) and axis + rebroadcast (F14).
//
// The reference reduces an axis with one thread per output element looping
// sequentially over k (vulkpy/shader/sum_axis.comp:20-32) and the whole array
// with a tree of ceil(n/64) passes (vulkpy/vkarray.py:1246-1274).  Here:
//  * rows (post == 1): one block (long rows), 8 to 64 lanes (medium) or one
//    thread (short rows, through LDS) per output, 128-bit loads at any
//    alignment, wave shuffle + LDS tree;
//  * strided axes (post > 1): few columns take whole rows a block and a tree over
//    them; otherwise one thread per group of 4 columns loops sequentially over
//    k -- the reference order -- and, when that leaves the GPU under-occupied, k
//    is split into chunks whose partials are combined in chunk order by a
//    second kernel;
//  * full reductions: grid-stride FP64 accumulation per thread, FP64 block
//    tree, FP64 cross-block combine, one rounding to FP32 at the end.
#include "common.h"
#include "fastdiv.h"

namespace vkh {

// 16 bytes of memory at any 4-byte alignment. NT: nontemporal, which streams an
// operand that the 256 MB cache cannot hold next to others (128 MB and more) about
// 10% faster and reads one that it holds slower: column sums of 200000 x 999 134 /
// 148 us (with / without), of a gradient of 16384 x 4096 49 / 58, of 200000 x 17
// 12.8 / 9.1, rows of 100 x 100000 28 / 18.
typedef __attribute__((ext_vector_type(4), aligned(4))) float f32x4u_t;
template <bool NT>
__device__ __forceinline__ f32x4u_t ld4u(const float* p) {
  if constexpr (NT) return __builtin_nontemporal_load(reinterpret_cast<const f32x4u_t*>(p));
  return *reinterpret_cast<const f32x4u_t*>(p);
}
static bool streams(uint64_t elements) { return elements >= (uint64_t(128) << 20) / sizeof(float); }

// 16 bytes of global memory straight into LDS (lane i's at dst + 16 i)
template <bool NT>
__device__ __forceinline__ void load_lds16(const float* src, float* dst) {
#ifdef __HIP_DEVICE_COMPILE__  // (the host pass would drop the launch stub of a template that uses the builtin)
  __builtin_amdgcn_global_load_lds(src, dst, 16, 0, NT ? 2 : 0);  // (2: nt)
#endif
}

template <int OP, typename T>
struct Red;
template <typename T>
struct Red<VKH_RSUM, T> {
  static __device__ __forceinline__ T init() { return T(0); }
  static __device__ __forceinline__ T f(T a, T b) { return a + b; }
};
template <typename T>
struct Red<VKH_RPROD, T> {
  static __device__ __forceinline__ T init() { return T(1); }
  static __device__ __forceinline__ T f(T a, T b) { return a * b; }
};
template <typename T>
struct Red<VKH_RMAX, T> {
  static __device__ __forceinline__ T init() { return -__builtin_huge_valf(); }
  static __device__ __forceinline__ T f(T a, T b) { return (a >= b || a != a) ? a : b; }
};
template <typename T>
struct Red<VKH_RMIN, T> {
  static __device__ __forceinline__ T init() { return __builtin_huge_valf(); }
  static __device__ __forceinline__ T f(T a, T b) { return (a <= b || a != a) ? a : b; }
};

template <int OP, typename T>
__device__ __forceinline__ T wave_reduce(T v) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v = Red<OP, T>::f(v, __shfl_xor(v, off, 64));
  return v;
}

// Block-wide reduction; every thread gets the result.  BLOCK is a multiple of 64.
template <int OP, typename T, int BLOCK>
__device__ __forceinline__ T block_reduce(T v, T* lds) {
  v = wave_reduce<OP, T>(v);
  constexpr int NW = BLOCK / 64;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (NW == 1) return v;
  if (lane == 0) lds[w] = v;
  __syncthreads();
  T r = lds[0];
#pragma unroll
  for (int i = 1; i < NW; ++i) r = Red<OP, T>::f(r, lds[i]);
  __syncthreads();
  return r;
}

__device__ __forceinline__ float epilogue(float v, float mul, float dv) {
  if (mul != 1.0f) v = v * mul;
  if (dv != 1.0f) v = v / dv;
  return v;
}

// ---- rows: post == 1, reduce each contiguous row of length L -----------------
constexpr int ROW_BLOCK = 256;

// one block per row (long rows)
// U: 128-bit loads in flight per thread (4 or 8); each thread still combines
// its elements in index order, so U never changes the result
// (rows of any alignment: 16-byte groups, then the last L % 4 elements)
template <int OP, int U, bool NT>
__global__ void __launch_bounds__(ROW_BLOCK)
k_rows_block(const float* a, float* out, uint64_t rows, uint64_t L, int rebroadcast, float mul, float dv) {
  __shared__ float lds[ROW_BLOCK / 64];
  using R = Red<OP, float>;
  for (uint64_t r = blockIdx.x; r < rows; r += gridDim.x) {
    const float* row = a + r * L;
    float acc = R::init();
    const uint64_t L4 = L / 4;
    uint64_t i = threadIdx.x;
    // U loads in flight, combined in the same order as the plain loop
    for (; i + (U - 1) * ROW_BLOCK < L4; i += U * ROW_BLOCK) {
      f32x4u_t v[U];
#pragma unroll
      for (int q = 0; q < U; ++q) v[q] = ld4u<NT>(row + 4 * (i + q * ROW_BLOCK));
#pragma unroll
      for (int q = 0; q < U; ++q) acc = R::f(acc, R::f(R::f(v[q][0], v[q][1]), R::f(v[q][2], v[q][3])));
    }
    for (; i < L4; i += ROW_BLOCK) {
      const f32x4u_t v = ld4u<NT>(row + 4 * i);
      acc = R::f(acc, R::f(R::f(v[0], v[1]), R::f(v[2], v[3])));
    }
    if (threadIdx.x < L % 4) acc = R::f(acc, row[4 * L4 + threadIdx.x]);
    float res = epilogue(block_reduce<OP, float, ROW_BLOCK>(acc, lds), mul, dv);
    if (!rebroadcast) {
      if (threadIdx.x == 0) out[r] = res;
    } else {
      float* orow = out + r * L;
      for (uint64_t i = threadIdx.x; i < L4; i += ROW_BLOCK)
        *reinterpret_cast<f32x4u_t*>(orow + 4 * i) = f32x4u_t{res, res, res, res};
      if (threadIdx.x < L % 4) orow[4 * L4 + threadIdx.x] = res;
    }
  }
}

// Medium rows (64 <= L < ROWS_BLOCK_MIN_L): LPR lanes a row, each with up to
// NV 16-byte groups, all loaded before the first is combined (any alignment);
// the last L % 4 elements go to the row's first lanes.  A lane combines its
// groups in pairs too: no sum is longer than in a wave a row and 4-byte loads
// (rms error over 20000 random rows 0.97 to 1.02 of that one's from 64 to 512 columns, less
// beyond; up to 1.03 with the groups one after the other).  With a wave a row and
// 4-byte loads 1500000 x 75 took 224 us, the second step of every row with 11 of
// 64 lanes; 77 now, 50000 x 999 29 against 41.  LINES: rows of whole 128-byte
// lines are read nontemporally (1500000 x 64 57 us, 64 without); a line that two
// rows share would then come from memory twice (1500000 x 75 102).
template <int OP, int LPR, int NV, bool LINES>
__global__ void __launch_bounds__(256)
k_rows_lanes(const float* a, float* out, uint64_t rows, uint32_t L, int rebroadcast, float mul, float dv) {
  using R = Red<OP, float>;
  constexpr int RPB = 256 / LPR;
  const int li = threadIdx.x % LPR;
  const uint32_t L4 = L / 4;
  for (uint64_t r = (uint64_t)blockIdx.x * RPB + threadIdx.x / LPR; r < rows; r += (uint64_t)gridDim.x * RPB) {
    const float* row = a + r * L;
    f32x4u_t v[NV];
#pragma unroll
    for (int q = 0; q < NV; ++q)
      if (li + q * LPR < L4)
        v[q] = ld4u<LINES>(row + 4 * (li + q * LPR));
    const bool tail = 4 * L4 + li < L;
    const float tv = tail ? row[4 * L4 + li] : 0.f;
    float g[NV];
#pragma unroll
    for (int q = 0; q < NV; ++q)
      g[q] = li + q * LPR < L4 ? R::f(R::f(v[q][0], v[q][1]), R::f(v[q][2], v[q][3])) : R::init();
    if (tail) g[NV - 1] = R::f(g[NV - 1], tv);
#pragma unroll
    for (int h = NV / 2; h >= 1; h /= 2)
#pragma unroll
      for (int q = 0; q < h; ++q) g[q] = R::f(g[q], g[q + h]);
    float acc = g[0];
#pragma unroll
    for (int off = LPR / 2; off >= 1; off >>= 1) acc = R::f(acc, __shfl_xor(acc, off, 64));
    const float res = epilogue(acc, mul, dv);
    if (!rebroadcast) {
      if (li == 0) out[r] = res;
    } else {
      float* o = out + r * L;
      for (uint32_t i = li; i < L4; i += LPR)
        *reinterpret_cast<f32x4u_t*>(o + 4 * i) = f32x4u_t{res, res, res, res};
      if (tail) o[4 * L4 + li] = res;
    }
  }
}

// one thread per row (short rows), sequential over the row like the reference
template <int OP>
__global__ void __launch_bounds__(256)
k_rows_thread(const float* a, float* out, uint64_t rows, uint64_t L, int rebroadcast, float mul, float dv) {
  const uint64_t stride = (uint64_t)gridDim.x * 256;
  for (uint64_t r = (uint64_t)blockIdx.x * 256 + threadIdx.x; r < rows; r += stride) {
    const float* row = a + r * L;
    float acc = row[0];
    for (uint64_t i = 1; i < L; ++i) acc = Red<OP, float>::f(acc, row[i]);
    float res = epilogue(acc, mul, dv);
    if (!rebroadcast) out[r] = res;
    else for (uint64_t i = 0; i < L; ++i) out[r * L + i] = res;
  }
}

// ---- strided axes: post > 1 ------------------------------------------------------
// k_cols: a viewed as [prev, K, post]; thread owns VW consecutive columns j of one p
// and reduces k in [k0, k1) sequentially.  Result goes to dst[(c * prev + p) *
// post + j] where c is the chunk index (blockIdx.y).  U rows are loaded at a
// time (VW == 4) and still combined in row order, so U never changes the result.
// With VW = 4 the last group of a row starts at post - 4 (the columns it shares
// with the group before are written twice, with the same values), at any
// alignment; VW = 1 is for fewer than 4 columns and where groups of 4 would
// leave fewer than 64 K threads (2000 x 2047: 13 us by fours).
template <int OP, int VW, int U, bool NT>
__global__ void __launch_bounds__(256)
k_cols(const float* a, float* dst, uint64_t prev, uint64_t K, uint64_t post, uint64_t kchunk,
       int final_pass, float mul, float dv) {
  const uint64_t groups = (post + VW - 1) / VW;
  const uint64_t total = prev * groups;
  const uint64_t c = blockIdx.y;
  const uint64_t k0 = c * kchunk;
  const uint64_t k1 = (k0 + kchunk < K) ? k0 + kchunk : K;
  const uint64_t stride = (uint64_t)gridDim.x * 256;
  for (uint64_t t = (uint64_t)blockIdx.x * 256 + threadIdx.x; t < total; t += stride) {
    const uint64_t p = t / groups, j = min((t - p * groups) * VW, post - VW);
    const float* base = a + (p * K) * post + j;
    if (VW == 4) {
      using R = Red<OP, float>;
      auto comb = [](f32x4u_t& acc, const f32x4u_t& v) {
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[q] = R::f(acc[q], v[q]);
      };
      f32x4u_t acc = ld4u<NT>(base + k0 * post);
      uint64_t k = k0 + 1;
      // U rows in flight, still combined in row order
      for (; k + (U - 1) < k1; k += U) {
        f32x4u_t v[U];
#pragma unroll
        for (int q = 0; q < U; ++q) v[q] = ld4u<NT>(base + (k + q) * post);
#pragma unroll
        for (int q = 0; q < U; ++q) comb(acc, v[q]);
      }
      for (; k < k1; ++k) comb(acc, ld4u<NT>(base + k * post));
      if (final_pass)
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[q] = epilogue(acc[q], mul, dv);
      *reinterpret_cast<f32x4u_t*>(dst + (c * prev + p) * post + j) = acc;
    } else {
      float acc = base[k0 * post];
      uint64_t k = k0 + 1;
      for (; k + (U - 1) < k1; k += U) {
        float v[U];
#pragma unroll
        for (int q = 0; q < U; ++q) v[q] = base[(k + q) * post];
#pragma unroll
        for (int q = 0; q < U; ++q) acc = Red<OP, float>::f(acc, v[q]);
      }
      for (; k < k1; ++k) acc = Red<OP, float>::f(acc, base[k * post]);
      if (final_pass) acc = epilogue(acc, mul, dv);
      dst[(c * prev + p) * post + j] = acc;
    }
  }
}

// Rows of 4 to ROWS_TILE_L elements: a wave takes 64 rows at a time straight into
// its own LDS (contiguous memory: whole aligned lines at any row length, and no
// registers for what is in flight), then each lane reduces a row, VW elements an
// LDS read, into eight accumulators (VW = 4: two reads') that are combined in
// pairs. ROT: lane l starts at its row's read l, where rows would start
// on the same banks.  HBM-bound: 2000000 x 32 38 us, 1000000 x 50 29 (58 both for
// a block's 256 rows through registers to LDS and a barrier), 4000000 x 5 16 (21).
// From 16 elements a row on and under 64 rows a CU, too few waves have rows and
// k_rows_lanes takes them: 500 x 63 4.9 against 7.8, 16000 x 63 5.1 against 12.
// WIDE: rows of 65 to 79 elements come here where the operand is larger than the
// caches (NT) and their length is odd (no bank conflicts for one row a lane), added in the
// order of a wave a row (lane_tree), whose error eight accumulators of 8 to 10
// elements exceed by 3 to 4%.  1500000 x 75 after the kernel that wrote it 78 us and the
// next kernel 90; k_rows_lanes takes 106 and 82 with nontemporal loads, 78 and
// 108 without.  Past 80 elements a compute unit has LDS for one block only: 1323529 x 85
// and the write of the operand together 236 us, 224 with k_rows_lanes (75 columns: 226, 65: 220).
constexpr uint32_t ROWS_TILE_L = 63, ROWS_TILE_L_NT = 79;

// The tree a wave makes of a row of 64 to 127 elements, lane i holding elements
// i and i + 64 (lanes i and i ^ 32 first, then i ^ 16, ...), by one thread.
template <int OP, int I = 0, int OFF = 1>
__device__ __forceinline__ float lane_tree(const float* row, uint32_t L) {
  using R = Red<OP, float>;
  if constexpr (OFF < 64) {
    return R::f(lane_tree<OP, I, OFF * 2>(row, L), lane_tree<OP, I + OFF, OFF * 2>(row, L));
  } else {
    const float v = R::f(R::init(), row[I]);
    if constexpr (I + 64 > ROWS_TILE_L_NT) return v;
    const bool two = I + 64 < L;
    const float w = R::f(v, row[two ? I + 64 : I]);
    return two ? w : v;
  }
}

template <int OP, int VW, bool ROT, bool NT, bool WIDE = false>
__global__ void __launch_bounds__(256)
k_rows_tile(const float* a, float* out, uint64_t rows, uint32_t L, float mul, float dv) {
  using Rd = Red<OP, float>;
  extern __shared__ __attribute__((aligned(16))) float tile_lds[];
  constexpr int A = 8 / VW;  // reads in flight with accumulators of their own
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  float* t = tile_lds + wave * 64 * L;
  const uint32_t n4 = 16 * L, U = L / VW;
  const uint64_t tiles = (rows + 63) / 64;
  const bool aligned = ((uintptr_t)a & 15u) == 0;
  for (uint64_t tile = (uint64_t)blockIdx.x * 4 + wave; tile < tiles; tile += (uint64_t)gridDim.x * 4) {
    const uint32_t nr = (uint32_t)min<uint64_t>(64, rows - tile * 64);
    const float* src = a + tile * 64 * L;
    if (nr == 64 && aligned) {
      for (uint32_t i = 0; i < n4; i += 64)
        if (i + lane < n4) load_lds16<NT>(src + (uint64_t)(i + lane) * 4, t + i * 4);
    } else if (nr == 64) {
      typedef __attribute__((ext_vector_type(4))) float f32x4_t;
#pragma unroll 4
      for (uint32_t i = lane; i < n4; i += 64) *reinterpret_cast<f32x4_t*>(t + i * 4) = ld4u<false>(src + i * 4);
    } else {
      for (uint32_t i = lane; i < nr * L; i += 64) t[i] = src[i];
    }
    __builtin_amdgcn_s_waitcnt(0);  // (a wave's own LDS: no barrier)
    __builtin_amdgcn_wave_barrier();
    if (WIDE) {
      if ((uint32_t)lane < nr) out[tile * 64 + lane] = epilogue(lane_tree<OP>(t + lane * L, L), mul, dv);
    } else if ((uint32_t)lane < nr) {
      typedef __attribute__((ext_vector_type(VW))) float vec_t;
      const vec_t* row = reinterpret_cast<const vec_t*>(t + lane * L);
      uint32_t e = ROT ? lane % U : 0;
      auto next = [&]() __attribute__((always_inline)) {
        const vec_t v = row[e];
        ++e;
        if (ROT && e == U) e = 0;
        return v;
      };
      vec_t acc[A];
      auto fold = [&](vec_t& x, vec_t y) __attribute__((always_inline)) {
        if constexpr (VW == 1) {
          x = Rd::f(x[0], y[0]);
        } else {
#pragma unroll
          for (int w = 0; w < VW; ++w) x[w] = Rd::f(x[w], y[w]);
        }
      };
      uint32_t k = min(U, (uint32_t)A);
#pragma unroll
      for (int q = 0; q < A; ++q)
        if (q < (int)k) acc[q] = next();
      for (; k + A <= U; k += A)
#pragma unroll
        for (int q = 0; q < A; ++q) fold(acc[q], next());
#pragma unroll
      for (int q = 0; q < A; ++q)
        if (k + q < U) fold(acc[q], next());
#pragma unroll
      for (int h = A / 2; h >= 1; h /= 2)
#pragma unroll
        for (int q = 0; q < h; ++q)
          if (q + h < (int)min(U, (uint32_t)A)) fold(acc[q], acc[q + h]);
      float r = acc[0][0];
      if constexpr (VW == 2) r = Rd::f(r, acc[0][1]);
      if constexpr (VW == 4) r = Rd::f(Rd::f(r, acc[0][1]), Rd::f(acc[0][2], acc[0][3]));
      out[tile * 64 + lane] = epilogue(r, mul, dv);
    }
    __builtin_amdgcn_s_waitcnt(0);  // the reads are done before the next rows arrive
    __builtin_amdgcn_wave_barrier();
  }
}

// Few columns: a block takes whole rows, thread t column group t % G of rows
// t / G, + R, + 2R ... of its chunk, so that a block reads its chunk as one
// contiguous run; the R sums of a column are then combined by a tree in LDS.
// Chunk partials dst[p][c][post] are reduced by the same kernel, in as many
// more passes as leave each thread about 16 rows.  Rows in flight are combined in
// pairs, eight, then four, two and one: where a row takes more than half of the
// block (513 columns and more), the last pass has up to 31 chunk sums a thread, and
// one after the other these made the rms error of 200 to 500 rows 1.03 to 1.31
// times that of k_cols (in pairs 0.71 to 0.95).  k_cols gives every chunk a block
// of which only G threads work (1000000 x 16: 4 of 256) and combines up to 1024
// chunks one after the other.  Against it: 1000000 x 16 18 against 161 us, 3000000
// x 3 11 against 371, 1500000 x 75 78 against 678, 50000 x 999 44 against 120
// (element loads), 50000 x 1000 43 against 60 (87 with one last pass over all 1024
// chunks).
template <int OP, int VW, bool NT>
__global__ void __launch_bounds__(256)
k_cols_narrow(const float* a, float* dst, uint64_t K, uint32_t post, uint64_t kchunk, uint32_t G, uint32_t R,
              int final_pass, float mul, float dv, float beta) {
  using Rd = Red<OP, float>;
  __shared__ float lds[256 * VW];
  const uint64_t c = blockIdx.x, p = blockIdx.y;
  const uint64_t k0 = c * kchunk, k1 = min(k0 + kchunk, K);
  const uint32_t rr = threadIdx.x / G, g = threadIdx.x - rr * G;
  const uint32_t j = min(g * VW, post - VW);
  uint32_t n = (uint32_t)min<uint64_t>(R, k1 - k0);  // rows of threads that have a row
  float acc[VW];
  auto load = [&](uint64_t k, float (&v)[VW]) {
    const float* q = a + (p * K + k) * post + j;
    if constexpr (VW == 4) {
      const f32x4u_t t = ld4u<NT>(q);
      v[0] = t[0]; v[1] = t[1]; v[2] = t[2]; v[3] = t[3];
    } else {
      v[0] = *q;
    }
  };
  if (rr < n) {
    load(k0 + rr, acc);
    uint64_t k = k0 + rr + R;
    auto rows = [&](auto count) {  // rows in flight, combined in pairs
      constexpr int N = decltype(count)::value;
      float v[N][VW];
#pragma unroll
      for (int q = 0; q < N; ++q) load(k + (uint64_t)q * R, v[q]);
#pragma unroll
      for (int s = 1; s < N; s *= 2)
#pragma unroll
        for (int q = 0; q < N; q += 2 * s)
#pragma unroll
          for (int w = 0; w < VW; ++w) v[q][w] = Rd::f(v[q][w], v[q + s][w]);
#pragma unroll
      for (int w = 0; w < VW; ++w) acc[w] = Rd::f(acc[w], v[0][w]);
      k += (uint64_t)N * R;
    };
    while (k + 7 * (uint64_t)R < k1) rows(std::integral_constant<int, 8>());
    if (k + 3 * (uint64_t)R < k1) rows(std::integral_constant<int, 4>());
    if (k + R < k1) rows(std::integral_constant<int, 2>());
    if (k < k1) rows(std::integral_constant<int, 1>());
#pragma unroll
    for (int w = 0; w < VW; ++w) lds[w * 256 + threadIdx.x] = acc[w];
  }
  __syncthreads();
  while (n > 1) {
    const uint32_t h = (n + 1) / 2;
    if (rr + h < n)
#pragma unroll
      for (int w = 0; w < VW; ++w)
        lds[w * 256 + threadIdx.x] = Rd::f(lds[w * 256 + threadIdx.x], lds[w * 256 + threadIdx.x + h * G]);
    __syncthreads();
    n = h;
  }
  if (rr == 0) {
    float* d = dst + (p * gridDim.x + c) * post + j;
#pragma unroll
    for (int w = 0; w < VW; ++w) {
      float r = lds[w * 256 + threadIdx.x];
      if (final_pass) r = epilogue(r, mul, dv);
      if (beta == 0.f) d[w] = r;
      else if (j + w >= g * VW) d[w] = beta * d[w] + r;  // (the last group's other columns are its neighbour's)
    }
  }
}

// combine nchunk partials [nchunk, m] in chunk order into out[m]
template <int OP>
__global__ void __launch_bounds__(256)
k_combine_chunks(const float* part, float* out, uint64_t m, uint64_t nchunk, float mul, float dv) {
  const uint64_t stride = (uint64_t)gridDim.x * 256;
  for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < m; i += stride) {
    float acc = part[i];
    uint64_t c = 1;
    for (; c + 8 <= nchunk; c += 8) {  // eight loads in flight, combined in chunk order
      float v[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) v[q] = part[(c + q) * m + i];
#pragma unroll
      for (int q = 0; q < 8; ++q) acc = Red<OP, float>::f(acc, v[q]);
    }
    for (; c < nchunk; ++c) acc = Red<OP, float>::f(acc, part[c * m + i]);
    out[i] = epilogue(acc, mul, dv);
  }
}

// red [prev, post] -> out [prev, K, post] (rebroadcast of a strided axis)
__global__ void __launch_bounds__(256)
k_rebroadcast_cols(const float* red, float* out, uint64_t prev, uint64_t K, uint64_t post) {
  const uint64_t total = prev * K * post;
  const uint64_t stride = (uint64_t)gridDim.x * 256;
  for (uint64_t t = (uint64_t)blockIdx.x * 256 + threadIdx.x; t < total; t += stride) {
    const uint64_t j = t % post, p = t / (K * post);
    out[t] = red[p * post + j];
  }
}

// ---- full reduction ----------------------------------------------------------------
constexpr int ALL_BLOCK = 256;

// U (4 or 8) 128-bit loads in flight per thread; a group of eight is combined
// as two consecutive groups of four, so for a given grid U never changes the
// result
template <int OP, int U>
__global__ void __launch_bounds__(ALL_BLOCK)
k_all_partial(const float* a, uint64_t n, double* part) {
  __shared__ double lds[ALL_BLOCK / 64];
  double acc = Red<OP, double>::init();
  const uint64_t stride = (uint64_t)gridDim.x * ALL_BLOCK;
  const uint64_t n4 = ((uintptr_t)a & 15u) == 0 ? n / 4 : 0;
  const float4* a4 = reinterpret_cast<const float4*>(a);
  using R = Red<OP, double>;
  auto quad = [](const float4& v) {
    return R::f(R::f((double)v.x, (double)v.y), R::f((double)v.z, (double)v.w));
  };
  uint64_t i = (uint64_t)blockIdx.x * ALL_BLOCK + threadIdx.x;
  if constexpr (U == 8) {
    for (; i + 7 * stride < n4; i += 8 * stride) {
      float4 v[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) v[q] = ld_stream(a4 + i + q * stride);
      acc = R::f(acc, R::f(R::f(quad(v[0]), quad(v[1])), R::f(quad(v[2]), quad(v[3]))));
      acc = R::f(acc, R::f(R::f(quad(v[4]), quad(v[5])), R::f(quad(v[6]), quad(v[7]))));
    }
  }
  for (; i + 3 * stride < n4; i += 4 * stride) {  // four loads in flight
    const float4 v0 = ld_stream(a4 + i), v1 = ld_stream(a4 + i + stride);
    const float4 v2 = ld_stream(a4 + i + 2 * stride), v3 = ld_stream(a4 + i + 3 * stride);
    acc = R::f(acc, R::f(R::f(quad(v0), quad(v1)), R::f(quad(v2), quad(v3))));
  }
  for (; i < n4; i += stride) acc = R::f(acc, quad(ld_stream(a4 + i)));
  for (uint64_t i = n4 * 4 + (uint64_t)blockIdx.x * ALL_BLOCK + threadIdx.x; i < n; i += stride)
    acc = Red<OP, double>::f(acc, (double)a[i]);
  double r = block_reduce<OP, double, ALL_BLOCK>(acc, lds);
  if (threadIdx.x == 0) part[blockIdx.x] = r;
}

template <int OP>
__global__ void __launch_bounds__(ALL_BLOCK)
k_all_final(const double* part, uint64_t nb, float* out, uint64_t n, int mean) {
  __shared__ double lds[ALL_BLOCK / 64];
  double acc = Red<OP, double>::init();
  for (uint64_t i = threadIdx.x; i < nb; i += ALL_BLOCK) acc = Red<OP, double>::f(acc, part[i]);
  double r = block_reduce<OP, double, ALL_BLOCK>(acc, lds);
  if (threadIdx.x == 0) out[0] = (float)(mean ? r / (double)n : r);
}

// ---- kernel configurations (vkh_reduce_autotune) ------------------------------
// unroll: 128-bit loads in flight per thread.  par: blocks per CU (full and row
// reductions: the grid cap) or target threads per CU (strided axes: decides
// how many chunks k is split into).  Index 0 of each family is the default.
struct RedCfg {
  int unroll, par;
};
static const RedCfg ALL_CFGS[] = {{4, 4}, {8, 4}, {4, 2}, {8, 2}, {4, 8}, {8, 8}, {4, 16}, {8, 16}};
static const RedCfg ROWS_CFGS[] = {{4, 16}, {8, 16}, {4, 8}, {8, 8}, {4, 32}, {8, 32}};
static const RedCfg COLS_CFGS[] = {{4, 512}, {8, 512}, {4, 256}, {8, 256},
                                   {4, 1024}, {8, 1024}, {4, 2048}, {8, 2048}};
constexpr int ROWS_BLOCK_MIN_L = 2048;  // shorter rows use the wave / thread kernels

static const RedCfg* red_cfgs(int fam, int& n) {
  switch (fam) {
    case VKH_RFAM_ALL: n = (int)(sizeof(ALL_CFGS) / sizeof(RedCfg)); return ALL_CFGS;
    case VKH_RFAM_ROWS: n = (int)(sizeof(ROWS_CFGS) / sizeof(RedCfg)); return ROWS_CFGS;
    case VKH_RFAM_COLS: n = (int)(sizeof(COLS_CFGS) / sizeof(RedCfg)); return COLS_CFGS;
  }
  n = 1;  // a single kernel choice
  return nullptr;
}

// family of a reduction: kind 0 = full (n = prev * K * post), 1 = axis
static int red_family(int kind, uint64_t K, uint64_t post) {
  if (kind == 0) return VKH_RFAM_ALL;
  if (post > 1) return VKH_RFAM_COLS;
  return K >= ROWS_BLOCK_MIN_L ? VKH_RFAM_ROWS : VKH_RFAM_NONE;
}

static std::array<uint64_t, 4> red_key(int fam, uint64_t prev, uint64_t K, uint64_t post) {
  if (fam == VKH_RFAM_ALL) return {(uint64_t)fam, 1, prev * K * post, 1};
  return {(uint64_t)fam, prev, K, post};
}

// configuration of a call: the explicit index when >= 0, else the one chosen
// for the shape on this context, else the default
static RedCfg red_cfg(vkh_gpu* g, int fam, uint64_t prev, uint64_t K, uint64_t post, int index) {
  int n = 0;
  const RedCfg* c = red_cfgs(fam, n);
  if (!c) return RedCfg{4, 0};
  if (index < 0) {
    auto it = g->red_cfg.find(red_key(fam, prev, K, post));
    index = it == g->red_cfg.end() ? 0 : it->second;
  }
  return c[index];
}

// blocks of a full reduction of n elements: one FP64 partial each
static unsigned all_blocks(vkh_gpu* g, uint64_t n, const RedCfg& c) {
  return stream_grid(g, ceil_div(n, 4 * 4), ALL_BLOCK, (unsigned)c.par);
}

// partial pass into part[0, nb), then the final combine into out[0]
template <int OP>
static void launch_all(vkh_gpu* g, const float* a, uint64_t n, float* out, int mean, const RedCfg& c,
                       unsigned nb, double* part) {
  if (c.unroll == 8)
    hipLaunchKernelGGL((k_all_partial<OP, 8>), dim3(nb), dim3(ALL_BLOCK), 0, g->stream, a, n, part);
  else
    hipLaunchKernelGGL((k_all_partial<OP, 4>), dim3(nb), dim3(ALL_BLOCK), 0, g->stream, a, n, part);
  check_launch("reduce_all partial");
  hipLaunchKernelGGL(k_all_final<OP>, dim3(1), dim3(ALL_BLOCK), 0, g->stream, part, (uint64_t)nb, out, n, mean);
  check_launch("reduce_all final");
}

template <int OP>
static void reduce_all(vkh_gpu* g, const float* a, uint64_t n, float* out, int mean, int index = -1) {
  const RedCfg c = red_cfg(g, VKH_RFAM_ALL, 1, n, 1, index);
  const unsigned nb = all_blocks(g, n, c);
  Workspace ws(g, sizeof(double) * nb);
  launch_all<OP>(g, a, n, out, mean, c, nb, (double*)ws.get());
}

// ---- allocation-free full reduction (vkh_reduce_all_noalloc) ------------------
// The FP64 block partials go to this file-scope device array instead of a
// workspace.  Each device holds its own copy at its own address, looked up
// once per device with hipGetSymbolAddress; host code passes that address,
// never the array's name (on the host the name is a stand-in, not device
// memory).  Every block writes its own partial before the final kernel reads
// it, so no call depends on what an earlier call left there.
constexpr unsigned NOALLOC_PARTIALS = 8192;  // 64 KiB: 256 CUs x 16 blocks per CU, twice over
static __device__ __align__(256) double scratch[NOALLOC_PARTIALS];

constexpr int MAX_DEVICES = 64;
static std::mutex g_scratch_mu;
static double* g_scratch_ptr[MAX_DEVICES] = {};

// address of this device's scratch; the device must be current
static double* scratch_address(vkh_gpu* g) {
  VKH_REQUIRE(g->device >= 0 && g->device < MAX_DEVICES, "reduce_all_noalloc: device index out of range");
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  double*& p = g_scratch_ptr[g->device];
  if (!p) {
    void* addr = nullptr;
    VKH_HIP(hipGetSymbolAddress(&addr, HIP_SYMBOL(scratch)));
    VKH_REQUIRE(addr != nullptr, "reduce_all_noalloc: no device address for the scratch array");
    p = (double*)addr;
  }
  return p;
}

template <int OP>
static void reduce_all_noalloc(vkh_gpu* g, const float* a, uint64_t n, float* out, int mean) {
  const RedCfg c = red_cfg(g, VKH_RFAM_ALL, 1, n, 1, -1);
  const unsigned nb = all_blocks(g, n, c);
  if (nb > NOALLOC_PARTIALS)
    fail(VKH_INVALID, "reduce_all_noalloc: " + std::to_string(nb) + " block partials exceed the " +
                          std::to_string(NOALLOC_PARTIALS) + " the scratch array holds");
  launch_all<OP>(g, a, n, out, mean, c, nb, scratch_address(g));
}

// Rows per chunk (and the chunk count) of the strided-axis reduction of
// [prev, K, post] in configuration cfg.  Split k when there are fewer than
// cfg.par threads of columns per CU and the axis is long enough to give every
// chunk a reasonable amount of work (default 512: on 8192 x 16384, 32 chunks
// of 256 rows reach 6.4 TB/s, 64 chunks 6.1).  The chunk count fixes the
// summation order of sums and products, so it is part of the shape's
// configuration.
static uint64_t cols_chunk(vkh_gpu* g, const RedCfg& cfg, uint64_t prev, uint64_t K, uint64_t post,
                           uint64_t& nchunk_out) {
  const unsigned cus = g->num_cus > 0 ? g->num_cus : 256;
  const uint64_t threads = prev * (post >= 4 ? ceil_div(post, 4) : post);
  const uint64_t want = (uint64_t)cus * (uint64_t)cfg.par;
  uint64_t nchunk = 1;
  if (threads < want && K >= 64) {
    nchunk = std::min<uint64_t>(ceil_div(want, threads), K / 32);
    if (nchunk > 1024) nchunk = 1024;
    if (nchunk < 1) nchunk = 1;
  }
  const uint64_t kchunk = ceil_div(K, nchunk);
  nchunk_out = ceil_div(K, kchunk);
  return kchunk;
}

// Shapes of k_cols_narrow: fewer than 1024 columns (a block holds a row) and
// too few columns in all to fill the chip with one thread a column group.  The
// column sums that the fused last-layer backward reproduces in order (one
// matrix, rows a multiple of 128, columns of 32: dense1_chunks in gemm.hip)
// keep k_cols, all shapes that it might take, with k_cols' times: 65536 x 64 42 us (x 65
// 9), 2^20 x 32 82 (x 33 28), 16384 x 256 26 (x 257 12), 256 x 64 6.6 (x 65 4.7).
static bool cols_narrow(vkh_gpu* g, uint64_t prev, uint64_t K, uint64_t post) {
  if (post >= 1024 || K < 64 || prev > 65535 || (prev == 1 && K % 128 == 0 && post % 32 == 0)) return false;
  const uint64_t cus = g->num_cus > 0 ? g->num_cus : 256;
  return prev * ceil_div(post, 4) < cus * 256;
}

template <int OP>
static void reduce_cols_narrow(vkh_gpu* g, const float* a, float* out, uint64_t prev, uint64_t K, uint64_t post,
                               float mul, float dv, float beta = 0.f) {
  const uint64_t cus = g->num_cus > 0 ? g->num_cus : 256;
  const uint32_t G = (uint32_t)(post >= 4 ? ceil_div(post, 4) : post), R = 256 / G;
  // about four blocks a CU, at least 16 rows a thread
  uint64_t nchunk = std::max<uint64_t>(1, std::min(ceil_div(4 * cus, prev), K / (16 * (uint64_t)R)));
  const uint64_t kchunk = ceil_div(K, nchunk);
  nchunk = ceil_div(K, kchunk);
  auto launch = [&](const float* src, float* dst, uint64_t k, uint64_t kc, uint64_t nc, int fin) {
    const dim3 grid((unsigned)nc, (unsigned)prev);
    auto kernel = post < 4 ? k_cols_narrow<OP, 1, false>
                           : (streams(prev * K * post) ? k_cols_narrow<OP, 4, true> : k_cols_narrow<OP, 4, false>);
    hipLaunchKernelGGL(kernel, grid, dim3(256), 0, g->stream, src, dst, k, (uint32_t)post, kc, G, R, fin, mul, dv,
                       fin ? beta : 0.f);
    check_launch("reduce cols (narrow)");
  };
  if (nchunk == 1) {
    launch(a, out, K, kchunk, 1, 1);
    return;
  }
  Workspace ws(g, sizeof(float) * prev * nchunk * post);
  launch(a, (float*)ws.get(), K, kchunk, nchunk, 0);
  reduce_cols_narrow<OP>(g, (const float*)ws.get(), out, prev, nchunk, post, mul, dv, beta);
}

template <int OP>
static void reduce_axis(vkh_gpu* g, const float* a, float* out, uint64_t prev, uint64_t K,
                        uint64_t post, int rebroadcast, float mul, float dv, int index = -1) {
  const unsigned cus = g->num_cus > 0 ? g->num_cus : 256;
  const RedCfg cfg = red_cfg(g, red_family(1, K, post), prev, K, post, index);
  if (post == 1) {
    const uint64_t rows = prev, L = K;
    if (L >= ROWS_BLOCK_MIN_L) {
      unsigned grid = (unsigned)std::min<uint64_t>(rows, (uint64_t)cus * cfg.par);
      auto kernel = cfg.unroll == 8 ? (streams(rows * L) ? k_rows_block<OP, 8, true> : k_rows_block<OP, 8, false>)
                                    : (streams(rows * L) ? k_rows_block<OP, 4, true> : k_rows_block<OP, 4, false>);
      hipLaunchKernelGGL(kernel, dim3(grid), dim3(ROW_BLOCK), 0, g->stream, a, out, rows, L, rebroadcast, mul, dv);
    } else if (L >= 4 && !rebroadcast &&
               (L <= ROWS_TILE_L ? L < 16 || rows >= (uint64_t)cus * 64
                                 : L <= ROWS_TILE_L_NT && L % 2 != 0 && streams(rows * L))) {
      const uint32_t vw = L % 4 == 0 ? 4 : (L % 2 == 0 ? 2 : 1);
      const size_t sh = sizeof(float) * 256 * L;
      const unsigned grid = (unsigned)std::min<uint64_t>(ceil_div(rows, 256), (uint64_t)cus * 8);
      auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(grid), dim3(256), sh, g->stream, a, out, rows, (uint32_t)L, mul, dv);
      };
      const bool rot = (L / vw) % 2 == 0, nt = streams(rows * L);
#define VKH_ROWS_TILE(VW, ROT) \
  do { if (nt) launch(k_rows_tile<OP, VW, ROT, true>); else launch(k_rows_tile<OP, VW, ROT, false>); } while (0)
      if (L > ROWS_TILE_L) launch(k_rows_tile<OP, 1, false, true, true>);
      else if (vw == 4 && rot) VKH_ROWS_TILE(4, true);
      else if (vw == 4) VKH_ROWS_TILE(4, false);
      else if (vw == 2 && rot) VKH_ROWS_TILE(2, true);
      else if (vw == 2) VKH_ROWS_TILE(2, false);
      else VKH_ROWS_TILE(1, false);
#undef VKH_ROWS_TILE
    } else if (L >= 64 || (L >= 16 && !rebroadcast)) {
      // lanes a row: up to 4 groups a lane, 8 of a whole wave
      auto launch = [&](auto kernel, int lpr) {
        const unsigned grid = (unsigned)std::min<uint64_t>(ceil_div(rows, 256 / lpr), (uint64_t)cus * 64);
        hipLaunchKernelGGL(kernel, dim3(grid), dim3(256), 0, g->stream, a, out, rows, (uint32_t)L, rebroadcast, mul, dv);
      };
      const uint64_t L4 = L / 4;
      const bool lines = L % 32 == 0 && ((uintptr_t)a & 127u) == 0;
#define VKH_ROWS_LANES(LPR, NV) \
  do { if (lines) launch(k_rows_lanes<OP, LPR, NV, true>, LPR); else launch(k_rows_lanes<OP, LPR, NV, false>, LPR); } while (0)
      if (L4 <= 32) VKH_ROWS_LANES(8, 4);
      else if (L4 <= 64) VKH_ROWS_LANES(16, 4);
      else if (L4 <= 128) VKH_ROWS_LANES(32, 4);
      else if (L4 <= 256) VKH_ROWS_LANES(64, 4);
      else VKH_ROWS_LANES(64, 8);
#undef VKH_ROWS_LANES
    } else {
      unsigned grid = (unsigned)std::min<uint64_t>(ceil_div(rows, 256), (uint64_t)cus * 16);
      hipLaunchKernelGGL(k_rows_thread<OP>, dim3(grid), dim3(256), 0, g->stream, a, out, rows, L, rebroadcast, mul, dv);
    }
    check_launch("reduce rows");
    return;
  }
  if (cols_narrow(g, prev, K, post)) {
    if (!rebroadcast) {
      reduce_cols_narrow<OP>(g, a, out, prev, K, post, mul, dv);
      return;
    }
    Workspace red(g, sizeof(float) * prev * post);
    reduce_cols_narrow<OP>(g, a, (float*)red.get(), prev, K, post, mul, dv);
    hipLaunchKernelGGL(k_rebroadcast_cols, dim3(stream_grid(g, prev * K * post, 256, 8)), dim3(256), 0, g->stream,
                       (const float*)red.get(), out, prev, K, post);
    check_launch("reduce rebroadcast");
    return;
  }
  uint64_t nchunk = 0;
  const uint64_t kchunk = cols_chunk(g, cfg, prev, K, post, nchunk);
  const uint64_t m = prev * post;
  const bool quads = post >= 4 && prev * ceil_div(post, 4) * nchunk >= (uint64_t)cus * 256;
  const uint64_t threads = prev * (quads ? ceil_div(post, 4) : post);
  Workspace ws(g, (nchunk > 1 || rebroadcast) ? sizeof(float) * nchunk * m : 1);
  float* dst = (nchunk > 1 || rebroadcast) ? (float*)ws.get() : out;
  unsigned gx = (unsigned)std::min<uint64_t>(ceil_div(threads, 256), (uint64_t)cus * 16);
  if (gx < 1) gx = 1;
  dim3 grid(gx, (unsigned)nchunk);
  const int final_pass = (nchunk == 1) ? 1 : 0;
  const bool nt = streams(prev * K * post);
  auto kernel = !quads ? k_cols<OP, 1, 8, false>
                : cfg.unroll == 8 ? (nt ? k_cols<OP, 4, 8, true> : k_cols<OP, 4, 8, false>)
                                  : (nt ? k_cols<OP, 4, 4, true> : k_cols<OP, 4, 4, false>);
  hipLaunchKernelGGL(kernel, grid, dim3(256), 0, g->stream, a, dst, prev, K, post, kchunk, final_pass, mul, dv);
  check_launch("reduce cols");
  float* red = dst;
  if (nchunk > 1) {
    // combine into the first chunk's slot when rebroadcasting, else into out
    float* target = rebroadcast ? dst : out;
    if (rebroadcast) {
      // the combine reads every chunk, so write to a separate buffer
      Workspace ws2(g, sizeof(float) * m);
      float* t2 = (float*)ws2.get();
      unsigned gb = (unsigned)std::min<uint64_t>(ceil_div(m, 256), (uint64_t)cus * 16);
      hipLaunchKernelGGL(k_combine_chunks<OP>, dim3(gb), dim3(256), 0, g->stream, dst, t2, m, nchunk, mul, dv);
      check_launch("reduce combine");
      unsigned gr = stream_grid(g, prev * K * post, 256, 8);
      hipLaunchKernelGGL(k_rebroadcast_cols, dim3(gr), dim3(256), 0, g->stream, t2, out, prev, K, post);
      check_launch("reduce rebroadcast");
      return;
    }
    unsigned gb = (unsigned)std::min<uint64_t>(ceil_div(m, 256), (uint64_t)cus * 16);
    hipLaunchKernelGGL(k_combine_chunks<OP>, dim3(gb), dim3(256), 0, g->stream, dst, target, m, nchunk, mul, dv);
    check_launch("reduce combine");
    return;
  }
  if (rebroadcast) {
    unsigned gr = stream_grid(g, prev * K * post, 256, 8);
    hipLaunchKernelGGL(k_rebroadcast_cols, dim3(gr), dim3(256), 0, g->stream, red, out, prev, K, post);
    check_launch("reduce rebroadcast");
  }
}

}  // namespace vkh

using namespace vkh;

extern "C" {

int vkh_reduce_all(vkh_gpu* g, int op, const float* a, uint64_t n, float* out, int mean) {
  return guarded([&] {
    use(g);
    VKH_REQUIRE(out, "reduce_all: null output");
    VKH_REQUIRE(n == 0 || a, "reduce_all: null input");
    if (n == 0) {
      VKH_REQUIRE(op == VKH_RSUM || op == VKH_RPROD,
                  "zero-size array to reduction operation which has no identity");
    }
    switch (op) {
      case VKH_RSUM: reduce_all<VKH_RSUM>(g, a, n, out, mean); break;
      case VKH_RPROD: reduce_all<VKH_RPROD>(g, a, n, out, mean); break;
      case VKH_RMAX: reduce_all<VKH_RMAX>(g, a, n, out, mean); break;
      case VKH_RMIN: reduce_all<VKH_RMIN>(g, a, n, out, mean); break;
      default: fail(VKH_INVALID, "unknown reduction op");
    }
  });
}

}  // extern "C"

namespace vkh {
// db = beta * db + the column sums of a [rows, cols] operand with no pass of
// its own for the addition, where those sums take k_cols_narrow (150 x 32: 3.7
// us, 9.1 with the sums in a workspace and an addition); false elsewhere
bool bias_grad_narrow(vkh_gpu* g, const float* a, float* db, uint64_t rows, uint64_t cols, float beta) {
  if (cols == 1 || !cols_narrow(g, 1, rows, cols)) return false;
  reduce_cols_narrow<VKH_RSUM>(g, a, db, 1, rows, cols, 1.0f, 1.0f, beta);
  return true;
}

// chunk length of the column sums of a [rows, cols] operand (vkh_bias_grad's
// reduction), for kernels that must sum in the same order; 0 where that order
// is not one of row chunks
uint64_t bias_grad_chunk(vkh_gpu* g, uint64_t rows, uint64_t cols) {
  if (cols == 1 || cols_narrow(g, 1, rows, cols)) return 0;
  const RedCfg cfg = red_cfg(g, red_family(1, rows, cols), 1, rows, cols, -1);
  uint64_t nchunk = 0;
  return cols_chunk(g, cfg, 1, rows, cols, nchunk);
}

// Chunk partials part[c][m] summed per output in chunk order: FROM_ZERO 0
// starts from part[0] (k_combine_chunks' order for a sum, no scaling), 1 from
// +0 (the column walk's combine).  For few outputs and many chunks: a block
// takes 64 outputs, its four waves load batches of up to 128 chunks (256-byte
// rows, every load of a thread issued before the first wait) into LDS, and
// lane j of the first wave adds output j's batch in order.  The same sums as
// the one-thread-per-output combines, with all their loads in flight at once.
constexpr int CC_OUT = 64, CC_BATCH = 128, CC_PER = CC_BATCH / 4;
template <int FROM_ZERO>
__global__ void __launch_bounds__(256)
k_combine_cols(const float* __restrict__ part, float* __restrict__ out, uint64_t m, uint64_t nchunk) {
  __shared__ float tile[CC_BATCH][CC_OUT + 1];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const uint64_t j = (uint64_t)blockIdx.x * CC_OUT + lane;
  float acc = 0.f;
  for (uint64_t c0 = 0; c0 < nchunk; c0 += CC_BATCH) {
    float r[CC_PER];
#pragma unroll
    for (int q = 0; q < CC_PER; ++q) {
      const uint64_t c = c0 + w + 4 * q;
      r[q] = (c < nchunk && j < m) ? part[c * m + j] : 0.f;
    }
#pragma unroll
    for (int q = 0; q < CC_PER; ++q) tile[w + 4 * q][lane] = r[q];
    __syncthreads();
    if (w == 0) {
      const int nb = (int)min<uint64_t>(CC_BATCH, nchunk - c0);
      for (int c = 0; c < nb; ++c) {
        const float v = tile[c][lane];
        acc = (!FROM_ZERO && c0 == 0 && c == 0) ? v : acc + v;
      }
    }
    __syncthreads();
  }
  if (w == 0 && j < m) out[j] = acc;
}

static void combine_cols(vkh_gpu* g, const float* part, float* out, uint64_t m, uint64_t nchunk, bool from_zero) {
  const unsigned grid = (unsigned)ceil_div(m, (uint64_t)CC_OUT);
  if (from_zero) hipLaunchKernelGGL(k_combine_cols<1>, dim3(grid), dim3(256), 0, g->stream, part, out, m, nchunk);
  else hipLaunchKernelGGL(k_combine_cols<0>, dim3(grid), dim3(256), 0, g->stream, part, out, m, nchunk);
  check_launch("combine chunks");
}

// combine of chunk partials [nchunk, m] in chunk order (k_combine_chunks' sums)
void sum_chunks(vkh_gpu* g, const float* part, float* out, uint64_t m, uint64_t nchunk) {
  combine_cols(g, part, out, m, nchunk, false);
}

// the same from +0 (the skinny column walk's combine, k_skinny_combine with
// alpha 1, beta 0 and no epilogue)
void sum_chunks_from_zero(vkh_gpu* g, const float* part, float* out, uint64_t m, uint64_t nchunk) {
  combine_cols(g, part, out, m, nchunk, true);
}
}  // namespace vkh

extern "C" {

int vkh_reduce_all_noalloc(vkh_gpu* g, int op, const float* a, uint64_t n, float* out, int mean) {
  return guarded([&] {
    use(g);
    VKH_REQUIRE(out, "reduce_all_noalloc: null output");
    VKH_REQUIRE(n == 0 || a, "reduce_all_noalloc: null input");
    if (n == 0) {
      VKH_REQUIRE(op == VKH_RSUM || op == VKH_RPROD,
                  "zero-size array to reduction operation which has no identity");
    }
    switch (op) {
      case VKH_RSUM: reduce_all_noalloc<VKH_RSUM>(g, a, n, out, mean); break;
      case VKH_RPROD: reduce_all_noalloc<VKH_RPROD>(g, a, n, out, mean); break;
      case VKH_RMAX: reduce_all_noalloc<VKH_RMAX>(g, a, n, out, mean); break;
      case VKH_RMIN: reduce_all_noalloc<VKH_RMIN>(g, a, n, out, mean); break;
      default: fail(VKH_INVALID, "unknown reduction op");
    }
  });
}

int vkh_reduce_axis(vkh_gpu* g, int op, const float* a, float* out, uint64_t prev, uint64_t axis,
                    uint64_t post, int rebroadcast, float mul, float dv) {
  return guarded([&] {
    use(g);
    VKH_REQUIRE(a && out, "reduce_axis: null pointer");
    if (prev == 0 || post == 0) return;
    if (axis == 0) {
      VKH_REQUIRE(op == VKH_RSUM || op == VKH_RPROD,
                  "zero-size array to reduction operation which has no identity");
      // empty axis: identity, scaled like any result
      float ident = op == VKH_RSUM ? 0.0f : 1.0f;
      if (mul != 1.0f) ident *= mul;
      if (dv != 1.0f) ident /= dv;
      if (!rebroadcast) {
        int r = vkh_fill_f32(g, out, ident, prev * post);
        if (r != VKH_OK) fail(r, vkh_last_error());
      }
      return;
    }
    switch (op) {
      case VKH_RSUM: reduce_axis<VKH_RSUM>(g, a, out, prev, axis, post, rebroadcast, mul, dv); break;
      case VKH_RPROD: reduce_axis<VKH_RPROD>(g, a, out, prev, axis, post, rebroadcast, mul, dv); break;
      case VKH_RMAX: reduce_axis<VKH_RMAX>(g, a, out, prev, axis, post, rebroadcast, mul, dv); break;
      case VKH_RMIN: reduce_axis<VKH_RMIN>(g, a, out, prev, axis, post, rebroadcast, mul, dv); break;
      default: fail(VKH_INVALID, "unknown reduction op");
    }
  });
}

int vkh_reduce_family(int kind, uint64_t prev, uint64_t axis, uint64_t post, int* family) {
  return guarded([&] {
    VKH_REQUIRE(family, "null out");
    VKH_REQUIRE(kind == 0 || kind == 1, "reduction kind must be 0 (full) or 1 (axis)");
    (void)prev;
    *family = red_family(kind, axis, post);
  });
}

int vkh_reduce_configs(int family, int* count) {
  return guarded([&] {
    VKH_REQUIRE(count, "null out");
    VKH_REQUIRE(family >= VKH_RFAM_NONE && family <= VKH_RFAM_COLS, "unknown reduction family");
    red_cfgs(family, *count);
  });
}

int vkh_reduce_config_info(int family, int index, int* unroll, int* par) {
  return guarded([&] {
    VKH_REQUIRE(unroll && par, "null out");
    VKH_REQUIRE(family >= VKH_RFAM_NONE && family <= VKH_RFAM_COLS, "unknown reduction family");
    int n = 0;
    const RedCfg* c = red_cfgs(family, n);
    VKH_REQUIRE(index >= 0 && index < n, "configuration index out of range");
    *unroll = c ? c[index].unroll : 0;
    *par = c ? c[index].par : 0;
  });
}

int vkh_reduce_get_config(vkh_gpu* g, int kind, uint64_t prev, uint64_t axis, uint64_t post,
                          int* index, int* tuned) {
  return guarded([&] {
    VKH_REQUIRE(g && index, "null argument");
    VKH_REQUIRE(kind == 0 || kind == 1, "reduction kind must be 0 (full) or 1 (axis)");
    const int fam = red_family(kind, axis, post);
    auto it = g->red_cfg.find(red_key(fam, prev, axis, post));
    const bool have = it != g->red_cfg.end();
    *index = have ? it->second : 0;
    if (tuned) *tuned = have ? 1 : 0;
  });
}

int vkh_reduce_set_config(vkh_gpu* g, int kind, uint64_t prev, uint64_t axis, uint64_t post,
                          int index) {
  return guarded([&] {
    VKH_REQUIRE(g, "null GPU handle");
    VKH_REQUIRE(kind == 0 || kind == 1, "reduction kind must be 0 (full) or 1 (axis)");
    const int fam = red_family(kind, axis, post);
    const auto key = red_key(fam, prev, axis, post);
    if (index < 0) { g->red_cfg.erase(key); return; }
    int n = 0;
    red_cfgs(fam, n);
    VKH_REQUIRE(index < n, "configuration index out of range");
    if (fam == VKH_RFAM_NONE) return;  // a single kernel choice: nothing to keep
    g->red_cfg[key] = index;
  });
}

int vkh_reduce_autotune(vkh_gpu* g, int kind, uint64_t prev, uint64_t axis, uint64_t post,
                        int reps, int same_order, int* best, float* ms_per_config) {
  return guarded([&] {
    use(g);
    VKH_REQUIRE(kind == 0 || kind == 1, "reduction kind must be 0 (full) or 1 (axis)");
    VKH_REQUIRE(!g->capturing, "reduce_autotune: not allowed during graph capture");
    VKH_REQUIRE(prev > 0 && axis > 0 && post > 0, "reduce_autotune: empty reduction");
    VKH_REQUIRE(g->alloc, "reduce_autotune needs a context with its own allocator");
    if (reps < 1) reps = 3;
    const int fam = red_family(kind, axis, post);
    int n = 0;
    const RedCfg* cfgs = red_cfgs(fam, n);
    if (fam == VKH_RFAM_NONE || (fam == VKH_RFAM_COLS && cols_narrow(g, prev, axis, post))) {  // a single kernel choice
      if (ms_per_config)
        for (int i = 0; i < n; ++i) ms_per_config[i] = -1.0f;
      if (best) *best = 0;
      return;
    }
    // scratch input and output of the reduction's own shape
    const uint64_t total = prev * axis * post;
    const uint64_t nout = kind == 0 ? 1 : prev * post;
    Workspace win(g, sizeof(float) * total), wout(g, sizeof(float) * nout);
    float* A = (float*)win.get();
    float* O = (float*)wout.get();
    hipLaunchKernelGGL(k_fill_noise, dim3(full_grid(total, 256)), dim3(256), 0, g->stream, A, total, 5u);
    check_launch("reduce_autotune fill");
    auto run = [&](int i) {
      if (kind == 0) reduce_all<VKH_RSUM>(g, A, total, O, 0, i);
      else reduce_axis<VKH_RSUM>(g, A, O, prev, axis, post, 0, 1.0f, 1.0f, i);
    };
    hipEvent_t e0, e1;
    VKH_HIP(hipEventCreate(&e0));
    VKH_HIP(hipEventCreate(&e1));
    int bi = -1;
    float bt = 0.0f;
    // same_order: only configurations whose summation order is the
    // default's (every ROWS configuration; ALL and COLS with the default
    // par), so the choice cannot change a result
    auto candidate = [&](int i) { return !same_order || fam == VKH_RFAM_ROWS || cfgs[i].par == cfgs[0].par; };
    try {
      for (int i = 0; i < n; ++i) {
        if (!candidate(i)) {
          if (ms_per_config) ms_per_config[i] = -1.0f;
          continue;
        }
        run(i);  // warm-up
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
    g->red_cfg[red_key(fam, prev, axis, post)] = bi;
    if (best) *best = bi;
  });
}

}  // extern "C"
