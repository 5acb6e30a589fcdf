// Xoshiro128++ PRNG (F18), Box-Muller, randrange, and gather (F17).
//
// Seeding follows vulkpy/_vkarray.cc:643-675 bit for bit: four chained
// splitmix64 outputs (589-595, 658-663) give state 0 and state i is the
// reference's jump() (597-621) applied to state i-1.  That jump assigns the
// state inside the loop over the four JUMP words without resetting its
// accumulators, so it is not Vigna's canonical 2^64 jump, but it is still
// linear over GF(2): the 128x128 bit matrix of one jump lets every host thread
// start at J^lo(state 0) and walk its own range of states sequentially.
//
// Generation replaces the chunked host loop of _vkarray.cc:697-717 (one
// dispatch of `size` threads per chunk, host wait between chunks) by one
// kernel: thread i keeps state i in registers and produces outputs
// i, i + S, i + 2S, ... < n, which is exactly the reference's mapping.
#include "common.h"
#include "fastdiv.h"
#include "bmath.h"

#include <algorithm>
#include <array>
#include <thread>

namespace vkh {

// ---- host seeding ---------------------------------------------------------------
struct St {
  uint32_t w[4];
};

static inline uint32_t rotl32(uint32_t x, int k) { return (x << k) | (x >> (32 - k)); }

static inline void next_host(St& s) {
  const uint32_t t = s.w[1] << 9;
  s.w[2] ^= s.w[0];
  s.w[3] ^= s.w[1];
  s.w[1] ^= s.w[2];
  s.w[0] ^= s.w[3];
  s.w[2] ^= t;
  s.w[3] = rotl32(s.w[3], 11);
}

static inline uint64_t splitmix64(uint64_t x) {
  uint64_t z = (x += 0x9e3779b97f4a7c15ull);
  z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
  z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
  return z ^ (z >> 31);
}

// the jump exactly as _vkarray.cc:597-621 writes it
static inline void jump_as_written(St& s) {
  static const uint32_t JUMP[4] = {0x8764000b, 0xf542d2d3, 0x6fa035c3, 0x77f2db5b};
  uint32_t a0 = 0, a1 = 0, a2 = 0, a3 = 0;
  for (uint32_t j : JUMP) {
    for (int b = 0; b < 32; ++b) {
      if (j & (1u << b)) { a0 ^= s.w[0]; a1 ^= s.w[1]; a2 ^= s.w[2]; a3 ^= s.w[3]; }
      next_host(s);
    }
    s.w[0] = a0; s.w[1] = a1; s.w[2] = a2; s.w[3] = a3;
  }
}

using Mat = std::array<St, 128>;  // column k = image of basis vector e_k

static St mat_apply(const Mat& M, const St& x) {
  St y{{0, 0, 0, 0}};
  for (int k = 0; k < 128; ++k)
    if (x.w[k >> 5] & (1u << (k & 31)))
      for (int q = 0; q < 4; ++q) y.w[q] ^= M[k].w[q];
  return y;
}

// A's images of every byte at every place, for many products with A: 16 table
// look-ups a vector instead of a test of 128 bits
struct ByteTable {
  std::vector<St> t;  // [16][256]
  explicit ByteTable(const Mat& A) : t(16 * 256) {
    for (int b = 0; b < 16; ++b) {
      St* u = &t[b * 256];
      u[0] = St{{0, 0, 0, 0}};
      for (int v = 1; v < 256; ++v) {
        const St& c = A[8 * b + __builtin_ctz(v)];
        for (int q = 0; q < 4; ++q) u[v].w[q] = u[v & (v - 1)].w[q] ^ c.w[q];
      }
    }
  }
  St apply(const St& x) const {
    St y{{0, 0, 0, 0}};
    for (int b = 0; b < 16; ++b) {
      const St& c = t[b * 256 + ((x.w[b >> 2] >> (8 * (b & 3))) & 255u)];
      for (int q = 0; q < 4; ++q) y.w[q] ^= c.w[q];
    }
    return y;
  }
  Mat after(const Mat& B) const {  // A after B
    Mat C;
    for (int k = 0; k < 128; ++k) C[k] = apply(B[k]);
    return C;
  }
};

static Mat compose(const Mat& A, const Mat& B) { return ByteTable(A).after(B); }  // A after B

static Mat identity() {
  Mat I;
  for (int k = 0; k < 128; ++k) {
    I[k] = St{{0, 0, 0, 0}};
    I[k].w[k >> 5] = 1u << (k & 31);
  }
  return I;
}

static Mat jump_matrix() {
  Mat J;
  for (int k = 0; k < 128; ++k) {
    St e{{0, 0, 0, 0}};
    e.w[k >> 5] = 1u << (k & 31);
    jump_as_written(e);
    J[k] = e;
  }
  return J;
}

static Mat mat_pow(Mat base, uint64_t p) {
  Mat r = identity();
  while (p) {
    if (p & 1) r = compose(base, r);
    base = compose(base, base);
    p >>= 1;
  }
  return r;
}

// one step of next() as a matrix (the state update is linear; the ++ output
// scrambler is not part of it)
static Mat step_matrix() {
  Mat M;
  for (int k = 0; k < 128; ++k) {
    St e{{0, 0, 0, 0}};
    e.w[k >> 5] = 1u << (k & 31);
    next_host(e);
    M[k] = e;
  }
  return M;
}

// M^(Lc * d * 16^j), j < ndigits, d = 1 .. 15, as [ndigits][15][128 columns][4
// words]: the start of chunk c takes one product for each hexadecimal digit of
// c that is not 0.  Kept per chunk length (generators made by the same
// initializer shapes share them), the last 32 lengths.
static void chunk_jumps(uint64_t Lc, int ndigits, std::vector<uint32_t>& out) {
  static std::mutex mu;
  static std::unordered_map<uint64_t, std::vector<uint32_t>> cache;
  std::lock_guard<std::mutex> lock(mu);
  if (cache.size() >= 32 && !cache.count(Lc)) cache.clear();
  std::vector<uint32_t>& v = cache[Lc];
  constexpr size_t DIGIT = 15 * 512;
  auto put = [&](int j, int d, const Mat& P) {
    for (int k = 0; k < 128; ++k) std::memcpy(&v[j * DIGIT + (size_t)(d - 1) * 512 + 4 * k], P[k].w, 16);
  };
  auto get = [&](int j, int d) {
    Mat P;
    for (int k = 0; k < 128; ++k) std::memcpy(P[k].w, &v[j * DIGIT + (size_t)(d - 1) * 512 + 4 * k], 16);
    return P;
  };
  const int have = (int)(v.size() / DIGIT);
  if (have < ndigits) v.resize(ndigits * DIGIT);
  for (int j = have; j < ndigits; ++j) {
    const Mat one = j == 0 ? mat_pow(step_matrix(), Lc) : compose(get(j - 1, 1), get(j - 1, 15));
    const ByteTable t(one);
    Mat P = one;
    put(j, 1, P);
    for (int d = 2; d < 16; ++d) put(j, d, P = t.after(P));
  }
  out.assign(v.begin(), v.begin() + ndigits * DIGIT);
}

static void seed_states(uint32_t S, uint64_t seed, std::vector<uint32_t>& out) {
  out.resize((size_t)4 * S);
  St s0;
  for (int i = 0; i < 4; ++i) {
    seed = splitmix64(seed);
    s0.w[i] = (uint32_t)seed;
  }
  unsigned T = std::thread::hardware_concurrency();
  if (T < 1) T = 1;
  if (T > 16) T = 16;
  if (S < 4096) T = 1;
  const uint64_t per = ceil_div(S, T);
  Mat J = T > 1 ? jump_matrix() : Mat{};
  auto work = [&](uint64_t lo, uint64_t hi) {
    St s = lo == 0 ? s0 : mat_apply(mat_pow(J, lo), s0);
    for (uint64_t i = lo; i < hi; ++i) {
      if (i > lo) jump_as_written(s);
      std::memcpy(&out[4 * i], s.w, 16);
    }
  };
  if (T == 1) { work(0, S); return; }
  std::vector<std::thread> th;
  for (unsigned t = 0; t < T; ++t) {
    uint64_t lo = t * per, hi = std::min<uint64_t>(S, lo + per);
    if (lo >= hi) break;
    th.emplace_back(work, lo, hi);
  }
  for (auto& x : th) x.join();
}

// ---- device generation ------------------------------------------------------------
__device__ __forceinline__ uint32_t drotl(uint32_t x, int k) { return (x << k) | (x >> (32 - k)); }

// prng_xoshiro128pp_uint32.comp:32-42
__device__ __forceinline__ uint32_t dnext(uint4& s) {
  const uint32_t result = drotl(s.x + s.w, 7) + s.x;
  const uint32_t t = s.y << 9;
  s.z ^= s.x;
  s.w ^= s.y;
  s.y ^= s.z;
  s.x ^= s.w;
  s.z ^= t;
  s.w = drotl(s.w, 11);
  return result;
}

// prng_xoshiro128pp_float.comp:33
__device__ __forceinline__ float to_unit(uint32_t r) {
  return __uint_as_float((r >> 9) | 0x3f800000u) - 1.0f;
}

constexpr int PRNG_BLOCK = 256;

// NT: nontemporal stores, where the states' outputs of a step are whole 128-byte
// lines (2^20 states, 2^28 outputs 201 us, 212 without, 2^22 6.7 and 7.5);
// elsewhere they would write lines in parts (65534 states, 2^26 outputs 104 us,
// 51 without, 500 states, 2^27 243 and 185).
template <bool NT, typename T>
__device__ __forceinline__ void store_out(T* p, T v) {
  if constexpr (NT) __builtin_nontemporal_store(v, p);
  else *p = v;
}

// OUT: 0 = uint32, 1 = float in [0, 1), 2 = randrange
template <int OUT, bool NT>
__global__ void __launch_bounds__(PRNG_BLOCK)
k_xoshiro(uint4* state, void* out, uint32_t S, uint64_t n, uint32_t low, uint32_t range) {
  const uint64_t i = (uint64_t)blockIdx.x * PRNG_BLOCK + threadIdx.x;
  if (i >= S || i >= n) return;
  uint4 s = state[i];
  for (uint64_t k = i; k < n; k += S) {
    const uint32_t r = dnext(s);
    if (OUT == 0) store_out<NT>(static_cast<uint32_t*>(out) + k, r);
    else if (OUT == 1) store_out<NT>(static_cast<float*>(out) + k, to_unit(r));
    else {
      // prng_randrange.comp:24-26: low + uint(float(range) * u)
      const float u = to_unit(r);
      store_out<NT>(static_cast<uint32_t*>(out) + k, low + __float2uint_rz((float)range * u));
    }
  }
  state[i] = s;
}

// ---- chunked generation for few states ---------------------------------------------
// With S states and n outputs each state takes up to ceil(n / S) sequential
// steps; when S is small (the reference's HeNormal uses 64 states,
// nn/initializers.py:75-89) that serial chain is the whole kernel.  Here
// thread (i, c) produces steps [c*Lc, (c+1)*Lc) of state i: it starts from
// M^(c*Lc) applied to the state (M = one next() step over GF(2)), one
// precomputed matrix M^(Lc * d * 16^j) for each hexadecimal digit d of c.  Outputs
// keep the mapping k = t*S + i.  Start states are read from a copy of the
// state buffer; the chunk holding a state's last step writes it back.
// UNI (64 states, or pairs, and more): a block has one c, so the matrices come
// by scalar loads, many columns ahead, and each column is a mask and four
// ands and xors.  With a matrix for each bit of c, every column a branch and a
// load, a start took longer than 256 steps. 64 states, 2^20 outputs 51 -> 14 us
// (normal 138 -> 33), 4822 states, 12.2 million 45 -> 22 (125 -> 45), 64 states, 2^24
// 75 -> 26 (188 -> 69). The matrices of a new chunk length take the host 0.1 ms (0.5).

// y = P x for a 128x128 bit matrix given by its columns (4 words each)
__device__ __forceinline__ uint4 gf2_apply(const uint32_t* __restrict__ P, uint4 x) {
  uint4 y = make_uint4(0u, 0u, 0u, 0u);
  const uint32_t w[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
  for (int q = 0; q < 4; ++q) {
#pragma unroll 8
    for (int b = 0; b < 32; ++b) {
      const uint4 col = *reinterpret_cast<const uint4*>(P + (q * 32 + b) * 4);
      const uint32_t m = 0u - ((w[q] >> b) & 1u);
      y.x ^= col.x & m; y.y ^= col.y & m; y.z ^= col.z & m; y.w ^= col.w & m;
    }
  }
  return y;
}

__device__ __forceinline__ uint4 chunk_start(uint4 s, const uint32_t* jumps, uint64_t c) {
  for (int j = 0; (c >> (4 * j)) != 0; ++j) {
    const uint32_t d = (uint32_t)(c >> (4 * j)) & 15u;
    if (d) s = gf2_apply(jumps + ((size_t)j * 15 + d - 1) * 512, s);
  }
  return s;
}

// the state (pair) and the chunk of a thread: UNI as a grid of blocks by chunks,
// otherwise one after the other
template <bool UNI>
__device__ __forceinline__ bool chunk_of(uint64_t units, uint64_t nchunks, uint64_t& u, uint64_t& c) {
  const uint64_t tid = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  u = UNI ? tid : tid % units;
  c = UNI ? blockIdx.y : tid / units;
  return UNI ? tid < units : c < nchunks;
}

// steps of state i when n outputs are taken round-robin from S states
__device__ __forceinline__ uint64_t steps_of(uint64_t i, uint64_t S, uint64_t n) {
  return n > i ? (n - 1 - i) / S + 1 : 0;
}

template <int OUT, bool UNI, bool NT>
__global__ void __launch_bounds__(PRNG_BLOCK)
k_xoshiro_chunked(const uint4* init, uint4* state, const uint32_t* jumps, void* out, uint32_t S,
                  uint64_t n, uint64_t Lc, uint64_t nchunks, uint32_t low, uint32_t range) {
  uint64_t i, c;
  if (!chunk_of<UNI>(S, nchunks, i, c)) return;
  const uint64_t L = steps_of(i, S, n);
  const uint64_t t0 = c * Lc;
  if (t0 >= L) return;
  const uint64_t t1 = min(t0 + Lc, L);
  uint4 s = chunk_start(init[i], jumps, c);
  for (uint64_t t = t0; t < t1; ++t) {
    const uint64_t k = t * S + i;
    const uint32_t r = dnext(s);
    if (OUT == 0) store_out<NT>(static_cast<uint32_t*>(out) + k, r);
    else if (OUT == 1) store_out<NT>(static_cast<float*>(out) + k, to_unit(r));
    else store_out<NT>(static_cast<uint32_t*>(out) + k, low + __float2uint_rz((float)range * to_unit(r)));
  }
  if (t1 == L) state[i] = s;
}

// ln t for t in [2^-23, 1] (t = 1 - u of a generated uniform): the hardware
// log2, times ln 2 held as two floats with the rounding error of the leading
// product recovered by an FMA.  On this range (no zero, denormal or infinite
// input) these are the device logf's own steps, so the result is the same
// without its range handling.
constexpr float LN2F_HI = 0x1.62e42ep-1f, LN2F_LO = 0x1.efa39ep-25f;  // hi + lo = ln 2
__device__ __forceinline__ float log_unit(float t) {
  const float l2 = __builtin_amdgcn_logf(t);
  const float p = l2 * LN2F_HI;
  const float e = fmaf(l2, LN2F_LO, fmaf(l2, LN2F_HI, -p));
  return p + e;
}

// Correctly rounded sqrt x for x in [0, 2^96): the hardware square root, then
// whichever neighbour's product with it brackets x (x = 0 stays 0: the lower
// neighbour's residual is NaN, the upper one's is -0).
__device__ __forceinline__ float sqrt_rn(float x) {
  const float s = __builtin_amdgcn_sqrtf(x);
  const float sm = __int_as_float(__float_as_int(s) - 1), sp = __int_as_float(__float_as_int(s) + 1);
  const float r = fmaf(-sm, s, x) <= 0.0f ? sm : s;
  return fmaf(-sp, s, x) > 0.0f ? sp : r;
}

// Box-Muller of one pair of uniforms (prng_box_muller.comp:25-31) in the
// reference's FP32 operation order; sin and cos come from sincos_small (the
// GLSL.std.450 functions the reference relies on are likewise FP32 within a
// few ulp).  GEN: u1 is a generated uniform in [0, 1), so log and sqrt take
// the range-specific forms above; otherwise (uniforms from a caller's
// buffer) the device logf and sqrtf.
template <bool GEN>
__device__ __forceinline__ void box_muller(float u1, float u2, float mean, float sd, float& o1, float& o2) {
  const float t = 1.0f - u1;
  const float l = GEN ? log_unit(t) : logf(t);
  const float r = (GEN ? sqrt_rn(-2.0f * l) : sqrtf(-2.0f * l)) * sd;
  const float angle = 6.28318530718f * u2;
  float s, c;
  sincos_small(angle, s, c);
  o1 = mean + r * s;
  o2 = mean + r * c;
}

typedef float vkh_f2v __attribute__((ext_vector_type(2)));

// out[j] (j < n) and out[j + 1] (j + 1 < n) of a normal pair; one 8-byte
// store when both are in range and out + j is 8-byte aligned
template <bool NT>
__device__ __forceinline__ void store_pair(float* out, uint64_t j, uint64_t n, float o1, float o2) {
  if (j + 1 < n && ((uintptr_t)(out + j) & 7u) == 0) {
    const vkh_f2v v = {o1, o2};
    store_out<NT>(reinterpret_cast<vkh_f2v*>(out + j), v);
  } else {
    if (j < n) store_out<NT>(out + j, o1);
    if (j + 1 < n) store_out<NT>(out + j + 1, o2);
  }
}

// Fused uniform + Box-Muller: thread p owns states 2p and 2p+1 (S even) and
// produces normal pairs at uniform indices j = c*S + 2p < nu (nu even).
// PAIRED: n == nu and out 8-byte aligned, so every pair is one 8-byte store.
template <bool PAIRED, bool NT>
__global__ void __launch_bounds__(PRNG_BLOCK)
k_xoshiro_normal(uint4* state, float* out, uint32_t S, uint64_t nu, uint64_t n, float mean, float sd) {
  const uint64_t p = (uint64_t)blockIdx.x * PRNG_BLOCK + threadIdx.x;
  const uint64_t i = 2 * p;
  if (i >= S || i >= nu) return;
  uint4 s1 = state[i], s2 = state[i + 1];
  for (uint64_t j = i; j < nu; j += S) {
    const float u1 = to_unit(dnext(s1));
    const float u2 = to_unit(dnext(s2));
    float o1, o2;
    box_muller<true>(u1, u2, mean, sd, o1, o2);
    if constexpr (PAIRED) {
      const vkh_f2v v = {o1, o2};
      store_out<NT>(reinterpret_cast<vkh_f2v*>(out + j), v);
    } else {
      store_pair<NT>(out, j, n, o1, o2);
    }
  }
  state[i] = s1;
  state[i + 1] = s2;
}

// chunked form of k_xoshiro_normal: thread (p, c) advances states 2p and 2p+1
// over steps [c*Lc, (c+1)*Lc); both take the same number of steps because S
// and nu are even
template <bool UNI, bool NT>
__global__ void __launch_bounds__(PRNG_BLOCK)
k_xoshiro_normal_chunked(const uint4* init, uint4* state, const uint32_t* jumps, float* out,
                         uint32_t S, uint64_t nu, uint64_t n, uint64_t Lc, uint64_t nchunks,
                         float mean, float sd) {
  uint64_t p, c;
  if (!chunk_of<UNI>(S / 2, nchunks, p, c)) return;
  const uint64_t i = 2 * p;
  const uint64_t L = steps_of(i, S, nu);
  const uint64_t t0 = c * Lc;
  if (t0 >= L) return;
  const uint64_t t1 = min(t0 + Lc, L);
  uint4 s1 = chunk_start(init[i], jumps, c), s2 = chunk_start(init[i + 1], jumps, c);
  for (uint64_t t = t0; t < t1; ++t) {
    const uint64_t j = t * S + i;
    const float u1 = to_unit(dnext(s1));
    const float u2 = to_unit(dnext(s2));
    float o1, o2;
    box_muller<true>(u1, u2, mean, sd, o1, o2);
    store_pair<NT>(out, j, n, o1, o2);
  }
  if (t1 == L) {
    state[i] = s1;
    state[i + 1] = s2;
  }
}

__global__ void __launch_bounds__(PRNG_BLOCK)
k_box_muller(const float* u, float* out, uint64_t npairs, uint64_t n, float mean, float sd) {
  const uint64_t stride = (uint64_t)gridDim.x * PRNG_BLOCK;
  for (uint64_t p = (uint64_t)blockIdx.x * PRNG_BLOCK + threadIdx.x; p < npairs; p += stride) {
    const uint64_t j = 2 * p;
    const float u1 = u[j], u2 = u[j + 1];
    float o1, o2;
    box_muller<false>(u1, u2, mean, sd, o1, o2);
    if (j < n) out[j] = o1;
    if (j + 1 < n) out[j + 1] = o2;
  }
}

// ---- gather --------------------------------------------------------------------------
__global__ void __launch_bounds__(256)
k_gather(const float* a, uint64_t na, const uint32_t* idx, float* c, uint64_t n) {
  const uint64_t stride = (uint64_t)gridDim.x * 256;
  for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += stride) {
    uint64_t k = idx[i];
    c[i] = a[k < na ? k : na - 1];
  }
}

// c[k, p, j] = a[p, min(idx[k], axis-1), j]: a copy of nidx * prev runs of post
// elements.  A thread moves 4 consecutive elements of a run (the last group of a
// run starts at post - 4; 16-byte accesses at any alignment), with the run and
// its k and p from 32-bit multiply-high divisions.  HBM-bound; against one
// element a thread with three 64-bit divisions: 8192 rows of 784 7.2 against 18
// us, 4096 of 4096 12 against 39, [1000, 100, 50] along axis 1 23.5 against 40.
typedef __attribute__((ext_vector_type(4), aligned(4))) uint32_t u32x4u_t;

__global__ void __launch_bounds__(256)
k_gather_runs(const uint32_t* a, const uint32_t* idx, uint32_t* c, FastDiv prev, uint64_t axis, uint32_t post,
              FastDiv upr, uint32_t units) {
  const uint32_t t = blockIdx.x * 256 + threadIdx.x;
  if (t >= units) return;
  const uint32_t r = upr.div(t), u = t - r * upr.d;  // run k * prev + p, its unit
  const uint32_t k = prev.div(r), p = r - k * prev.d;
  const uint64_t b = min((uint64_t)idx[k], axis - 1);
  const uint32_t j = min(u * 4, post - 4);
  const u32x4u_t v = *reinterpret_cast<const u32x4u_t*>(a + ((uint64_t)p * axis + b) * post + j);
  __builtin_nontemporal_store(v, reinterpret_cast<u32x4u_t*>(c + (uint64_t)r * post + j));
}

// the same one element a thread: runs of 1 to 3 elements
__global__ void __launch_bounds__(256)
k_gather_elems(const uint32_t* a, const uint32_t* idx, uint32_t* c, FastDiv prev, uint64_t axis, FastDiv post,
               uint32_t total) {
  const uint32_t t = blockIdx.x * 256 + threadIdx.x;
  if (t >= total) return;
  const uint32_t r = post.div(t), j = t - r * post.d;
  const uint32_t k = prev.div(r), p = r - k * prev.d;
  const uint64_t b = min((uint64_t)idx[k], axis - 1);
  c[t] = a[((uint64_t)p * axis + b) * post.d + j];
}

// any size
__global__ void __launch_bounds__(256)
k_gather_axis(const float* a, const uint32_t* idx, float* c, uint64_t prev, uint64_t axis,
              uint64_t post, uint64_t nidx) {
  const uint64_t total = nidx * prev * post;
  const uint64_t stride = (uint64_t)gridDim.x * 256;
  for (uint64_t t = (uint64_t)blockIdx.x * 256 + threadIdx.x; t < total; t += stride) {
    const uint64_t j = t % post;
    const uint64_t q = t / post;
    const uint64_t p = q % prev;
    const uint64_t k = q / prev;
    uint64_t b = idx[k];
    if (b >= axis) b = axis - 1;
    c[t] = a[(p * axis + b) * post + j];
  }
}

// out[k, j] = 1 if min(idx[k], classes - 1) == j else 0: the one-hot rows the
// reference gathers from an identity matrix (vkarray.py:239-253), out-of-range
// labels clamped like gather_axis.  Four outputs a thread over the flat output
// (n * classes < 2^31; a group may cross rows): 8192 x 1000 7 against 10 us one
// at a time.
__global__ void __launch_bounds__(256)
k_onehot4(const uint32_t* idx, float* out, uint32_t total, FastDiv classes) {
  const uint32_t i = (blockIdx.x * 256 + threadIdx.x) * 4;
  if (i >= total) return;
  uint32_t k = classes.div(i), j = i - k * classes.d;
  const uint32_t n = min(4u, total - i);
  float v[4];
  uint32_t lab = min(idx[k], classes.d - 1);
#pragma unroll
  for (uint32_t q = 0; q < 4; ++q) {
    v[q] = lab == j ? 1.0f : 0.0f;
    if (++j == classes.d) {
      j = 0;
      if (q + 1 < n) lab = min(idx[++k], classes.d - 1);
    }
  }
  if (n == 4) {
    typedef __attribute__((ext_vector_type(4), aligned(4))) float f32x4u_t;
    *reinterpret_cast<f32x4u_t*>(out + i) = f32x4u_t{v[0], v[1], v[2], v[3]};
  } else {
    for (uint32_t q = 0; q < n; ++q) out[i + q] = v[q];
  }
}

// any size
__global__ void __launch_bounds__(256)
k_onehot(const uint32_t* idx, float* out, uint64_t n, uint32_t classes) {
  const uint64_t total = n * classes;
  const uint64_t stride = (uint64_t)gridDim.x * 256;
  for (uint64_t t = (uint64_t)blockIdx.x * 256 + threadIdx.x; t < total; t += stride) {
    const uint64_t k = t / classes;
    const uint32_t j = (uint32_t)(t - k * classes);
    const uint32_t lab = min(idx[k], classes - 1);
    out[t] = lab == j ? 1.0f : 0.0f;
  }
}

}  // namespace vkh

struct JumpTable {
  uint64_t lc = 0;  // chunk length
  int ndigits = 0;
  uint32_t* dev = nullptr;
  uint64_t used = 0;  // number of the last draw that took it
};

struct vkh_xoshiro {
  vkh_gpu* gpu = nullptr;
  uint32_t size = 0;
  uint32_t* state = nullptr;  // [size][4]
  bool from_alloc = false;
  // jump matrices of the chunked kernels, for the chunk lengths used last
  std::vector<JumpTable> jumps;
  uint64_t draws = 0;
};

using namespace vkh;

static unsigned prng_grid(uint64_t threads) { return (unsigned)ceil_div(threads, PRNG_BLOCK); }

namespace {

struct ChunkPlan {
  bool use = false;
  uint64_t Lc = 0, C = 1;
  int ndigits = 0;
  bool uni = false;  // one chunk a block
  dim3 grid, block;
};

constexpr uint64_t CHUNK_FULL = 128, CHUNK_MIN = 64, CHUNK_MIN_NORMAL = 32;  // steps of a chunk, at least
constexpr uint64_t CHUNKED_MIN = 512, CHUNKED_MIN_NORMAL = 128;                       // steps of a chain, at least

// Chunk the per-state chains when `units` parallel chains (states, or state
// pairs) are too few to fill the GPU and each is long.  Up to 512 threads per
// compute unit a chunk may be as short as `least` steps, its start-state products
// hidden by other waves' work, up to 1024 as CHUNK_FULL; fewer than four chunks
// do not pay for the copy of the states (65534 states, 2^23 outputs 14.6 us in
// two chunks, 10.6 without), nor do uniform chains under eight chunks for the first
// draws of new sizes (64 states, 8200 to 32700 outputs, no size twice: 24 us a draw in
// chunks, 15 without; normal 23 and 71; 2^14 outputs again and again 9.6 and 12.5).  Under
// 64 units a block of one chunk has idle lanes, which only pays where the chip
// has room for every such wave (32 pairs, 2^20 outputs 33 us against 53, 2^28 548
// against 363).  Not during graph capture (the jump matrices are uploaded
// synchronously).
ChunkPlan plan_chunks(const vkh_gpu* g, uint64_t units, uint64_t steps, uint64_t least, uint64_t chain) {
  ChunkPlan p;
  if (g->capturing || steps < chain) return p;
  const uint64_t cus = g->num_cus > 0 ? g->num_cus : 256, target = cus * 1024;
  if (units * 4 >= target) return p;
  const uint64_t full = std::min(ceil_div(target, units), steps / CHUNK_FULL);
  uint64_t C = std::max(full, std::min(ceil_div(target / 2, units), steps / least));
  p.uni = units >= 64 ? C < 65536 : units >= 16 && C <= 4 * cus;
  if (!p.uni) C = full;
  if (C < 2) return p;
  p.Lc = ceil_div(steps, C);
  p.C = ceil_div(steps, p.Lc);
  if (p.C < 2) return p;
  p.use = true;
  while (((p.C - 1) >> (4 * p.ndigits)) != 0) ++p.ndigits;  // digits of c < C
  if (p.uni) {
    p.block = dim3((unsigned)std::min<uint64_t>(PRNG_BLOCK, ceil_div(units, 64) * 64));
    p.grid = dim3((unsigned)ceil_div(units, p.block.x), (unsigned)p.C);
  } else {
    p.block = dim3(PRNG_BLOCK);
    p.grid = dim3(prng_grid(units * p.C));
  }
  return p;
}

// At most 8 lengths a generator (30 to 120 KB each): uniform and normal draws of
// a size have different ones, and draws of several sizes alternate.  A known length
// costs nothing.  A new one goes to memory of its own, which no kernel reads yet, so
// its copy waits for no queued work; only the memory of a length given up does.
// 2^20 uniform and 2^20 normal draws from 64 states in turn 46 us the two, 105 with
// one length a generator and a wait for every switch.
constexpr size_t JUMP_TABLES = 8;

const uint32_t* prepare_jumps(vkh_xoshiro* r, const ChunkPlan& p) {
  const uint64_t now = ++r->draws;
  auto& ts = r->jumps;
  auto t = std::find_if(ts.begin(), ts.end(), [&](const JumpTable& x) { return x.lc == p.Lc; });
  if (t != ts.end() && t->ndigits >= p.ndigits) {
    t->used = now;
    return t->dev;
  }
  if (t == ts.end() && ts.size() == JUMP_TABLES)
    t = std::min_element(ts.begin(), ts.end(), [](const JumpTable& a, const JumpTable& b) { return a.used < b.used; });
  std::vector<uint32_t> host;
  chunk_jumps(p.Lc, p.ndigits, host);
  if (t != ts.end()) {  // too few digits, or the least recently used: queued draws may read it
    VKH_HIP(hipStreamSynchronize(r->gpu->stream));
    uint32_t* old = t->dev;
    ts.erase(t);
    VKH_HIP(hipFree(old));
  }
  const size_t nbytes = host.size() * sizeof(uint32_t);
  JumpTable n{p.Lc, p.ndigits, nullptr, now};
  ts.reserve(JUMP_TABLES);
  VKH_HIP(hipMalloc(&n.dev, nbytes));
  const hipError_t e = hipMemcpy(n.dev, host.data(), nbytes, hipMemcpyHostToDevice);
  if (e != hipSuccess) {
    (void)hipFree(n.dev);
    check_hip(e, "hipMemcpy");
  }
  ts.push_back(n);
  return n.dev;
}

// the stores of store_out<true>: see there
bool whole_lines(const vkh_xoshiro* r, const void* out) {
  return r->size % 32 == 0 && ((uintptr_t)out & 127u) == 0;
}

template <int OUT>
void launch_uniform(vkh_xoshiro* r, void* out, uint64_t n, uint32_t low, uint32_t range) {
  vkh_gpu* g = r->gpu;
  const bool nt = whole_lines(r, out);
  const ChunkPlan cp = plan_chunks(g, r->size, ceil_div(n, r->size), CHUNK_MIN, CHUNKED_MIN);
  if (cp.use) {
    const uint32_t* jumps = prepare_jumps(r, cp);
    const size_t sb = (size_t)16 * r->size;
    Workspace init(g, sb);
    VKH_HIP(hipMemcpyAsync(init.get(), r->state, sb, hipMemcpyDeviceToDevice, g->stream));
    auto kernel = !cp.uni ? k_xoshiro_chunked<OUT, false, false>
                  : nt    ? k_xoshiro_chunked<OUT, true, true>
                          : k_xoshiro_chunked<OUT, true, false>;
    hipLaunchKernelGGL(kernel, cp.grid, cp.block, 0, g->stream, (const uint4*)init.get(), (uint4*)r->state, jumps, out,
                       r->size, n, cp.Lc, cp.C, low, range);
  } else {
    // one state per thread (measured 197 us for 2^28 outputs from 2^20 states;
    // four states per thread with 16-byte stores: 232 us; four steps of a
    // block's 256 states staged through LDS so that each wave stores one
    // 1 KB row segment with 16-byte stores: no faster)
    const uint64_t th = std::min<uint64_t>(r->size, n);
    auto kernel = nt ? k_xoshiro<OUT, true> : k_xoshiro<OUT, false>;
    hipLaunchKernelGGL(kernel, dim3(prng_grid(th)), dim3(PRNG_BLOCK), 0, g->stream, (uint4*)r->state, out, r->size, n,
                       low, range);
  }
  check_launch("xoshiro");
}

}  // namespace

extern "C" {

int vkh_xoshiro_create(vkh_gpu* g, uint32_t size, uint64_t seed, vkh_xoshiro** out) {
  return guarded([&] {
    use(g);
    VKH_REQUIRE(out, "null out");
    VKH_REQUIRE(size >= 1, "Xoshiro128pp size must be at least 1");
    std::vector<uint32_t> host;
    seed_states(size, seed, host);
    auto* r = new vkh_xoshiro();
    r->gpu = g;
    r->size = size;
    const size_t nbytes = sizeof(uint32_t) * 4 * (size_t)size;
    try {
      if (g->alloc) {
        r->state = (uint32_t*)g->alloc->allocate(nbytes);
        r->from_alloc = true;
      } else {
        VKH_HIP(hipMalloc(&r->state, nbytes));
      }
      // synchronous copy: the host vector dies at the end of this call
      VKH_HIP(hipMemcpyAsync(r->state, host.data(), nbytes, hipMemcpyHostToDevice, g->stream));
      VKH_HIP(hipStreamSynchronize(g->stream));
    } catch (...) {
      if (r->state) { if (r->from_alloc) g->alloc->release(r->state); else (void)hipFree(r->state); }
      delete r;
      throw;
    }
    *out = r;
  });
}

int vkh_xoshiro_destroy(vkh_xoshiro* r) {
  return guarded([&] {
    if (!r) return;
    use(r->gpu);
    VKH_REQUIRE(!r->gpu->capturing, "xoshiro_destroy: not allowed during graph capture");
    if (r->from_alloc) r->gpu->alloc->release(r->state);
    else { VKH_HIP(hipStreamSynchronize(r->gpu->stream)); VKH_HIP(hipFree(r->state)); }
    if (!r->jumps.empty()) VKH_HIP(hipStreamSynchronize(r->gpu->stream));
    for (const JumpTable& t : r->jumps) VKH_HIP(hipFree(t.dev));
    delete r;
  });
}

int vkh_xoshiro_size(vkh_xoshiro* r, uint32_t* out) {
  return guarded([&] { VKH_REQUIRE(r && out, "null argument"); *out = r->size; });
}

int vkh_xoshiro_state(vkh_xoshiro* r, uint32_t** out) {
  return guarded([&] { VKH_REQUIRE(r && out, "null argument"); *out = r->state; });
}

int vkh_xoshiro_uint32(vkh_xoshiro* r, uint32_t* out, uint64_t n) {
  return guarded([&] {
    VKH_REQUIRE(r, "null generator");
    use(r->gpu);
    if (n == 0) return;
    VKH_REQUIRE(out, "null output");
    launch_uniform<0>(r, out, n, 0u, 0u);
  });
}

int vkh_xoshiro_float(vkh_xoshiro* r, float* out, uint64_t n) {
  return guarded([&] {
    VKH_REQUIRE(r, "null generator");
    use(r->gpu);
    if (n == 0) return;
    VKH_REQUIRE(out, "null output");
    launch_uniform<1>(r, out, n, 0u, 0u);
  });
}

int vkh_xoshiro_randrange(vkh_xoshiro* r, uint32_t* out, uint64_t n, uint32_t low, uint32_t high_incl) {
  return guarded([&] {
    VKH_REQUIRE(r, "null generator");
    use(r->gpu);
    if (n == 0) return;
    VKH_REQUIRE(out, "null output");
    uint32_t range = high_incl - low + 1u;  // uint32 arithmetic as in the shader
    launch_uniform<2>(r, out, n, low, range);
  });
}

int vkh_box_muller(vkh_gpu* g, const float* u, float* out, uint64_t n, float mean, float sd) {
  return guarded([&] {
    use(g);
    if (n == 0) return;
    VKH_REQUIRE(u && out, "null pointer");
    uint64_t npairs = ceil_div(n, 2);
    unsigned grid = stream_grid(g, npairs, PRNG_BLOCK, 8);
    hipLaunchKernelGGL(k_box_muller, dim3(grid), dim3(PRNG_BLOCK), 0, g->stream, u, out, npairs, n, mean, sd);
    check_launch("box_muller");
  });
}

int vkh_xoshiro_normal(vkh_xoshiro* r, float* out, uint64_t n, float mean, float sd) {
  return guarded([&] {
    VKH_REQUIRE(r, "null generator");
    vkh_gpu* g = r->gpu;
    use(g);
    if (n == 0) return;
    VKH_REQUIRE(out, "null output");
    const uint64_t nu = n + (n & 1);  // random.py:105-123: n even, or n + 1 uniforms
    if (r->size % 2 == 0) {
      const bool nt = whole_lines(r, out);
      const ChunkPlan cp = plan_chunks(g, r->size / 2, ceil_div(nu, r->size), CHUNK_MIN_NORMAL, CHUNKED_MIN_NORMAL);
      if (cp.use) {
        const uint32_t* jumps = prepare_jumps(r, cp);
        const size_t sb = (size_t)16 * r->size;
        Workspace init(g, sb);
        VKH_HIP(hipMemcpyAsync(init.get(), r->state, sb, hipMemcpyDeviceToDevice, g->stream));
        auto kernel = !cp.uni ? k_xoshiro_normal_chunked<false, false>
                      : nt    ? k_xoshiro_normal_chunked<true, true>
                              : k_xoshiro_normal_chunked<true, false>;
        hipLaunchKernelGGL(kernel, cp.grid, cp.block, 0, g->stream, (const uint4*)init.get(), (uint4*)r->state, jumps,
                           out, r->size, nu, n, cp.Lc, cp.C, mean, sd);
      } else {
        uint64_t th = std::min<uint64_t>(r->size, nu) / 2;
        const bool paired = n == nu && ((uintptr_t)out & 7u) == 0;
        auto kernel = paired ? (nt ? k_xoshiro_normal<true, true> : k_xoshiro_normal<true, false>)
                             : (nt ? k_xoshiro_normal<false, true> : k_xoshiro_normal<false, false>);
        hipLaunchKernelGGL(kernel, dim3(prng_grid(th)), dim3(PRNG_BLOCK), 0, g->stream, (uint4*)r->state, out, r->size,
                           nu, n, mean, sd);
      }
      check_launch("xoshiro normal");
      return;
    }
    // odd number of states: uniforms first, then the transform
    Workspace ws(g, sizeof(float) * nu);
    float* u = (float*)ws.get();
    launch_uniform<1>(r, u, nu, 0u, 0u);
    uint64_t npairs = nu / 2;
    unsigned grid = stream_grid(g, npairs, PRNG_BLOCK, 8);
    hipLaunchKernelGGL(k_box_muller, dim3(grid), dim3(PRNG_BLOCK), 0, g->stream, u, out, npairs, n, mean, sd);
    check_launch("box_muller");
  });
}

int vkh_gather(vkh_gpu* g, const float* a, uint64_t na, const uint32_t* idx, float* c, uint64_t n) {
  return guarded([&] {
    use(g);
    if (n == 0) return;
    VKH_REQUIRE(a && idx && c, "gather: null pointer");
    VKH_REQUIRE(na >= 1, "gather from an empty array");
    unsigned grid = stream_grid(g, n, 256, 8);
    hipLaunchKernelGGL(k_gather, dim3(grid), dim3(256), 0, g->stream, a, na, idx, c, n);
    check_launch("gather");
  });
}

int vkh_onehot(vkh_gpu* g, const uint32_t* idx, uint64_t n, uint32_t classes, float* out) {
  return guarded([&] {
    use(g);
    VKH_REQUIRE(classes >= 1, "onehot: need at least one class");
    if (n == 0) return;
    VKH_REQUIRE(idx && out, "onehot: null pointer");
    if (n < (uint64_t(1) << 31) / classes) {
      const uint32_t total = (uint32_t)(n * classes);
      hipLaunchKernelGGL(k_onehot4, dim3((unsigned)ceil_div(total, 1024)), dim3(256), 0, g->stream, idx, out, total,
                         FastDiv(classes));
      check_launch("onehot");
      return;
    }
    unsigned grid = stream_grid(g, n * classes, 256, 8);
    hipLaunchKernelGGL(k_onehot, dim3(grid), dim3(256), 0, g->stream, idx, out, n, classes);
    check_launch("onehot");
  });
}

int vkh_gather_axis(vkh_gpu* g, const float* a, const uint32_t* idx, float* c, uint64_t prev,
                    uint64_t axis, uint64_t post, uint64_t nidx) {
  return guarded([&] {
    use(g);
    uint64_t total = nidx * prev * post;
    if (total == 0) return;
    VKH_REQUIRE(a && idx && c, "gather_axis: null pointer");
    VKH_REQUIRE(axis >= 1, "gather along an empty axis");
    const uint64_t lim = uint64_t(1) << 31, runs = nidx * prev;
    if (total < lim && prev < lim && nidx < lim && post >= 4) {
      const uint64_t upr = ceil_div(post, 4);  // (runs * upr <= total)
      const uint32_t units = (uint32_t)(runs * upr);
      hipLaunchKernelGGL(k_gather_runs, dim3((unsigned)ceil_div(units, 256)), dim3(256), 0, g->stream,
                         (const uint32_t*)a, idx, (uint32_t*)c, FastDiv((uint32_t)prev), axis, (uint32_t)post,
                         FastDiv((uint32_t)upr), units);
      check_launch("gather_axis");
      return;
    }
    if (total < lim && post >= 1) {
      hipLaunchKernelGGL(k_gather_elems, dim3((unsigned)ceil_div(total, 256)), dim3(256), 0, g->stream,
                         (const uint32_t*)a, idx, (uint32_t*)c, FastDiv((uint32_t)prev), axis, FastDiv((uint32_t)post),
                         (uint32_t)total);
      check_launch("gather_axis");
      return;
    }
    unsigned grid = stream_grid(g, total, 256, 8);
    hipLaunchKernelGGL(k_gather_axis, dim3(grid), dim3(256), 0, g->stream, a, idx, c, prev, axis, post, nidx);
    check_launch("gather_axis");
  });
}

}  // extern "C"
