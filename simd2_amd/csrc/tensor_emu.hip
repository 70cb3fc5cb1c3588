// FP16-input / FP32-accumulate semiring GEMM: the reference's "tensor core
// emulation" semantics (kernel/tensor_srgemm.cuh:37-218) and its FP32<->FP16
// conversions (kernel/precision.cuh:5-33).
//
// Per (i, j) and k in order 0..K-1: the (x) is evaluated in half precision
// (one FP16 rounding), converted to float and folded into a float
// accumulator with fminf / fmaxf / +.  Accumulators start where the
// reference starts them: +inf for min-based ops (__float2half(FLT_MAX)
// overflows to +inf), 0 for max-based ops (__float2half(FLT_MIN) underflows
// to 0 -- so max-based results are clamped below at 0), 0 for the rest.  The
// epilogue folds C the same way; or_and treats values > 0 as true.
//
// Two neighbouring columns share a register (v_pk_*_f16), so a term costs half
// an instruction.  The min- and max-based folds stay in half precision: they
// only select among the half-precision terms, so folding first and converting
// once gives the float the reference ends with.  Two k fold in one
// v_pk_minimum3_f16 / v_pk_maximum3_f16; these keep NaN where the reference's
// fminf / fmaxf drop it, so a workgroup that ends with a NaN runs its tile
// again with v_pk_min_f16 / v_pk_max_f16, which drop it too.  The sums add
// each half-precision term to the float accumulator in k order
// (v_fma_mix_f32, times 1, one rounding).
// Bound: VALU issue; v_pk_* and the three-input forms issue at 0.93 per CU and
// cycle and do not pair, 0.75 instructions a term for min / max, 1.5 and 2 for
// the sums.  min_plus 2048^3 with C: 228 us, 4096^3 1549 (1.23 terms per CU, cycle
// and lane at 2.4 GHz, the bound's 1.24); one output per thread with a
// conversion per term took 811 and 6390.
#include <hip/hip_fp16.h>

#include <algorithm>
#include <type_traits>

#include "internal.hpp"

namespace simd2 {

namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef _Float16 half2v __attribute__((ext_vector_type(2)));

constexpr uint32_t H_INF = 0x7c00u, H_NINF = 0xfc00u;
constexpr int emu_add = 0, emu_mul = 1, emu_min = 2, emu_max = 3, emu_sub2 = 4;

// The operators by opcode: term, fold (0 min, 1 max, 2 sum), and the halves
// that pad A and B past k (their term leaves every accumulator as it is).
template <int OP> struct Emu;
#define EMU(op, t, f, px, py)                                                   \
  template <> struct Emu<op> {                                                  \
    static constexpr int term = t, fold = f;                                    \
    static constexpr uint32_t pad_x = px * 0x10001u, pad_y = py * 0x10001u;     \
  };
EMU(0, emu_add, 0, H_INF, H_INF)     // min_plus
EMU(1, emu_mul, 2, 0u, 0u)           // plus_mul
EMU(2, emu_add, 1, H_NINF, H_NINF)   // max_plus
EMU(3, emu_min, 1, H_NINF, H_NINF)   // max_min
EMU(4, emu_mul, 1, H_NINF, H_INF)    // max_mul
EMU(5, emu_mul, 0, H_INF, H_INF)     // min_mul
EMU(6, emu_max, 0, H_INF, H_INF)     // min_max
EMU(7, emu_min, 1, 0u, 0u)           // or_and: inputs made 0 / 1 when staged
EMU(8, emu_sub2, 2, 0u, 0u)          // minus_square
#undef EMU

// A(i, k) (x) the two columns of b; a holds k (low) and k + 1 (high).  Plain
// vector code: an asm term feeding the asm folds costs an s_nop a pair.
template <int OP, bool HI> __device__ __forceinline__ uint32_t emu_term(uint32_t aw, uint32_t bw) {
  constexpr int t = Emu<OP>::term;
  const half2v av = __builtin_bit_cast(half2v, aw), b = __builtin_bit_cast(half2v, bw);
  const half2v a = HI ? __builtin_shufflevector(av, av, 1, 1) : __builtin_shufflevector(av, av, 0, 0);
  half2v r;
  if constexpr (t == emu_add) r = a + b;
  if constexpr (t == emu_mul) r = a * b;
  if constexpr (t == emu_min) r = __builtin_elementwise_min(a, b);
  if constexpr (t == emu_max) r = __builtin_elementwise_max(a, b);
  if constexpr (t == emu_sub2) {
    const half2v d = a - b;
    r = d * d;
  }
  return __builtin_bit_cast(uint32_t, r);
}

// fold of two / three packed values (min or max); NANS: dropping NaN
template <bool MAX> __device__ __forceinline__ uint32_t emu_fold2(uint32_t x, uint32_t y) {
  uint32_t r;
  if (MAX) asm("v_pk_max_f16 %0, %1, %2" : "=v"(r) : "v"(x), "v"(y));
  else asm("v_pk_min_f16 %0, %1, %2" : "=v"(r) : "v"(x), "v"(y));
  return r;
}
template <bool MAX, bool NANS>
__device__ __forceinline__ uint32_t emu_fold3(uint32_t acc, uint32_t x, uint32_t y) {
  if (NANS) return emu_fold2<MAX>(emu_fold2<MAX>(acc, x), y);
  uint32_t r;
  if (MAX) asm("v_pk_maximum3_f16 %0, %1, %2, %3" : "=v"(r) : "v"(acc), "v"(x), "v"(y));
  else asm("v_pk_minimum3_f16 %0, %1, %2, %3" : "=v"(r) : "v"(acc), "v"(x), "v"(y));
  return r;
}

// acc + float(half of p), one rounding
__device__ __forceinline__ float add_low(float acc, uint32_t p) {
  asm("v_fma_mix_f32 %0, %1, 1.0, %0 op_sel_hi:[1,0,0]" : "+v"(acc) : "v"(p));
  return acc;
}
__device__ __forceinline__ float add_high(float acc, uint32_t p) {
  asm("v_fma_mix_f32 %0, %1, 1.0, %0 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "+v"(acc) : "v"(p));
  return acc;
}

__device__ __forceinline__ float half_to_float(uint32_t h) {
  return __half2float(__ushort_as_half((unsigned short)h));
}

__device__ __forceinline__ float emu_epilogue(int op, float acc, float c) {
  switch (op) {
  case 0: case 5: case 6: return fminf(acc, c);
  case 2: case 3: case 4: return fmaxf(acc, c);
  case 7: return (float)((int)acc || (int)c);
  default: return acc + c;
  }
}

// A T x T tile, 256 threads, TM x TM outputs each as blocks of GR x GR spaced
// T / (TM / GR) apart (valu_tile.hpp's arrangement); KS k per slab.
template <int T_, int TM_> struct EmuTile {
  static constexpr int T = T_, TM = TM_, GR = TM < 4 ? TM : 4, KS = T < 64 ? 64 : 32;
  static constexpr int L = T * KS / 8 / 256;           // 16-byte loads per thread and operand
  static constexpr int NTX = T / TM, S = T / (TM / GR);
  struct Smem {
    // A as [k pair][row] (k low, k + 1 high); B as [k pair][GR columns][2 k][GR]
    __attribute__((aligned(16))) uint32_t A[2][KS / 2][T + 4];
    __attribute__((aligned(16))) uint32_t B[2][KS / 2][T];
  };
  static_assert(L >= 1 && NTX * NTX == 256, "tile");
};

// or_and: a half > 0 as 1, else 0 (both halves of a word).
__device__ __forceinline__ uint32_t as_bool(uint32_t w) {
  const uint32_t lo = half_to_float(w & 0xffffu) > 0.f ? 0x3c00u : 0u;
  const uint32_t hi = half_to_float(w >> 16) > 0.f ? 0x3c000000u : 0u;
  return lo | hi;
}

// Main loop over the slabs [s0, s1) of one tile.
template <int OP, class Tile, bool NANS, bool VEC, class ACC>
__device__ __forceinline__ void emu_loop(typename Tile::Smem &sm, int tid,
                                         const __half *__restrict__ a,
                                         const __half *__restrict__ b, int row0, int col0, int m,
                                         int n, int k, int s0, int s1, ACC &acc) {
  constexpr int T = Tile::T, TM = Tile::TM, GR = Tile::GR, KS = Tile::KS, L = Tile::L;
  constexpr bool SUM = Emu<OP>::fold == 2, MAX = Emu<OP>::fold == 1;
  typedef uint32_t group __attribute__((ext_vector_type(GR)));
  const int tx = tid % Tile::NTX, ty = tid / Tile::NTX;
  u32x4 xv[L], yv[L];
  // 8 halves at p (even when p is only 2-byte aligned)
  auto get = [](const __half *p) {
    if (VEC) return *reinterpret_cast<const u32x4 *>(p);
    const unsigned short *q = reinterpret_cast<const unsigned short *>(p);
    u32x4 v;
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = (uint32_t)q[2 * e] | (uint32_t)q[2 * e + 1] << 16;
    return v;
  };
  // m, n and k are multiples of 16: 8 halves lie inside or outside together.
  // Rows and columns outside are clamped (their outputs are not stored).
  auto load = [&](int s) {
    const int k0 = s * KS;
#pragma unroll
    for (int h = 0; h < L; ++h) {
      const int f = tid + 256 * h;
      const int r = min(row0 + f / (KS / 8), m - 1), kk = k0 + f % (KS / 8) * 8;
      xv[h] = get(a + (int64_t)r * k + min(kk, k - 8));
      const int kb = min(k0 + f / (T / 8), k - 1), c = min(col0 + f % (T / 8) * 8, n - 8);
      yv[h] = get(b + (int64_t)kb * n + c);
    }
  };
  auto store = [&](int s, int buf) {
    const int k0 = s * KS;
#pragma unroll
    for (int h = 0; h < L; ++h) {
      const int f = tid + 256 * h;
      const int r = f / (KS / 8), kk = f % (KS / 8) * 8;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        uint32_t w = k0 + kk < k ? xv[h][e] : Emu<OP>::pad_x;
        if (OP == 7) w = as_bool(w);
        sm.A[buf][kk / 2 + e][r] = w;
      }
      const int kb = f / (T / 8), c = f % (T / 8) * 8;
      const bool in = k0 + kb < k;
      uint32_t w[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        w[e] = in ? yv[h][e] : Emu<OP>::pad_y;
        if (OP == 7) w[e] = as_bool(w[e]);
      }
      if constexpr (GR == 4) {
        *reinterpret_cast<u32x2 *>(&sm.B[buf][kb / 2][c + kb % 2 * 2]) = u32x2{w[0], w[1]};
        *reinterpret_cast<u32x2 *>(&sm.B[buf][kb / 2][c + 4 + kb % 2 * 2]) = u32x2{w[2], w[3]};
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) sm.B[buf][kb / 2][c + 2 * e + kb % 2] = w[e];
      }
    }
  };
  if (s1 > s0) {
    load(s0);
    store(s0, 0);
  }
  __syncthreads();
  for (int s = s0; s < s1; ++s) {
    const int buf = (s - s0) & 1, nx = s + 1 < s1 ? s + 1 : s;
    load(nx);  // the last slab again past the end: written, never read
#pragma unroll
    for (int kp = 0; kp < KS / 2; ++kp) {
      // keeps a k pair's reads next to its arithmetic in the large tiles; the
      // small one has few waves and registers to spare, so its reads may move up
      if (GR == 4 || kp % 8 == 0) __builtin_amdgcn_sched_barrier(0);
      uint32_t av[TM], b0[TM / 2], b1[TM / 2];  // b: k and k + 1
#pragma unroll
      for (int g = 0; g < TM / GR; ++g) {
        *reinterpret_cast<group *>(&av[g * GR]) =
            *reinterpret_cast<const group *>(&sm.A[buf][kp][g * Tile::S + ty * GR]);
        const group v = *reinterpret_cast<const group *>(&sm.B[buf][kp][g * Tile::S + tx * GR]);
#pragma unroll
        for (int e = 0; e < GR / 2; ++e) b0[g * GR / 2 + e] = v[e], b1[g * GR / 2 + e] = v[GR / 2 + e];
      }
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TM / 2; ++j) {
          const uint32_t t0 = emu_term<OP, false>(av[i], b0[j]);
          const uint32_t t1 = emu_term<OP, true>(av[i], b1[j]);
          if constexpr (SUM) {
            acc[i][2 * j] = add_low(add_low(acc[i][2 * j], t0), t1);
            acc[i][2 * j + 1] = add_high(add_high(acc[i][2 * j + 1], t0), t1);
          } else {
            acc[i][j] = emu_fold3<MAX, NANS>(acc[i][j], t0, t1);
          }
        }
    }
    store(nx, buf ^ 1);
    __syncthreads();
  }
}

// One tile per workgroup of 256 G threads; G > 1 (min and max folds only,
// whose terms may be regrouped): each group of 256 takes a range of slabs and
// the partial results are folded at the end.
template <int OP, class Tile, int G, bool VEC>
__global__ __launch_bounds__(256 * G) void tensor_emu_kernel(
    const __half *__restrict__ a, const __half *__restrict__ b, const float *c, float *d, int m,
    int n, int k, int do_epilogue, int tiles_c) {
  constexpr int T = Tile::T, TM = Tile::TM, GR = Tile::GR;
  constexpr bool SUM = Emu<OP>::fold == 2, MAX = Emu<OP>::fold == 1;
  constexpr int W = SUM ? TM : TM / 2;
  static_assert(G == 1 || !SUM, "sums keep their order");
  __shared__ typename Tile::Smem sm[G];
  const int g = tid_x() / 256, tid = tid_x() % 256;
  const int row0 = bid_x() / tiles_c * T, col0 = bid_x() % tiles_c * T;
  // every group runs `per` slabs (and barriers): ranges that would pass the
  // end repeat slabs, which a min or max does not notice
  const int slabs = (k + Tile::KS - 1) / Tile::KS, per = (slabs + G - 1) / G;
  const int s0 = max(0, min(g * per, slabs - per)), s1 = s0 + per;
  using word = typename std::conditional<SUM, float, uint32_t>::type;
  word acc[TM][W];
  auto clear = [&] {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < W; ++j) acc[i][j] = SUM || MAX ? (word)0 : (word)(H_INF * 0x10001u);
  };
  clear();
  emu_loop<OP, Tile, false, VEC>(sm[g], tid, a, b, row0, col0, m, n, k, s0, s1, acc);
  if constexpr (!SUM) {
    bool nan = false;
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < W; ++j)
        nan |= (acc[i][j] & 0x7fffu) > H_INF || (acc[i][j] & 0x7fff0000u) > H_INF << 16;
    if (__syncthreads_or(nan)) {
      clear();
      emu_loop<OP, Tile, true, VEC>(sm[g], tid, a, b, row0, col0, m, n, k, s0, s1, acc);
    }
    if constexpr (G > 1) {
      static_assert(TM * W * 256 * 4 <= sizeof(typename Tile::Smem), "partial tile");
      uint32_t *part = reinterpret_cast<uint32_t *>(&sm[g]);
      if (g > 0) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < W; ++j) part[(i * W + j) * 256 + tid] = acc[i][j];
      }
      __syncthreads();
      if (g > 0) return;
#pragma unroll
      for (int q = 1; q < G; ++q) {
        const uint32_t *other = reinterpret_cast<const uint32_t *>(&sm[q]);
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < W; ++j)
            acc[i][j] = emu_fold2<MAX>(acc[i][j], other[(i * W + j) * 256 + tid]);
      }
    }
  }
  typedef float outs __attribute__((ext_vector_type(GR)));
  const int tx = tid % Tile::NTX, ty = tid / Tile::NTX;
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int r = row0 + i / GR * Tile::S + ty * GR + i % GR;
    if (r >= m) continue;
#pragma unroll
    for (int q = 0; q < TM / GR; ++q) {
      const int cc = col0 + q * Tile::S + tx * GR;
      if (cc >= n) continue;
      outs v;
#pragma unroll
      for (int e = 0; e < GR; ++e) {
        if constexpr (SUM) v[e] = acc[i][q * GR + e];
        else v[e] = half_to_float(acc[i][(q * GR + e) / 2] >> (e % 2 * 16) & 0xffffu);
      }
      const int64_t at = (int64_t)r * n + cc;
      if (VEC) {
        if (do_epilogue) {
          const outs o = *reinterpret_cast<const outs *>(c + at);
#pragma unroll
          for (int e = 0; e < GR; ++e) v[e] = emu_epilogue(OP, v[e], o[e]);
        }
        *reinterpret_cast<outs *>(d + at) = v;
      } else {
#pragma unroll
        for (int e = 0; e < GR; ++e)
          d[at + e] = do_epilogue ? emu_epilogue(OP, v[e], c[at + e]) : v[e];
      }
    }
  }
}

// A 16x16 tile, one output a thread, any alignment: for the fewest outputs,
// where the length of a thread's chain counts and not the instructions, and for
// the shortest K, which the slabs of the tiles above would mostly pad.
constexpr int TE = 16;

template <int OP> __device__ __forceinline__ float emu_step(float acc, __half x, __half y) {
  constexpr int t = Emu<OP>::term, f = Emu<OP>::fold;
  if constexpr (OP == 7)
    return (float)(acc > 0.f || (__half2float(x) > 0.f && __half2float(y) > 0.f));
  __half r;
  if constexpr (t == emu_add) r = __hadd(x, y);
  if constexpr (t == emu_mul) r = __hmul(x, y);
  if constexpr (t == emu_min) r = __hmin(x, y);
  if constexpr (t == emu_max) r = __hmax(x, y);
  if constexpr (t == emu_sub2) {
    r = __hsub(x, y);
    r = __hmul(r, r);
  }
  const float v = __half2float(r);
  return f == 0 ? fminf(acc, v) : f == 1 ? fmaxf(acc, v) : acc + v;
}

template <int OP>
__global__ __launch_bounds__(256) void tensor_emu16_kernel(const __half *__restrict__ a,
                                                           const __half *__restrict__ b,
                                                           const float *c, float *d, int m, int n,
                                                           int k, int do_epilogue) {
  __shared__ __half As[TE][TE + 2];
  __shared__ __half Bs[TE][TE + 2];
  const int tx = tid_x() % TE;   // column within the tile
  const int ty = tid_x() / TE;   // row within the tile
  const int row0 = bid_y() * TE, col0 = bid_x() * TE;
  float acc = Emu<OP>::fold == 0 ? __builtin_inff() : 0.f;
  for (int k0 = 0; k0 < k; k0 += TE) {
    As[ty][tx] = a[(int64_t)(row0 + ty) * k + k0 + tx];
    Bs[ty][tx] = b[(int64_t)(k0 + ty) * n + col0 + tx];
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < TE; ++kk) acc = emu_step<OP>(acc, As[ty][kk], Bs[kk][tx]);
    __syncthreads();
  }
  const int64_t idx = (int64_t)(row0 + ty) * n + col0 + tx;
  d[idx] = do_epilogue ? emu_epilogue(OP, acc, c[idx]) : acc;
}

template <int OP, class Tile, int G, bool VEC>
void launch_emu_tiles(const __half *a, const __half *b, const float *c, float *d, int m, int n,
                      int k, int do_epilogue, hipStream_t s) {
  const int tiles_r = (m + Tile::T - 1) / Tile::T, tiles_c = (n + Tile::T - 1) / Tile::T;
  tensor_emu_kernel<OP, Tile, G, VEC><<<dim3(tiles_r * tiles_c), dim3(256 * G), 0, s>>>(
      a, b, c, d, m, n, k, do_epilogue, tiles_c);
}

// Where a 16x16 tile with one output a thread takes no longer than the tiles (us,
// one output a thread / best tile): few outputs, up to `most` 16x16 tiles per CU;
// more for K below a slab of the 32x32 tiles (64) or just past one, which those
// pad.  min_plus 512^2 of K = 16: 2.8 / 4.6, 64: 4.8 / 4.7, 128: 7.5 / 6.0; plus_mul
// 800^2 of K = 16: 3.7 / 5.8, 80: 8.4 / 8.7, 128: 11.9 / 8.8.  Sums cannot split
// K, so they keep it at any K (minus_square 320^2 of K = 1024 27.6 / 32.0, 16x2048
// 26.8 / 31.9) unless B leaves the L2 (4 MiB: 48x4096 of K = 1024 39.8 / 32.2).
// Where the operands are not 16-byte aligned the 64x64 tiles load element by
// element (minus_square 640^2 of K = 256: 16.7 / 28.4, min_plus 15.7 / 19.6) and
// pay for whole tiles (16x65536 of K = 128: 18.8 / 37.4).
template <int OP> bool one_output_a_thread(bool aligned, int64_t m, int64_t n, int64_t k) {
  constexpr bool SUM = Emu<OP>::fold == 2, SQUARES = Emu<OP>::term == emu_sub2;
  const int64_t cus = device_cu_count(), tiles = m / TE * (n / TE);
  if (m / TE > 65535) return false;  // the grid's second dimension
  const bool thin = std::min(m, n) == TE;  // 32x32 tiles would be half empty
  double most;
  if (!aligned) {
    if (std::min(m, n) < 64) return true;
    most = k <= 16   ? 40
           : k <= 32 ? (SUM ? 36 : 25)
           : k <= 48 ? (SUM ? 30 : 16)
                     : k <= 128 ? (SUM ? 16 : 12) : (SUM ? 12 : 8);
  } else {
    most = k <= 16 ? 36 : k <= 48 ? 10 : k <= 96 ? 4.5 : k <= 128 ? 2.5 : 0;
    if (k > 128 && k <= 176) most = SUM ? 4.2 : 3.5;  // three slabs of 64
    if (SUM && k > 64 && k <= 80) most = 10;
    if (SUM && k > 176 && k * n <= 1 << 21) most = 2;
    if (SQUARES && k > 80) most *= k > 176 ? 1.5 : 2;
    if (SQUARES && thin && tiles >= 4 * cus) return true;
    if (thin) most *= 2;
  }
  return tiles <= most * cus;
}

template <int OP>
void launch_emu_op(const __half *a, const __half *b, const float *c, float *d, int m, int n, int k,
                   int do_epilogue, hipStream_t s) {
  auto aligned = [](const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
  const bool vec = aligned(a) && aligned(b) && aligned(d) && (!do_epilogue || aligned(c));
  const int64_t cus = device_cu_count();
  const int64_t t32 = (int64_t)((m + 31) / 32) * ((n + 31) / 32);
  const int64_t t64 = (int64_t)((m + 63) / 64) * ((n + 63) / 64);
  const int64_t t128 = (int64_t)((m + 127) / 128) * ((n + 127) / 128);
  using Large = EmuTile<128, 8>;
  using Mid = EmuTile<64, 4>;
  using Small = EmuTile<32, 2>;
  if (one_output_a_thread<OP>(vec, m, n, k)) {
    tensor_emu16_kernel<OP><<<dim3(n / TE, m / TE), dim3(256), 0, s>>>(a, b, c, d, m, n, k,
                                                                       do_epilogue);
    return;
  }
  if (!vec) return launch_emu_tiles<OP, Mid, 1, false>(a, b, c, d, m, n, k, do_epilogue, s);
  const bool thin = std::min(m, n) <= 32;  // larger tiles would be half empty
  // 128x128 tiles from two per CU up (min_plus 4096^3 1549 us; one per CU, at
  // 2048^3, loses: 296 us against 228 in 64x64).
  if (t128 >= 2 * cus && std::min(m, n) > 64)
    return launch_emu_tiles<OP, Large, 1, true>(a, b, c, d, m, n, k, do_epilogue, s);
  if constexpr (Emu<OP>::fold == 2) {
    // Sums cannot split K: 32x32 tiles (1296^3 125 us, 150 in 64x64; 640^2 of K =
    // 64 4.9 and 7.9) unless K is short, or fills its last 64-k slab badly and the
    // 64x64 tiles are many (1280^2 of K = 96 15.4 and 14.6).
    if (thin || k >= 128 ||
        (k >= 48 && (k % 64 == 0 || k % 64 >= 48 || t64 < cus)))
      return launch_emu_tiles<OP, Small, 1, true>(a, b, c, d, m, n, k, do_epilogue, s);
  } else {
    // Few tiles: 32x32 ones below 1024^2 / 2 outputs (512^3 9 us, 18 in 64x64;
    // 1040x784x304 24 and 15.5), twice as many for a K that is not worth splitting
    // (800^2 of K = 64 5.6, 9.0 in 64x64), and of thin products (16x8192 of K = 1024 14.8,
    // 32.8 in 64x64), K in four parts when it has four slabs.
    if (t32 <= 2 * cus && k >= 256)
      return launch_emu_tiles<OP, Small, 4, true>(a, b, c, d, m, n, k, do_epilogue, s);
    if (thin || t32 <= (k < 256 ? 4 : 2) * cus)
      return launch_emu_tiles<OP, Small, 1, true>(a, b, c, d, m, n, k, do_epilogue, s);
    if (t64 < 2 * cus && k >= 128)
      return launch_emu_tiles<OP, Mid, 4, true>(a, b, c, d, m, n, k, do_epilogue, s);
  }
  launch_emu_tiles<OP, Mid, 1, true>(a, b, c, d, m, n, k, do_epilogue, s);
}

__global__ void f2h_kernel(const float *in, __half *out, int64_t n) {
  for (int64_t i = (int64_t)bid_x() * blockDim.x + tid_x(); i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    out[i] = __float2half(in[i]);
}

__global__ void h2f_kernel(const __half *in, float *out, int64_t n) {
  for (int64_t i = (int64_t)bid_x() * blockDim.x + tid_x(); i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    out[i] = __half2float(in[i]);
}

}  // namespace

hipError_t launch_tensor_emu(int op, const void *a, const void *b, const float *c, float *d,
                             int m, int n, int k, int do_epilogue, hipStream_t s) {
  // m, n, k are multiples of 16 (checked by the caller).
  const __half *A = static_cast<const __half *>(a);
  const __half *B = static_cast<const __half *>(b);
  switch (op) {
  case 0: launch_emu_op<0>(A, B, c, d, m, n, k, do_epilogue, s); break;
  case 1: launch_emu_op<1>(A, B, c, d, m, n, k, do_epilogue, s); break;
  case 2: launch_emu_op<2>(A, B, c, d, m, n, k, do_epilogue, s); break;
  case 3: launch_emu_op<3>(A, B, c, d, m, n, k, do_epilogue, s); break;
  case 4: launch_emu_op<4>(A, B, c, d, m, n, k, do_epilogue, s); break;
  case 5: launch_emu_op<5>(A, B, c, d, m, n, k, do_epilogue, s); break;
  case 6: launch_emu_op<6>(A, B, c, d, m, n, k, do_epilogue, s); break;
  case 7: launch_emu_op<7>(A, B, c, d, m, n, k, do_epilogue, s); break;
  default: launch_emu_op<8>(A, B, c, d, m, n, k, do_epilogue, s); break;
  }
  return hipGetLastError();
}

hipError_t launch_f2h(void *out, const float *in, int64_t n, hipStream_t s) {
  int64_t blocks = (n + 255) / 256;
  if (blocks > 4096) blocks = 4096;
  if (blocks < 1) blocks = 1;
  f2h_kernel<<<(int)blocks, 256, 0, s>>>(in, static_cast<__half *>(out), n);
  return hipGetLastError();
}

hipError_t launch_h2f(float *out, const void *in, int64_t n, hipStream_t s) {
  int64_t blocks = (n + 255) / 256;
  if (blocks > 4096) blocks = 4096;
  if (blocks < 1) blocks = 1;
  h2f_kernel<<<(int)blocks, 256, 0, s>>>(static_cast<const __half *>(in), out, n);
  return hipGetLastError();
}

}  // namespace simd2
