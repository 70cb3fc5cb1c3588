// plus_mul on the gfx950 matrix cores (the (+,*) semiring is the only float
// one MFMA computes natively).  From K = 256 up each FP32 operand is split into
// three BF16 parts (plusmul_split_kernel); shorter products, and tiles whose values
// do not split exactly, run v_mfma_f32_16x16x4_f32, FP32 in, FP32 accumulate
// (plusmul_tile):
//
// A 256-thread workgroup computes a 128x128 tile; its 4 waves own 64x64
// quadrants, each a 4x4 grid of 16x16 MFMA blocks (64 accumulator registers
// per lane).  K advances in 16-deep slabs staged in LDS (X transposed to
// k-major), double-buffered with one barrier per slab; the slab is consumed
// in 4 MFMA k-steps of 4.  Operand layout of the 16x16x4 f32 instruction:
// lane l supplies A[l%16][l/16] and B[l/16][l%16]; accumulator element v of
// lane l is D[4*(l/16)+v][l%16].  LDS rows are padded by 16 floats so the
// four k-rows a wave reads at once land in distinct banks.
//
// Every shape runs here: VEC loads operands as float4 (leading dimensions
// and bases 16-byte aligned, K and N multiples of 4), otherwise one float at
// a time; rows, columns and k past the matrix are read as zeros and never
// stored (a zero contributes an exact +0 to every sum it enters).
#include "internal.hpp"

namespace simd2 {

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int KB = 16, LDP = 16;

// TILE x TILE output tile (128, or 64 when the 128 tiles would leave CUs
// idle); each wave owns a (TILE/2)^2 quadrant of NB x NB 16x16 blocks.  An
// element's sum runs over the same k slabs in the same order for either
// tile size, so the results are identical.
template <int TILE> struct PlusMulSmem {
  __attribute__((aligned(16))) float Xs[2][KB][TILE + LDP];
  __attribute__((aligned(16))) float Ys[2][KB][TILE + LDP];
};

// The tile body for threads `tid` 0 .. 255 of the workgroup (or of each half
// of it: every thread calls it, for the barriers).
template <int TILE, bool VEC, bool VEC_OUT>
__device__ __forceinline__ void plusmul_tile(PlusMulSmem<TILE> &sm, int tid, int row0, int col0, int R,
                                             int Cn, int K, const float *__restrict__ X,
                                             int64_t ldx, const float *__restrict__ Y, int64_t ldy,
                                             float *O, int64_t ldo, const float *C, int64_t ldc) {
  constexpr int QB = TILE / 2;       // quadrant edge
  constexpr int NB = QB / 16;        // 16x16 blocks per quadrant edge
  constexpr int XPT = TILE / 64;     // float4 loads per thread per slab, X and Y each
  constexpr int YROWS = 1024 / TILE; // k rows of Y one pass of 256 threads covers
  auto &Xs = sm.Xs;
  auto &Ys = sm.Ys;
  const int lane = tid % 64;
  const int wave = tid / 64;
  const int wr = wave / 2, wc = wave % 2;
  f32x4 acc[NB][NB];
#pragma unroll
  for (int i = 0; i < NB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  // Slab loads: X TILE rows x 16 k, Y 16 x TILE, XPT float4 of each per thread.
  const int xr = tid / 4, xk = (tid % 4) * 4;
  const int yk = tid / (TILE / 4), yc = (tid % (TILE / 4)) * 4;
  float4 xv[XPT], yv[XPT];
  // 4 consecutive floats of row r of a matrix from column c; zeros past (rows, cols)
  auto ld4 = [&](const float *M, int64_t ld, int r, int c, int rows, int cols) {
    float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
    if (r < rows) {
      const float *p = M + (int64_t)r * ld + c;
      if (VEC) {
        if (c < cols) v = *reinterpret_cast<const float4 *>(p);
      } else {
        if (c < cols) v.x = p[0];
        if (c + 1 < cols) v.y = p[1];
        if (c + 2 < cols) v.z = p[2];
        if (c + 3 < cols) v.w = p[3];
      }
    }
    return v;
  };
  auto fetch = [&](int k0) {
#pragma unroll
    for (int q = 0; q < XPT; ++q) {
      xv[q] = ld4(X, ldx, row0 + xr + 64 * q, k0 + xk, R, K);
      yv[q] = ld4(Y, ldy, k0 + yk + YROWS * q, col0 + yc, K, Cn);
    }
  };
  auto stage = [&](int b) {
#pragma unroll
    for (int q = 0; q < XPT; ++q) {
      Xs[b][xk + 0][xr + 64 * q] = xv[q].x;
      Xs[b][xk + 1][xr + 64 * q] = xv[q].y;
      Xs[b][xk + 2][xr + 64 * q] = xv[q].z;
      Xs[b][xk + 3][xr + 64 * q] = xv[q].w;
      *reinterpret_cast<float4 *>(&Ys[b][yk + YROWS * q][yc]) = yv[q];
    }
  };
  const int nkt = (K + KB - 1) / KB;
  if (nkt > 0) {
    fetch(0);
    stage(0);
  }
  __syncthreads();
  const int lr = lane % 16, lk = lane / 16;
  for (int kt = 0; kt < nkt; ++kt) {
    const int buf = kt & 1;
    const bool more = kt + 1 < nkt;
    if (more) fetch((kt + 1) * KB);
#pragma unroll
    for (int ks = 0; ks < KB; ks += 4) {
      float a[NB], b[NB];
#pragma unroll
      for (int i = 0; i < NB; ++i) a[i] = Xs[buf][ks + lk][wr * QB + i * 16 + lr];
#pragma unroll
      for (int j = 0; j < NB; ++j) b[j] = Ys[buf][ks + lk][wc * QB + j * 16 + lr];
#pragma unroll
      for (int i = 0; i < NB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], b[j], acc[i][j], 0, 0, 0);
    }
    if (more) stage(buf ^ 1);
    __syncthreads();
  }

  // Stores through LDS, 16 rows of the wave's quadrant at a time: written in
  // the accumulator layout (one column per lane, 4 rows per 16 lanes) to the
  // wave's own padded region and read back row-major, so C is read and O
  // written 16 bytes per lane along rows.  The loop's last barrier has
  // retired every read of Xs; only this wave touches its region.
  constexpr int TLD = QB + 4;
  static_assert(4 * 16 * TLD <= 2 * KB * (TILE + LDP), "store staging fits in Xs");
  float *T = &Xs[0][0][0] + wave * 16 * TLD;
  const int qr0 = row0 + wr * QB, qc0 = col0 + wc * QB;
#pragma unroll
  for (int i = 0; i < NB; ++i) {
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int v = 0; v < 4; ++v) T[(4 * lk + v) * TLD + j * 16 + lr] = acc[i][j][v];
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int h = 0; h < QB / 16; ++h) {
      const int idx = lane + 64 * h;
      const int rr = idx / (QB / 4), cc = (idx % (QB / 4)) * 4;
      const int r = qr0 + i * 16 + rr, c = qc0 + cc;
      f32x4 o = *reinterpret_cast<const f32x4 *>(&T[rr * TLD + cc]);
      if (r >= R) continue;
      if (VEC_OUT && c + 3 < Cn) {
        if (C) o += *reinterpret_cast<const f32x4 *>(C + (int64_t)r * ldc + c);
        *reinterpret_cast<f32x4 *>(O + (int64_t)r * ldo + c) = o;
      } else {
#pragma unroll
        for (int q = 0; q < 4; ++q)
          if (c + q < Cn) O[(int64_t)r * ldo + c + q] = C ? o[q] + C[(int64_t)r * ldc + c + q] : o[q];
      }
    }
    __builtin_amdgcn_wave_barrier();
  }
}

template <int TILE, bool VEC, bool VEC_OUT>
__global__ __launch_bounds__(256) void plusmul_mfma_kernel(
    int R, int Cn, int K, const float *__restrict__ X, int64_t ldx,
    const float *__restrict__ Y, int64_t ldy, float *O, int64_t ldo,
    const float *C, int64_t ldc, int tiles_c) {
  __shared__ PlusMulSmem<TILE> sm;
  plusmul_tile<TILE, VEC, VEC_OUT>(sm, tid_x(), (bid_x() / tiles_c) * TILE, (bid_x() % tiles_c) * TILE, R,
                                   Cn, K, X, ldx, Y, ldy, O, ldo, C, ldc);
}

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int SP_K = 16;  // k per slab: one 32x32x16 BF16 product

// Two floats rounded to BF16, packed (low half first).
__device__ __forceinline__ uint32_t pack_bf16(float a, float b) {
  uint32_t r;
  asm("v_cvt_pk_bf16_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}

// WR x WC waves, each MB x NB blocks of 32x32; a T x T tile, G 16-k steps a
// slab.
template <int MB, int NB, int WR, int WC, int G> struct SplitCfg {
  static constexpr int T = WR * MB * 32, NT = WR * WC * 64;
  static_assert(WC * NB * 32 == T && NT == 2 * T * G, "a thread stages 8 k of a row and a column");
};

// One T x T tile of the product with every FP32 operand split into three BF16
// parts, x = h + m + l exactly (each part is the rest rounded to nearest, 8
// significant bits and a sign each), and the six products of parts down to
// 2^-18 of the term (lh, hl, mm, mh, hm, hh) summed in FP32 by
// v_mfma_f32_32x32x16_bf16.  The three products left out are below 2^-26 of
// the term with random signs, so the result is as near to the exact product
// as the FP32 matrix instruction's, whose roundings (one for each 4 k) it
// has fewer of: relative 2-norm error on normal data 3.4e-8 against 7.4e-8 at
// K = 16, 4.9e-7 against 5.7e-7 at 1024, 1.0e-6 against 1.15e-6 at 4096.
//
// Bounds: six BF16 products a term at 2.4 PFLOP/s measured (400 TFLOP/s of
// FP32 terms) against the FP32 instruction's 157 -- and the card's power:
// 4096^3 takes 493 us on small integers and 629-690 us on normal data
// (1093 us with FP32 instructions).  256x256 tiles halve the conversions (7 VALU
// instructions an element) a product needs; three LDS buffers let the
// fragments of the next slab be read, and the slab after it be written,
// between the products of this one.
//
// Each thread converts 8 k of one X row and of one Y column per slab and
// writes the parts in fragment order.
template <int MB, int NB, int WR, int WC, int G, bool VEC>
__global__ __launch_bounds__(WR * WC * 64, 2) void plusmul_split_kernel(
    int R, int Cn, int K, const float *__restrict__ X, int64_t ldx,
    const float *__restrict__ Y, int64_t ldy, float *O, int64_t ldo,
    const float *C, int64_t ldc, int tiles_r, int tiles_c) {
  constexpr int T = SplitCfg<MB, NB, WR, WC, G>::T;
  constexpr int F = T < 128 ? T : 128;  // tile of the FP32 form
  // [buffer][part][8-k group][row or column]: 8 k, 16 bytes
  struct Parts { u32x4 X[3][3][2 * G][T], Y[3][3][2 * G][T]; };
  __shared__ union {
    Parts sp;
    PlusMulSmem<F> f32[WR * WC / 4];
  } sm;
  const int tid = tid_x();
  const int lane = tid % 64;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int wr = wave / WC, wc = wave % WC;
  // XCD-aware order, tile rows in groups of 8 (neighbours share panels in L2)
  const int nt = tiles_r * tiles_c;
  int t = bid_x();
  if (nt % 8 == 0) t = (t % 8) * (nt / 8) + t / 8;
  const int group = t / (8 * tiles_c), gsz = min(tiles_r - group * 8, 8);
  const int in = t - group * 8 * tiles_c;
  const int row0 = (group * 8 + in % gsz) * T, col0 = (in / gsz) * T;

  const int line = tid % T, g = tid / T;
  const float *xp = X + (int64_t)min(row0 + line, R - 1) * ldx;
  const float *yp = Y + min(col0 + line, Cn - 1);
  // 16-k steps: the partial one, if K has one, comes first, and before it
  // steps of zeros that fill up slab 0, so that the loop has whole steps and
  // no branch.  An element sums the same steps in the same order in every
  // tile size (zeros change nothing), so the tile sizes agree bit for bit.
  const int tail = K % SP_K, nstep = (K + SP_K - 1) / SP_K, nslab = (nstep + G - 1) / G;
  const int lead = nslab * G - nstep;
  auto kof = [&](int s) {  // the thread's first k in slab s
    const int step = s * G + g / 2 - lead;
    return (tail ? (step > 0 ? step - 1 : K / SP_K) : step) * SP_K + g % 2 * 8;
  };
  auto load_first = [&](float (&xv)[8], float (&yv)[8]) {
    const int k = kof(0);
    const bool real = g / 2 >= lead;
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int kk = max(0, min(k + q, K - 1));
      const float a = xp[kk], b = yp[(int64_t)kk * ldy];
      xv[q] = real && k + q < K ? a : 0.f;
      yv[q] = real && k + q < K ? b : 0.f;
    }
  };
  // A slab of whole steps.  Past the last slab it is asked for again and
  // nothing uses it; with a single slab that is slab 0, whose k may lie
  // outside [0, K): clamped (K >= 8).
  auto load = [&](int s, float (&xv)[8], float (&yv)[8]) {
    const int k = max(0, min(kof(s), K - 8));
    if (VEC) {
      *reinterpret_cast<f32x4 *>(&xv[0]) = *reinterpret_cast<const f32x4 *>(xp + k);
      *reinterpret_cast<f32x4 *>(&xv[4]) = *reinterpret_cast<const f32x4 *>(xp + k + 4);
    } else {
#pragma unroll
      for (int q = 0; q < 8; ++q) xv[q] = xp[k + q];
    }
    const float *y = yp + (int64_t)k * ldy;
#pragma unroll
    for (int q = 0; q < 8; ++q) yv[q] = y[q * ldy];
  };
  uint32_t least = ~0u;  // of (bits << 1) - 1: zeros count as large
  auto split = [&](const float (&v)[8], u32x4 (*dst)[2 * G][T]) {
    u32x4 p[3];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      float a = v[2 * q], b = v[2 * q + 1];
      least = min(least, min((__float_as_uint(a) << 1) - 1u, (__float_as_uint(b) << 1) - 1u));
#pragma unroll
      for (int s = 0; s < 3; ++s) {
        const uint32_t h = pack_bf16(a, b);
        p[s][q] = h;
        a -= __uint_as_float(h << 16);
        b -= __uint_as_float(h & 0xffff0000u);
      }
    }
#pragma unroll
    for (int s = 0; s < 3; ++s) dst[s][g][line] = p[s];
  };

  f32x16 acc[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

  // The slabs two and (in the small tiles, which have fewer products to hide
  // a load behind: 1024^3 32 -> 30 us) three ahead of the products wait in
  // registers.
  constexpr bool DEEP = MB <= 2;
  float x0[8], y0[8], x1[8], y1[8];
  load_first(x0, y0);
  load(min(1, nslab - 1), x1, y1);
  split(x0, sm.sp.X[0]);
  split(y0, sm.sp.Y[0]);
  load(min(2, nslab - 1), x0, y0);
  split(x1, sm.sp.X[1]);
  split(y1, sm.sp.Y[1]);
  if (DEEP) load(min(3, nslab - 1), x1, y1);
  __syncthreads();
  u32x4 a[3], b[NB][3];
  auto read_a = [&](int buf, int j, int i) {
#pragma unroll
    for (int p = 0; p < 3; ++p)
      a[p] = sm.sp.X[buf][p][2 * j + lane / 32][(wr * MB + i) * 32 + lane % 32];
  };
  auto read_b = [&](int buf, int j) {
#pragma unroll
    for (int p = 0; p < 3; ++p)
#pragma unroll
      for (int c = 0; c < NB; ++c)
        b[c][p] = sm.sp.Y[buf][p][2 * j + lane / 32][(wc * NB + c) * 32 + lane % 32];
  };
  read_b(0, 0);
  read_a(0, 0, 0);
  int buf = 0;
  auto slab = [&](int s, float (&xv)[8], float (&yv)[8]) {
    const int b1 = buf == 2 ? 0 : buf + 1, b2 = b1 == 2 ? 0 : b1 + 1;
    constexpr int NU = G * MB;  // row blocks of the slab's steps
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      const int j = u / MB, i = u % MB;
      u32x4 ai[3] = {a[0], a[1], a[2]};
      if (u + 1 < NU) read_a(buf, (u + 1) / MB, (u + 1) % MB);
      else read_a(b1, 0, 0);
      if (u == 0) split(xv, sm.sp.X[b2]);
      if (u == (NU > 2 ? 1 : 0)) split(yv, sm.sp.Y[b2]);
      if (u == (NU > 2 ? 2 : 1)) load(min(s + (DEEP ? 4 : 3), nslab - 1), xv, yv);
      // smallest products first
      constexpr int pa[6] = {2, 0, 1, 1, 0, 0}, pb[6] = {0, 2, 1, 0, 1, 0};
#pragma unroll
      for (int q = 0; q < 6; ++q)
#pragma unroll
        for (int c = 0; c < NB; ++c)
          acc[i][c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
              __builtin_bit_cast(bf16x8, ai[pa[q]]), __builtin_bit_cast(bf16x8, b[c][pb[q]]),
              acc[i][c], 0, 0, 0);
      if (u < NU - 1) {  // a few VALU instructions between two products
#pragma unroll
        for (int q = 0; q < 6 * NB; ++q) {
          __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
          __builtin_amdgcn_sched_group_barrier(0x2, 3, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      if (i == MB - 1) {
        if (j + 1 < G) read_b(buf, j + 1);
        else read_b(b1, 0);
      }
    }
    __syncthreads();
    buf = b1;
  };
  for (int s = 0; s < nslab; s += DEEP ? 2 : 1) {
    slab(s, x0, y0);
    if (DEEP && s + 1 < nslab) slab(s + 1, x1, y1);
  }

  // Where the parts do not hold or sum up exactly the tile is computed again
  // in FP32: a value below 2^-100 (its last bits leave BF16's range), an
  // infinity, a NaN or a value that rounds to one (NaN or infinity in the
  // sums), a sum below 2^-80 (the small products leave FP32's range).
  uint32_t most = 0, faint = ~0u;
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) {
          const uint32_t b = __float_as_uint(acc[i][j][v]) << 1;
          most = max(most, b);
          faint = min(faint, b - 1u);
        }
  if (__syncthreads_or(least < (27u << 24) - 1u || most >= 255u << 24 ||
                      faint < (47u << 24) - 1u)) {
    constexpr int GROUPS = WR * WC / 4, ROW = T / F;  // 256 threads an F x F part
    const int own = wave / 4;
#pragma unroll 1
    for (int q = 0; q < ROW * ROW; q += GROUPS) {
      const int part = q + own;
      plusmul_tile<F, VEC, false>(sm.f32[own], tid % 256, row0 + part / ROW * F,
                                  col0 + part % ROW * F, R, Cn, K, X, ldx, Y, ldy, O, ldo, C, ldc);
      __syncthreads();
    }
    return;
  }
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int v = 0; v < 16; ++v) {
      const int r = row0 + (wr * MB + i) * 32 + 8 * (v / 4) + 4 * (lane / 32) + v % 4;
      if (r >= R) continue;
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        const int c = col0 + (wc * NB + j) * 32 + lane % 32;
        if (c < Cn) {
          float o = acc[i][j][v];
          if (C) o += C[(int64_t)r * ldc + c];
          O[(int64_t)r * ldo + c] = o;
        }
      }
    }
}

template <class Cfg, int MB, int NB, int WR, int WC, int G>
void launch_split(bool vec, SplitCfg<MB, NB, WR, WC, G>, int R, int Cn, int K, const float *X,
                  int64_t ldx, const float *Y, int64_t ldy, float *O, int64_t ldo, const float *C,
                  int64_t ldc, hipStream_t s) {
  const int tiles_r = (R + Cfg::T - 1) / Cfg::T, tiles_c = (Cn + Cfg::T - 1) / Cfg::T;
  const dim3 grid(tiles_r * tiles_c), block(Cfg::NT);
  if (vec)
    plusmul_split_kernel<MB, NB, WR, WC, G, true><<<grid, block, 0, s>>>(
        R, Cn, K, X, ldx, Y, ldy, O, ldo, C, ldc, tiles_r, tiles_c);
  else
    plusmul_split_kernel<MB, NB, WR, WC, G, false><<<grid, block, 0, s>>>(
        R, Cn, K, X, ldx, Y, ldy, O, ldo, C, ldc, tiles_r, tiles_c);
}
using SplitL = SplitCfg<4, 2, 2, 4, 1>;  // 256x256, 8 waves
using SplitM = SplitCfg<2, 2, 2, 2, 1>;  // 128x128, 4 waves
using SplitS = SplitCfg<1, 1, 2, 2, 2>;  // 64x64, 4 waves

template <int TILE>
void launch_tile(bool vec, bool vec_out, int R, int Cn, int K, const float *X, int64_t ldx,
                 const float *Y, int64_t ldy, float *O, int64_t ldo, const float *C, int64_t ldc,
                 hipStream_t s) {
  const int tiles_c = (Cn + TILE - 1) / TILE;
  const dim3 grid(((R + TILE - 1) / TILE) * tiles_c), block(256);
  if (vec && vec_out)
    plusmul_mfma_kernel<TILE, true, true><<<grid, block, 0, s>>>(R, Cn, K, X, ldx, Y, ldy, O, ldo,
                                                                 C, ldc, tiles_c);
  else if (vec)
    plusmul_mfma_kernel<TILE, true, false><<<grid, block, 0, s>>>(R, Cn, K, X, ldx, Y, ldy, O,
                                                                  ldo, C, ldc, tiles_c);
  else if (vec_out)
    plusmul_mfma_kernel<TILE, false, true><<<grid, block, 0, s>>>(R, Cn, K, X, ldx, Y, ldy, O,
                                                                  ldo, C, ldc, tiles_c);
  else
    plusmul_mfma_kernel<TILE, false, false><<<grid, block, 0, s>>>(R, Cn, K, X, ldx, Y, ldy, O,
                                                                   ldo, C, ldc, tiles_c);
}

}  // namespace

hipError_t launch_plusmul_mfma(int R, int Cn, int K, const float *X,
                               int64_t ldx, const float *Y, int64_t ldy,
                               float *O, int64_t ldo, const float *C,
                               int64_t ldc, hipStream_t s) {
  auto aligned = [](const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
  const bool vec = K % 4 == 0 && Cn % 4 == 0 && ldx % 4 == 0 && ldy % 4 == 0 && aligned(X) &&
                   aligned(Y);
  // 16-byte stores (and C loads) when every row of O and C is 16-byte aligned
  const bool vec_out = ldo % 4 == 0 && aligned(O) && (!C || (ldc % 4 == 0 && aligned(C)));
  const int64_t cus = device_cu_count();
  const int64_t tiles128 = (int64_t)((R + 127) / 128) * ((Cn + 127) / 128);
  const int64_t tiles256 = (int64_t)((R + 255) / 256) * ((Cn + 255) / 256);
  // The split kernel from K = 256 up, by K alone, so that a product's bits do
  // not depend on its other sizes: 64x64xK, K = 256 / 1024 / 4096, 10.6 / 36 /
  // 138 -> 10.3 / 27 / 99 us, 1024x1024x256 11.9 -> 11.6, 2048x2048x512 51 ->
  // 38; below, its longer start-up costs small products more (K = 128 7.4 ->
  // 9.2 us) than it gains large ones.
  if (K >= 256) {
    // 64x64 tiles while the 128x128 ones are fewer than half the CUs (1024^3
    // 30 us, 59 in 128x128; 1536^3, 144 tiles, 95 and 89).  Then by rounds: one
    // of 256x256 tiles (one per CU) takes 5/3 of one of 128x128 tiles (two per
    // CU): 2900x2900x1024 138 (256) and 152 us (128), 4352x4352x1024 300 and
    // 261, 5120x5120x1024 307 and 350.
    const int64_t large = (tiles256 + cus - 1) / cus, mid = (tiles128 + 2 * cus - 1) / (2 * cus);
    if (tiles128 * 2 < cus)
      launch_split<SplitS>(vec, SplitS{}, R, Cn, K, X, ldx, Y, ldy, O, ldo, C, ldc, s);
    else if (5 * large <= 3 * mid)
      launch_split<SplitL>(vec, SplitL{}, R, Cn, K, X, ldx, Y, ldy, O, ldo, C, ldc, s);
    else
      launch_split<SplitM>(vec, SplitM{}, R, Cn, K, X, ldx, Y, ldy, O, ldo, C, ldc, s);
  } else if (tiles128 < cus) {
    // 64x64 tiles when the 128x128 tiles would not give every CU one
    launch_tile<64>(vec, vec_out, R, Cn, K, X, ldx, Y, ldy, O, ldo, C, ldc, s);
  } else {
    launch_tile<128>(vec, vec_out, R, Cn, K, X, ldx, Y, ldy, O, ldo, C, ldc, s);
  }
  return hipGetLastError();
}

}  // namespace simd2
