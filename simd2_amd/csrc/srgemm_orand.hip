// or_and semiring on gfx950: D = [C |] OR_k A(i,k) & B(k,j).
//
// Packed kernel (simd2_orand_packed): rows of A are K-bit vectors, rows of B
// and D are N-bit vectors, 32 columns per word.  The product is a count of
// common ones that is compared with zero, so it runs on the matrix cores in
// their densest format: each bit becomes an FP4 value (0.5 ... 2, or 0) and
// v_mfma_f32_32x32x64_f8f6f4 sums the products in FP32, every term at least
// 0.25 and none negative, so the sum is zero exactly when no term is 1.
// Bounds: 65536 FP4 operations an instruction, 9.3 PFLOP/s measured with
// operands in registers.  4096^3 at density 0.5 takes 39 us and 8192^3 269 us
// (4.1 P ops/s, 44% of the matrix cores' cycles); the VALU form before it,
// 32 (and, or) terms per v_and_or_b32, took 124 and 830 us.  What is left is
// the conversion of bits to FP4 (80 VALU and 82 scalar instructions per wave
// and 128 k), which two waves per SIMD overlap only in part with 512 cycles
// of products.
//
// When one output tile has a long K and the tiles are few, K is split over
// several workgroups whose partial words are OR-ed into D with atomics (OR is
// idempotent and commutative, so the result is exact): D is first set to C
// (or zero) and the change flag is taken by a pass of its own afterwards.
//
// int32 product (cuasr_orand_srsgemm drop-in): booleans stored one per int.
// The operands are packed into the output's own rows, multiplied there and
// the result unpacked in place (orand_i32_packed), which moves each int once.
// The one-kernel form below serves the shapes whose output rows do not hold
// the packed operands, and the smallest ones: it packs on the fly, X rows (k
// contiguous) along k with wave ballots, Y columns by each lane walking its
// own column, and a thread then ORs the AND of 32-k words per output element
// (v_and_or_b32, 32 terms per instruction).
#include <algorithm>

#include "internal.hpp"

namespace simd2 {

namespace {

// acc | (a & b) as one instruction; written as asm because the compiler
// otherwise pairs terms into v_and + v_or3 (1.5 instructions per term).
__device__ __forceinline__ uint32_t and_or(uint32_t a, uint32_t b, uint32_t acc) {
  uint32_t r;
  asm("v_and_or_b32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(acc));
  return r;
}

// Whether this launch belongs to a squaring behind one that changed nothing.
__device__ __forceinline__ bool flag_done(const FlagStep &f) {
  return f.flag && f.step > 1 && *f.flag < f.step - 1;
}

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4u __attribute__((ext_vector_type(4), aligned(4)));
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef int i32x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

typedef int i32x2 __attribute__((ext_vector_type(2)));

constexpr int OA_KW = 4;  // K-words per slab: 128 k, two 32x32x64 products

// 32 bits as 32 FP4 (E2M1) values: bit b goes to position 8 (b % 4) + b / 4
// (register b % 4, nibble b / 4) as 0.5, 1, 2 or 1.  Any positive values do,
// and any order along k as long as both operands use it.
__device__ __forceinline__ u32x4 bits_to_fp4(uint32_t w) {
  return u32x4{w & 0x11111111u, w & 0x22222222u, w & 0x44444444u, (w >> 2) & 0x22222222u};
}

// 32x32 bit transpose within each half of a wave: lane i's bit j becomes lane
// j's bit i.  Five exchanges with the lane `s` away; each side keeps one half
// of every 2s-bit group and takes the other from the partner, rotated by s.
template <int N> __device__ __forceinline__ void transpose_bits(uint32_t (&x)[N], int lane) {
  constexpr uint32_t low[5] = {0x0000ffffu, 0x00ff00ffu, 0x0f0f0f0fu, 0x33333333u, 0x55555555u};
#pragma unroll
  for (int q = 0; q < 5; ++q) {
    const int s = 16 >> q;
    const uint32_t keep = (lane & s) ? ~low[q] : low[q];
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const uint32_t t = (uint32_t)__shfl_xor((int)x[i], s);
      const uint32_t r = __builtin_amdgcn_alignbit(t, t, (lane & s) ? s : 32 - s);
      x[i] = (x[i] & keep) | (r & ~keep);
    }
  }
}

// Row k of B is at B + (k & bmask) * ldb + (k >> bshift) * bband words: plain
// rows (bmask ~0, bshift 31), or bands of bmask + 1 rows side by side.
struct OrandB {
  const uint32_t *p;
  uint32_t ld, band;
  int mask, shift;
};

// WR x WC waves, each MB x NB blocks of 32x32 outputs; a BM x BM tile.
template <int MB, int NB, int WR, int WC> struct OrandCfg {
  static constexpr int BM = WR * MB * 32, NT = WR * WC * 64;
  static constexpr int WPT = 2 * BM * OA_KW / NT;  // words a thread stages per slab
  static_assert(WC * NB * 32 == BM && (WPT == 2 || WPT == 4) && MB % 2 == 0, "tile");
};

// One BM x BM tile of bits.  Half of the threads stage A, one row and WPT
// K-words each; the other half B, one k and WPT words of columns each.  Both
// write FP4 values: A as [32-k group][row][32 k], B as [k][column], each k at
// its FP4 position, from where the transposing LDS read gives a lane the 16 k
// of one column.  A word's columns are then in position order too; the
// epilogue undoes that.
template <int MB, int NB, int WR, int WC, bool VEC>
__global__ __launch_bounds__(WR * WC * 64) void orand_packed_kernel(
    int M, int NW, int K, const uint32_t *__restrict__ A, uint32_t lda, OrandB B, const uint32_t *C,
    int64_t ldc, uint32_t *D, int64_t ldd, const uint32_t *P, int64_t ldp, FlagStep flag,
    uint32_t last_mask, int tiles_c, int ksplit, int kw_per) {
  using Cfg = OrandCfg<MB, NB, WR, WC>;
  constexpr int BM = Cfg::BM, NT = Cfg::NT, WPT = Cfg::WPT;
  // row pitch of B: 16-byte granules, 8-byte reads of 16 rows in distinct banks
  constexpr int BLD = BM / 2 + 16;
  typedef uint32_t uwords __attribute__((ext_vector_type(WPT)));
  __shared__ u32x4 As[2][OA_KW][BM];
  __shared__ __attribute__((aligned(16))) unsigned char Bs[2][OA_KW * 32][BLD];
  // bit 2 rb + h: A rows 32 rb.. hold a 1 in 64-k half h; bit 16 + 2 cb + h:
  // the same for B columns 32 cb..
  __shared__ uint32_t some[3];
  __shared__ uint64_t occ[NT / 64];
  if (flag_done(flag)) return;
  const int tid = tid_x();
  const int lane = tid % 64;
  const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int wr = wave / WC, wc = wave % WC;
  const int ntiles = (M + BM - 1) / BM * tiles_c;
  int tile = bid_x() / ksplit;
  const int split = bid_x() % ksplit;
  // consecutive tiles (which share A rows) on one XCD
  if (ksplit == 1 && ntiles % 8 == 0) tile = (tile % 8) * (ntiles / 8) + tile / 8;
  const int row0 = (tile / tiles_c) * BM;
  const int w0 = (tile % tiles_c) * (BM / 32);
  const int nkw = (K + 31) / 32;
  const int kw0 = split * kw_per;
  const int kw_end = min(nkw, kw0 + kw_per);
  const bool stage_a = wave < NT / 128;
  const int t = stage_a ? tid : tid - NT / 2;
  // A: tile row and first K-word; B: k and first word of columns
  const int line = stage_a ? t % BM : t % (OA_KW * 32);
  // the k whose position in its group of 32 (bits_to_fp4's order) is `line`
  const int kline = (line & ~31) + 4 * (line % 8) + (line % 32) / 8;
  const int word = __builtin_amdgcn_readfirstlane(stage_a ? t / BM : t / (OA_KW * 32)) * WPT;

  // The thread's words of the slab starting at word kw.  Addresses past the
  // matrix are clamped into it instead of masked, so that no branch merges a
  // loaded value (a merge waits for it): rows past M and words past NW only
  // feed outputs that are not stored, and k past K meets A bits cleared in
  // stage().  Every path issues the same number of loads, so waits can count
  // them.
  auto load = [&](int kw) {
    const int k = min(kw * 32 + kline, K - 1);
    const uint32_t row = stage_a ? min(row0 + line, M - 1) : k & B.mask;
    const uint32_t ld = stage_a ? lda : B.ld;
    const uint32_t *p = (stage_a ? A : B.p) + (uint64_t)row * ld;
    const int col = stage_a ? kw + word : w0 + word, last = stage_a ? nkw - 1 : NW - 1;
    if (!stage_a) p += (uint32_t)(k >> B.shift) * B.band;
    uwords v;
    if (VEC) {
      v = *reinterpret_cast<const uwords *>(p + min(col, last / OA_KW * OA_KW + OA_KW - WPT));
    } else {
#pragma unroll
      for (int q = 0; q < WPT; ++q) v[q] = p[min(col + q, last)];
    }
    return v;
  };
  const uint32_t ktail = (K & 31) ? (1u << (K & 31)) - 1u : ~0u;
  auto stage = [&](uwords v, int kw, int buf, int slot) {
    uint32_t bits = 0;
    if (stage_a) {
#pragma unroll
      for (int q = 0; q < WPT; ++q) {
        const int w = kw + word + q;
        v[q] &= w >= kw_end ? 0u : w == nkw - 1 ? ktail : ~0u;
        As[buf][word + q][line] = bits_to_fp4(v[q]);
      }
#pragma unroll
      for (int q = 0; q < WPT; q += 2) {
        const uint64_t b = __ballot((v[q] | v[q + 1]) != 0u);
        const int at = (wave * 2 % (BM / 32)) * 2 + (word + q) / 2;
        bits |= ((uint32_t)((uint32_t)b != 0u) | (uint32_t)((b >> 32) != 0u) << 2) << at;
      }
    } else {
#pragma unroll
      for (int q = 0; q < WPT; ++q) {
        *reinterpret_cast<u32x4 *>(&Bs[buf][line][(word + q) * 16]) = bits_to_fp4(v[q]);
        bits |= (uint32_t)(__ballot(v[q] != 0u) != 0) << (16 + (word + q) * 2 + wave % 2);
      }
    }
    if (lane == 0 && bits) atomicOr(&some[slot], bits);
  };

  // Starting below zero by less than any product (>= 0.25) makes the sign the
  // answer: set while no term of the element is 1.
  f32x16 acc[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = -0.125f;

  const int nslab = max(0, kw_end - kw0 + OA_KW - 1) / OA_KW;
  typedef __attribute__((address_space(3))) i32x2 *lds2;
  u32x4 a[2][MB];
  i32x2 b[2][NB][2];
  auto fragments = [&](int buf, int h) {
    const int g = h * 2 + lane / 32;
#pragma unroll
    for (int i = 0; i < MB; ++i) a[h][i] = As[buf][g][(wr * MB + i) * 32 + lane % 32];
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int q = 0; q < 2; ++q)
        b[h][j][q] = __builtin_amdgcn_ds_read_tr4_b64_v2i32(
            (lds2)&Bs[buf][g * 32 + q * 16 + lane % 16]
                     [(wc * NB + j) * 16 + (lane / 16 % 2) * 8]);
  };
  auto multiply = [&](uint32_t on, int h) {
    // any of the wave's A rows, and any of its columns, in half h
    constexpr uint32_t arow = MB == 4 ? 0x55u : 0x5u, bcol = 0x5u;
    if (!(on & (arow << (wr * MB * 2 + h))) || !(on & (bcol << (16 + wc * NB * 2 + h)))) return;
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(
            __builtin_shufflevector(i32x4(a[h][i]), i32x4(a[h][i]), 0, 1, 2, 3, -1, -1, -1, -1),
            __builtin_shufflevector(b[h][j][0], b[h][j][1], 0, 1, 2, 3, -1, -1, -1, -1), acc[i][j],
            4, 4, 0, 0, 0, 0);
  };
  // Slabs are taken one after the other until the tile's A rows hold no 1 in two
  // of them (or in the first two).  What is left is looked over SCAN slabs at a
  // time, a wave reading whole rows with a slab per lane, and only those with a 1
  // in A are taken: a slab that is merely loaded and converted costs 0.7 us of the
  // 1.0 us of one that is multiplied.  8192^3, every slab taken and here: no bit at
  // all 187 -> 44 us, blocks of 64 on the diagonal 187 -> 54, density 1e-5 188 ->
  // 103, 1e-4 204 -> 210, 0.5 266 -> 269 (4096^3 38.3 -> 38.5).  A loop of its own
  // for the second part would leave the first as it was, but needs a second set
  // of accumulator registers.
  constexpr int SCAN = 60;  // leaves lanes for the slabs asked for past the last
  int count = nslab;        // slabs to take, the s-th (s < 64 but for all) ...
  int order = kw0 + lane * OA_KW;  // ... from word order[s % 64] + (s - s % 64) * OA_KW
  int rest = nslab;                // the first slab not looked at
  for (bool all = true; count > 0; all = false) {
    // At slab s: its fragments are in registers, the fragments of s + 1 are
    // read from LDS between the products, the words of s + 2 are converted
    // into LDS and those of s + 4 are on their way from memory.  The waves
    // that stage A do so before their products, the others after, so that one
    // half converts while the other keeps the matrix cores busy.  `some` is
    // read one slab ahead too and cleared one slab before it is collected.
    // Words past the last slab are kw_end or more: read from inside the matrix
    // (load), A's taken as zero (stage).
    auto word_of = [&](int s) {
      return __builtin_amdgcn_readlane(order, s & 63) + (s & ~63) * OA_KW;
    };
    if (tid < 3) some[tid] = 0;
    int kwa = word_of(0), kwb = word_of(1);
    uwords pre0 = load(kwa), pre1 = load(kwb);
    __syncthreads();
    stage(pre0, kwa, 0, 0);
    stage(pre1, kwb, 1, 1);
    kwa = word_of(2), kwb = word_of(3);
    pre0 = load(kwa);
    pre1 = load(kwb);
    __syncthreads();
    fragments(0, 0);
    fragments(0, 1);
    uint32_t on = some[0], now = 0;
    constexpr uint32_t a_bits = 0xffffu;
    const bool none = !(__builtin_amdgcn_readfirstlane(on | some[1]) & a_bits);
    __syncthreads();
    int slot = 0;  // s % 3
    auto step = [&](int s, uwords &pre, int &kw) {
      const int buf = s & 1, s1 = slot == 2 ? 0 : slot + 1, s2 = s1 == 2 ? 0 : s1 + 1;
      now = __builtin_amdgcn_readfirstlane(on);
      on = some[s1];
      if (tid == 0) some[slot] = 0;
      if (stage_a) stage(pre, kw, buf, s2);
      multiply(now, 0);
      __builtin_amdgcn_sched_barrier(0);
      fragments(buf ^ 1, 0);
      __builtin_amdgcn_sched_barrier(0);
      multiply(now, 1);
      __builtin_amdgcn_sched_barrier(0);
      fragments(buf ^ 1, 1);
      if (!stage_a) stage(pre, kw, buf, s2);
      kw = word_of(s + 4);
      pre = load(kw);
      slot = s1;
      __syncthreads();
    };
    int s = all && none ? 2 : 0, end = s ? 0 : count;
    const uint32_t hold = all ? 0u : 1u;  // listed slabs hold a 1 (or padding that may)
    while (s < end) {
      step(s, pre0, kwa);
      uint32_t was = now | hold;
      if (s + 1 < count) step(s + 1, pre1, kwb);
      s += 2;
      was |= now;
      end = was & a_bits ? end : 0;
    }
    if (end == 0) rest = s;
    for (count = 0; count == 0 && rest < nslab; rest += SCAN) {
      constexpr int ROWS = BM * 64 / NT, BATCH = 8;
      const int w = min(kw0 + (rest + lane) * OA_KW, nkw - OA_KW);  // nkw >= 4: nslab > 2
      uint32_t any = 0;
#pragma unroll 1
      for (int i = 0; i < ROWS; i += BATCH) {
        u32x4u v[BATCH];
#pragma unroll
        for (int q = 0; q < BATCH; ++q)
          v[q] = *reinterpret_cast<const u32x4u *>(
              A + (uint64_t)(uint32_t)min(row0 + wave * ROWS + i + q, M - 1) * lda + w);
#pragma unroll
        for (int q = 0; q < BATCH; ++q) any |= v[q][0] | v[q][1] | v[q][2] | v[q][3];
      }
      const uint64_t mine = __ballot(any != 0u && lane < SCAN && rest + lane < nslab);
      if (lane == 0) occ[wave] = mine;
      __syncthreads();
      uint64_t full = 0;
#pragma unroll
      for (int q = 0; q < NT / 64; ++q) full |= occ[q];
      __syncthreads();
      // the slabs taken go to the first lanes in order, the others' lanes get kw_end
      const int rank = __popcll(full & ((1ull << lane) - 1));
      const bool taken = full >> lane & 1;
      count = __builtin_amdgcn_readfirstlane(__popcll(full));
      order = __builtin_amdgcn_ds_permute((taken ? rank : count + lane - rank) * 4,
                                          taken ? kw0 + (rest + lane) * OA_KW : kw_end);
    }
  }

  // Lane = column position, element v of block i = row i * 32 + 8 (v / 4) +
  // 4 (lane / 32) + v % 4.  The signs of two row blocks make 32 bits per
  // lane; with the lanes put in column order their transpose is one packed
  // output word per lane.
  const int from = (lane & 32) + 8 * (lane % 4) + (lane % 32) / 4;
  bool changed = false;
#pragma unroll
  for (int i = 0; i < MB; i += 2) {
    uint32_t out[NB];
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      uint32_t m = 0;
#pragma unroll
      for (int v = 31; v >= 0; --v)
        m = __builtin_amdgcn_alignbit(m, __float_as_uint(acc[i + v / 16][j][v % 16]), 31);
      out[j] = ~(uint32_t)__builtin_amdgcn_ds_bpermute(from * 4, (int)m);
    }
    transpose_bits(out, lane);
    const int v = lane % 32, vv = v % 16;
    const int r = row0 + (wr * MB + i + v / 16) * 32 + 8 * (vv / 4) + 4 * (lane / 32) + vv % 4;
    if (r < M) {
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        const int w = w0 + wc * NB + j;
        if (w >= NW) continue;
        const uint32_t mask = w == NW - 1 ? last_mask : ~0u;
        uint32_t o = out[j];
        if (ksplit > 1) {  // partial words into D (set to C or zero beforehand)
          o &= mask;
          if (o) atomicOr(&D[(int64_t)r * ldd + w], o);
        } else {
          if (C) o |= C[(int64_t)r * ldc + w];
          o &= mask;
          if (P) changed |= o != (P[(int64_t)r * ldp + w] & mask);
          D[(int64_t)r * ldd + w] = o;
        }
      }
    }
  }
  // one atomic per tile at most: the memory takes those to one address at 3 ns each
  if (flag.flag && ksplit == 1)
    if (__syncthreads_or(changed) && tid == 0) atomicMax(flag.flag, flag.step);
}

using OrandL = OrandCfg<4, 2, 2, 4>;  // 256x256, 8 waves
using OrandS = OrandCfg<2, 2, 2, 2>;  // 128x128, 4 waves

// D = C (or zero), last word masked: the start of a K-split product.
__global__ __launch_bounds__(256) void orand_init_kernel(int M, int NW, const uint32_t *C,
                                                         int64_t ldc, uint32_t *D, int64_t ldd,
                                                         uint32_t last_mask, FlagStep flag) {
  if (flag_done(flag)) return;
  const int64_t total = (int64_t)M * NW;
  for (int64_t e = (int64_t)bid_x() * 256 + tid_x(); e < total; e += (int64_t)gridDim.x * 256) {
    const int r = (int)(e / NW), w = (int)(e % NW);
    const uint32_t v = C ? C[(int64_t)r * ldc + w] : 0u;
    D[(int64_t)r * ldd + w] = v & (w == NW - 1 ? last_mask : ~0u);
  }
}

// *flag = 1 when D differs from P (last word masked): the change test of a
// K-split product.  One atomic per workgroup at most (a workgroup-wide OR
// first): when most words changed, one per wave serialised on the flag.
__global__ __launch_bounds__(256) void orand_diff_kernel(int M, int NW, const uint32_t *D,
                                                         int64_t ldd, const uint32_t *P,
                                                         int64_t ldp, uint32_t last_mask,
                                                         FlagStep flag) {
  if (flag_done(flag)) return;
  const int64_t total = (int64_t)M * NW;
  bool changed = false;
  for (int64_t e = (int64_t)bid_x() * 256 + tid_x(); e < total; e += (int64_t)gridDim.x * 256) {
    const int r = (int)(e / NW), w = (int)(e % NW);
    const uint32_t m = w == NW - 1 ? last_mask : ~0u;
    changed |= (D[(int64_t)r * ldd + w] & m) != (P[(int64_t)r * ldp + w] & m);
  }
  if (__syncthreads_or(changed) && tid_x() == 0) atomicMax(flag.flag, flag.step);
}

// ---- int32 booleans -------------------------------------------------------
constexpr int IB_BM = 64;   // output rows per tile
constexpr int IB_BN = 64;   // output columns per tile
constexpr int IB_BKW = 8;   // 32-bit k-words per slab (256 k)

__global__ __launch_bounds__(256) void orand_i32_kernel(
    int R, int Cn, int K, const int *__restrict__ X, int64_t ldx,
    const int *__restrict__ Y, int64_t ldy, const int *C, int64_t ldc,
    int *O, int64_t ldo, const int *P, int64_t ldp, int *flag, int tiles_c) {
  __shared__ uint32_t Xp[IB_BM][IB_BKW + 1];   // rows packed along k
  __shared__ uint32_t Yp[IB_BN][IB_BKW + 1];   // columns packed along k
  const int tid = tid_x();
  const int lane = tid % 64;
  const int wave = tid / 64;
  const int row0 = (bid_x() / tiles_c) * IB_BM;
  const int col0 = (bid_x() % tiles_c) * IB_BN;
  const int tr = tid / 16;  // 16 x 16 threads, 4 x 4 outputs each
  const int tc = tid % 16;

  uint32_t acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = 0u;

  for (int k0 = 0; k0 < K; k0 += IB_BKW * 32) {
    // Loads are issued in batches before any is used (addresses clamped into
    // the matrix, values outside it taken as false), so a batch waits for
    // memory once.
    // X: each wave packs 16 rows, 4 at a time; per row, 4 ballots of 64
    // consecutive k.
    for (int rr = 0; rr < IB_BM / 4; rr += 4) {
      int v[4][IB_BKW / 2];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int r = min(row0 + wave * (IB_BM / 4) + rr + i, R - 1);
#pragma unroll
        for (int ch = 0; ch < IB_BKW / 2; ++ch)
          v[i][ch] = X[(int64_t)r * ldx + min(k0 + ch * 64 + lane, K - 1)];
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int lr = wave * (IB_BM / 4) + rr + i;
#pragma unroll
        for (int ch = 0; ch < IB_BKW / 2; ++ch) {
          const int k = k0 + ch * 64 + lane;
          const uint64_t m = __ballot(row0 + lr < R && k < K && v[i][ch] != 0);
          if (lane == 0) {
            Xp[lr][ch * 2] = (uint32_t)m;
            Xp[lr][ch * 2 + 1] = (uint32_t)(m >> 32);
          }
        }
      }
    }
    // Y: lane = column, each wave walks 64 k (two words) of its quarter.
    {
      const int c = col0 + lane, cc = min(c, Cn - 1);
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        const int kb = k0 + wave * 64 + half * 32;
        int v[32];
#pragma unroll
        for (int q = 0; q < 32; ++q) v[q] = Y[(int64_t)min(kb + q, K - 1) * ldy + cc];
        uint32_t wv = 0;
#pragma unroll
        for (int q = 0; q < 32; ++q)
          wv |= (uint32_t)(c < Cn && kb + q < K && v[q] != 0) << q;
        Yp[lane][wave * 2 + half] = wv;
      }
    }
    __syncthreads();
#pragma unroll
    for (int w = 0; w < IB_BKW; ++w) {
      uint32_t xa[4], yb[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) xa[i] = Xp[tr * 4 + i][w];
#pragma unroll
      for (int j = 0; j < 4; ++j) yb[j] = Yp[tc * 4 + j][w];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = and_or(xa[i], yb[j], acc[i][j]);
    }
    __syncthreads();
  }

  bool changed = false;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = row0 + tr * 4 + i;
    if (r >= R) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int c = col0 + tc * 4 + j;
      if (c >= Cn) continue;
      int v = acc[i][j] != 0u;
      if (C) v = v || (C[(int64_t)r * ldc + c] != 0);
      if (P) changed |= (v != P[(int64_t)r * ldp + c]);
      O[(int64_t)r * ldo + c] = v;
    }
  }
  if (flag && __syncthreads_or(changed) && tid == 0) atomicOr(flag, 1);
}

}  // namespace

namespace {

template <class Cfg, bool VEC, int MB, int NB, int WR, int WC>
void launch_orand_tiles(OrandCfg<MB, NB, WR, WC>, int M, int NW, int K, const uint32_t *A,
                        int64_t lda, const OrandB &B, const uint32_t *C, int64_t ldc, uint32_t *D,
                        int64_t ldd, const uint32_t *P, int64_t ldp, FlagStep flag,
                        uint32_t last_mask, int ksplit, int kw_per, hipStream_t s) {
  const int tiles_r = (M + Cfg::BM - 1) / Cfg::BM;
  const int tiles_c = (NW + Cfg::BM / 32 - 1) / (Cfg::BM / 32);
  orand_packed_kernel<MB, NB, WR, WC, VEC><<<dim3(tiles_r * tiles_c * ksplit), dim3(Cfg::NT), 0,
                                             s>>>(M, NW, K, A, lda, B, C, ldc, D, ldd, P, ldp,
                                                  flag, last_mask, tiles_c, ksplit, kw_per);
}

// padded: the rows of A and B hold whole groups of four words (whatever is in
// the words past K and N).
hipError_t launch_orand_rows(int M, int N, int K, const uint32_t *A, int64_t lda, const OrandB &B,
                             bool padded, const uint32_t *C, int64_t ldc, uint32_t *D, int64_t ldd,
                             const uint32_t *P, int64_t ldp, FlagStep flag, hipStream_t s) {
  const int NW = (N + 31) / 32;
  if (M <= 0 || NW <= 0) return hipSuccess;
  const uint32_t last_mask = (N & 31) ? ((1u << (N & 31)) - 1u) : ~0u;
  const int cus = device_cu_count();
  auto tiles = [&](int bm, int bw) { return (int64_t)((M + bm - 1) / bm) * ((NW + bw - 1) / bw); };
  // 256x256 tiles once they give every CU one: twice the products per
  // converted word (8192^3 287 against 382 us, 4096^3 42 against 58 us); below
  // that their idle CUs cost more (2048^3 27 against 15 us).  K is split when
  // the 128x128 tiles leave CUs idle, in parts of at least 16 slabs: below
  // that the two more launches cost what the split gains (about 0.4 us a slab).
  const bool large = tiles(256, 8) >= cus;
  const int nslab = ((K + 31) / 32 + OA_KW - 1) / OA_KW;
  int ksplit = 1;
  if (!large)
    ksplit = (int)std::max<int64_t>(1, std::min<int64_t>(2 * cus / tiles(128, 4), nslab / 16));
  const int kw_per = std::max(1, (nslab + ksplit - 1) / ksplit) * OA_KW;
  if (nslab > 0) ksplit = (nslab * OA_KW + kw_per - 1) / kw_per;
  const int64_t words = (int64_t)M * NW;
  const int egrid = (int)std::min<int64_t>((words + 255) / 256, 2048);
  if (ksplit > 1)
    orand_init_kernel<<<dim3(egrid), dim3(256), 0, s>>>(M, NW, C, ldc, D, ldd, last_mask, flag);
  auto aligned = [](const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
  // 16-byte loads read whole groups of four words: rows must hold them
  const bool vec = aligned(A) && aligned(B.p) && lda % 4 == 0 && B.ld % 4 == 0 &&
                   B.band % 4 == 0 && (padded || (NW % 4 == 0 && (K + 31) / 32 % 4 == 0));
  if (large && vec)
    launch_orand_tiles<OrandL, true>(OrandL{}, M, NW, K, A, lda, B, C, ldc, D, ldd, P, ldp, flag,
                                     last_mask, ksplit, kw_per, s);
  else if (large)
    launch_orand_tiles<OrandL, false>(OrandL{}, M, NW, K, A, lda, B, C, ldc, D, ldd, P, ldp, flag,
                                      last_mask, ksplit, kw_per, s);
  else if (vec)
    launch_orand_tiles<OrandS, true>(OrandS{}, M, NW, K, A, lda, B, C, ldc, D, ldd, P, ldp, flag,
                                     last_mask, ksplit, kw_per, s);
  else
    launch_orand_tiles<OrandS, false>(OrandS{}, M, NW, K, A, lda, B, C, ldc, D, ldd, P, ldp, flag,
                                      last_mask, ksplit, kw_per, s);
  if (ksplit > 1 && P && flag.flag)
    orand_diff_kernel<<<dim3(egrid), dim3(256), 0, s>>>(M, NW, D, ldd, P, ldp, last_mask, flag);
  return hipGetLastError();
}

// int32 booleans (nonzero = 1) <-> packed rows (bit c % 32 of word c / 32),
// one wave per row.  Both may work in place, the words at the start of the
// row's own ints: packing walks the row forwards (the words of the columns
// before c lie below int c), unpacking backwards (the words of the columns
// before c lie below int c too, and int c on is all that is written).  The
// row pointers are not __restrict__ and every chunk's loads precede its
// stores, which is what in-place use relies on.
// VEC: rows 16-byte aligned, a lane moves 4 neighbouring columns at a time.
struct PackJob {
  const int *src = nullptr;
  uint32_t *dst = nullptr;
  int64_t lds = 0, ldd = 0, band = 0;  // row r of dst: (r & mask) * ldd + (r >> shift) * band
  int rows = 0, cols = 0, mask = -1, shift = 31;
  int *nonbool = nullptr;              // set if src holds a value other than 0 / 1
};

template <int CTRL> __device__ __forceinline__ uint32_t or_dpp(uint32_t x) {
  return x | (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, CTRL, 0xf, 0xf, true);
}

template <bool VEC>
__global__ __launch_bounds__(256) void pack_rows_kernel(PackJob j0, PackJob j1, PackJob j2) {
  const int lane = tid_x() % 64;
  int64_t g = (int64_t)bid_x() * 4 + __builtin_amdgcn_readfirstlane(tid_x() / 64);
  PackJob j = j0;
  if (g >= j.rows) {
    g -= j.rows;
    j = j1;
    if (g >= j.rows) {
      g -= j.rows;
      j = j2;
      if (g >= j.rows) return;
    }
  }
  const int r = (int)g;
  const int *x = j.src + (int64_t)r * j.lds;
  uint32_t *w = j.dst + (int64_t)(r & j.mask) * j.ldd + (int64_t)(r >> j.shift) * j.band;
  const int nw = (j.cols + 31) / 32;
  bool odd = false;
  if (VEC) {
    for (int c0 = 0; c0 < j.cols; c0 += 1024) {
      i32x4 v[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int c = c0 + q * 256 + lane * 4;
        v[q] = i32x4{0, 0, 0, 0};
        if (c + 3 < j.cols) {
          v[q] = *reinterpret_cast<const i32x4 *>(x + c);
        } else {
#pragma unroll
          for (int e = 0; e < 3; ++e)
            if (c + e < j.cols) v[q][e] = x[c + e];
        }
      }
      uint32_t mine = 0;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        uint32_t nib = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          odd |= (unsigned)v[q][e] > 1u;
          nib |= (uint32_t)(v[q][e] != 0) << e;
        }
        // the eight lanes of a word: neighbours, pairs, halves of eight
        uint32_t u = nib << (4 * (lane % 8));
        u = or_dpp<0xB1>(u);
        u = or_dpp<0x4E>(u);
        u = or_dpp<0x141>(u);
        if (lane % 8 == q) mine = u;
      }
      const int word = c0 / 32 + (lane % 8) * 8 + lane / 8;
      if (lane % 8 < 4 && word < nw) w[word] = mine;
    }
  } else {
    for (int c0 = 0; c0 < j.cols; c0 += 256) {
      int v[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int c = c0 + q * 64 + lane;
        v[q] = c < j.cols ? x[c] : 0;
      }
      uint64_t b[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        odd |= (unsigned)v[q] > 1u;
        b[q] = __ballot(v[q] != 0);
      }
      const int word = c0 / 32 + lane;
      if (lane < 8 && word < nw) {
        const uint64_t bq = (lane >> 1) == 0 ? b[0] : (lane >> 1) == 1 ? b[1] : (lane >> 1) == 2 ? b[2] : b[3];
        w[word] = (lane & 1) ? (uint32_t)(bq >> 32) : (uint32_t)bq;
      }
    }
  }
  if (j.nonbool && __any(odd) && lane == 0) atomicOr(j.nonbool, 1);
}

template <bool VEC>
__global__ __launch_bounds__(256) void unpack_rows_kernel(int rows, int cols, const uint32_t *P,
                                                          int64_t ldp, int *X, int64_t ldx) {
  const int lane = tid_x() % 64;
  const int64_t r = (int64_t)bid_x() * 4 + __builtin_amdgcn_readfirstlane(tid_x() / 64);
  if (r >= rows) return;
  const uint32_t *p = P + r * ldp;
  int *x = X + r * ldx;
  constexpr int CH = VEC ? 1024 : 256;
  for (int c0 = (cols - 1) / CH * CH; c0 >= 0; c0 -= CH) {
    uint32_t u[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int c = VEC ? c0 + q * 256 + lane * 4 : c0 + q * 64 + lane;
      u[q] = c < cols ? p[c / 32] >> (c % 32) : 0u;
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if (VEC) {
        const int c = c0 + q * 256 + lane * 4;
        const i32x4 o = {(int)(u[q] & 1u), (int)(u[q] >> 1 & 1u), (int)(u[q] >> 2 & 1u),
                         (int)(u[q] >> 3 & 1u)};
        if (c + 3 < cols) {
          *reinterpret_cast<i32x4 *>(x + c) = o;
        } else {
#pragma unroll
          for (int e = 0; e < 3; ++e)
            if (c + e < cols) x[c + e] = o[e];
        }
      } else {
        const int c = c0 + q * 64 + lane;
        if (c < cols) x[c] = (int)(u[q] & 1u);
      }
    }
  }
}

bool int_rows_vec(const void *p, int64_t ld) {
  return (reinterpret_cast<uintptr_t>(p) & 15) == 0 && ld % 4 == 0;
}

hipError_t launch_pack_rows(const PackJob &j0, const PackJob &j1, const PackJob &j2,
                            hipStream_t s) {
  const int64_t rows = (int64_t)j0.rows + j1.rows + j2.rows;
  if (rows <= 0) return hipSuccess;
  bool vec = true;
  for (const PackJob *j : {&j0, &j1, &j2})
    if (j->rows > 0) vec = vec && int_rows_vec(j->src, j->lds);
  const dim3 grid((unsigned)((rows + 3) / 4));
  if (vec)
    pack_rows_kernel<true><<<grid, dim3(256), 0, s>>>(j0, j1, j2);
  else
    pack_rows_kernel<false><<<grid, dim3(256), 0, s>>>(j0, j1, j2);
  return hipGetLastError();
}

PackJob pack_job(int rows, int cols, const int *src, int64_t lds, uint32_t *dst, int64_t ldd) {
  PackJob j;
  j.src = src;
  j.lds = lds;
  j.dst = dst;
  j.ldd = ldd;
  j.rows = rows;
  j.cols = cols;
  return j;
}

}  // namespace

hipError_t launch_orand_packed(int M, int N, int K, const uint32_t *A,
                               int64_t lda, const uint32_t *B, int64_t ldb,
                               const uint32_t *C, int64_t ldc, uint32_t *D,
                               int64_t ldd, const uint32_t *P, int64_t ldp,
                               FlagStep flag, hipStream_t s) {
  return launch_orand_rows(M, N, K, A, lda, OrandB{B, (uint32_t)ldb, 0, -1, 31}, false, C, ldc, D, ldd, P, ldp,
                           flag, s);
}

hipError_t launch_pack_i32(int rows, int cols, const int *X, int64_t ldx, uint32_t *P, int64_t ldp,
                           int *nonbool, hipStream_t s) {
  if (rows <= 0 || cols <= 0) return hipSuccess;
  PackJob j = pack_job(rows, cols, X, ldx, P, ldp);
  j.nonbool = nonbool;
  return launch_pack_rows(j, PackJob{}, PackJob{}, s);
}

hipError_t launch_unpack_i32(int rows, int cols, const uint32_t *P, int64_t ldp, int *X,
                             int64_t ldx, hipStream_t s) {
  if (rows <= 0 || cols <= 0) return hipSuccess;
  const dim3 grid((unsigned)(((int64_t)rows + 3) / 4));
  if (int_rows_vec(X, ldx))
    unpack_rows_kernel<true><<<grid, dim3(256), 0, s>>>(rows, cols, P, ldp, X, ldx);
  else
    unpack_rows_kernel<false><<<grid, dim3(256), 0, s>>>(rows, cols, P, ldp, X, ldx);
  return hipGetLastError();
}

namespace {

// The packed route of the int32 product: C, X and Y are packed into O itself
// (row r of O: the packed result row, then packed X row r, then rows of
// packed Y), the packed product runs there, and each row is unpacked in
// place.  K goes in parts when O's rows do not hold all of the operands.
// Taken when at least 512 k fit, nothing but the plain product is asked for,
// and C is either O itself or apart from it; and when the one-kernel form
// would take more than one round of one 256-k slab: it packs every operand
// panel again for each 64x64 tile, at about 7 us a slab and round, against
// four launches (13.5 us) here.  With C, one-kernel and packed: 256^3 13.0 and
// 13.9 us, 512^3 20.3 and 13.6, 2048x2048x64 28.7 and 15.2, 4096^3 at density
// 0.02 896 and 86: 128 MiB of operands and 64 of C packed at 6 TB/s, the
// product, 64 MiB of output unpacked at 4.5 TB/s.  Returns false when it does
// not apply.
bool orand_i32_packed(int R, int Cn, int K, const int *X, int64_t ldx, const int *Y, int64_t ldy,
                      int *O, int64_t ldo, const int *C, int64_t ldc, hipStream_t s,
                      hipError_t *status) {
  if (R <= 0 || Cn <= 0 || K <= 0) return false;
  const int64_t tiles =
      (int64_t)((R + IB_BM - 1) / IB_BM) * ((Cn + IB_BN - 1) / IB_BN);
  if (K <= IB_BKW * 32 && tiles <= device_cu_count()) return false;
  if (C && (C != O || ldc != ldo)) {
    const uintptr_t c0 = reinterpret_cast<uintptr_t>(C), o0 = reinterpret_cast<uintptr_t>(O);
    const uintptr_t c1 = c0 + ((uint64_t)(R - 1) * ldc + Cn) * 4;
    const uintptr_t o1 = o0 + ((uint64_t)(R - 1) * ldo + Cn) * 4;
    if (c0 < o1 && o0 < c1) return false;
  }
  // Y's rows go side by side in bands of the largest power of two <= R rows
  int shift = 0;
  while (shift < 30 && (2 << shift) <= R) ++shift;
  auto words = [](int n) { return (int64_t)((n + 127) / 128) * 4; };  // of a packed row, padded
  const int64_t nwp = words(Cn);
  auto fits = [&](int k) {
    return nwp + words(k) + (((int64_t)k + (1 << shift) - 1) >> shift) * nwp <= Cn;
  };
  int part = K;
  while (!fits(part) && part > 512) part = (part / 2 + 127) / 128 * 128;
  if (!fits(part)) return false;
  uint32_t *res = reinterpret_cast<uint32_t *>(O), *px = res + nwp, *py = px + words(part);
  PackJob jc;
  if (C) jc = pack_job(R, Cn, C, ldc, res, ldo);
  hipError_t e = hipSuccess;
  if (C == O) {  // C's rows are packed before X and Y overwrite them
    e = launch_pack_rows(jc, PackJob{}, PackJob{}, s);
    jc = PackJob{};
  }
  for (int k0 = 0; k0 < K && e == hipSuccess; k0 += part) {
    const int k = std::min(part, K - k0);
    PackJob jx = pack_job(R, k, X + k0, ldx, px, ldo);
    PackJob jy = pack_job(k, Cn, Y + (int64_t)k0 * ldy, ldy, py, ldo);
    jy.band = nwp;
    jy.mask = (1 << shift) - 1;
    jy.shift = shift;
    e = launch_pack_rows(jx, jy, jc, s);
    jc = PackJob{};
    if (e == hipSuccess)
      e = launch_orand_rows(R, Cn, k, px, ldo,
                            OrandB{py, (uint32_t)ldo, (uint32_t)nwp, jy.mask, shift}, true,
                            C || k0 > 0 ? res : nullptr, ldo, res, ldo, nullptr, 0, FlagStep{}, s);
  }
  if (e == hipSuccess) e = launch_unpack_i32(R, Cn, res, ldo, O, ldo, s);
  *status = e;
  return true;
}

}  // namespace

hipError_t launch_orand_i32(int R, int Cn, int K, const int *X, int64_t ldx,
                            const int *Y, int64_t ldy, int *O, int64_t ldo,
                            const int *C, int64_t ldc, const int *P,
                            int64_t ldp, int *flag, hipStream_t s) {
  hipError_t status = hipSuccess;
  if (!P && !flag && orand_i32_packed(R, Cn, K, X, ldx, Y, ldy, O, ldo, C, ldc, s, &status))
    return status;
  const int tiles_r = (R + IB_BM - 1) / IB_BM;
  const int tiles_c = (Cn + IB_BN - 1) / IB_BN;
  orand_i32_kernel<<<dim3(tiles_r * tiles_c), dim3(256), 0, s>>>(
      R, Cn, K, X, ldx, Y, ldy, C, ldc, O, ldo, P, ldp, flag, tiles_c);
  return hipGetLastError();
}

}  // namespace simd2
