// LDS-tiled VALU semiring GEMM for gfx950 (the seven float semirings whose
// (+) is min/max, plus the direct minus_square and a VALU plus_mul).
//
// Work decomposition (row-major problem of internal.hpp):
//   * one workgroup computes a BM x BN output tile; each thread a TM x TN
//     register tile, split into 4x4 sub-blocks spaced BM/(TM/4) rows and
//     BN/(TN/4) columns apart so that every LDS read is one ds_read_b128 and
//     the 16 (or more) lanes reading one row of Y hit distinct banks;
//   * K advances in BK-deep slabs, double-buffered in LDS: the next slab's
//     global loads (16 bytes a lane at any row alignment, coalesced along K
//     for X and along columns for Y)
//     are issued before the current slab's arithmetic and written to the
//     other LDS buffer afterwards, one barrier per slab;
//   * X is stored transposed in LDS (k-major, padded by 4 floats so the
//     transposing 32-bit writes of a wave fall in distinct banks);
//   * the inner step handles two k at once: per output, two (x) and one
//     three-input (+) (v_min3_f32 / v_max3_f32), i.e. 3 VALU instructions
//     per 4 semiring operations;
//   * the epilogue fuses C, the convergence change test and per-tile change
//     flags, so the repeated-squaring driver needs no separate pass.
// Tiles are walked XCD-aware: the 8 XCDs receive workgroups round-robin, so
// each XCD is handed one contiguous range of tiles, and inside it tiles are
// visited in groups of GROUP tile-rows so neighbours share panels in L2.
#include <cmath>
#include <mutex>

#include "valu_tile.hpp"

namespace simd2 {

namespace {

// OFFGRID: the shape is not a whole number of tiles and slabs.  Tiles inside
// the matrix differ only in the last, partial K slab, which is loaded element
// by element with the op's padding; edge tiles keep 16-byte loads wherever a
// 4-float group lies inside the matrix (rows past R read as padding, a column
// group past Cn element by element) and mask their stores.  Rows need no
// alignment (valu_tile.hpp).
template <class Op, int BM, int BN, int TM, int TN, int BK, int WAVES, bool OFFGRID>
__global__ __launch_bounds__((BM / TM) * (BN / TN))
__attribute__((amdgpu_waves_per_eu(WAVES))) void srgemm_valu_kernel(
    int R, int Cn, int K, const float *__restrict__ X, int64_t ldx,
    const float *__restrict__ Y, int64_t ldy, float *O, int64_t ldo,
    Epilogue e, int tiles_r, int tiles_c) {
  __shared__ ValuSmem<BM, BN, BK> sm;
  if (flag_done(e.flag, e.step)) return;
  int tr, tc;
  map_tile(bid_x(), tiles_r, tiles_c, tr, tc);
  if (e.gate && e.gate[tr * e.gate_ld + tc] == 0) return;
  int *flag = e.tile_flags ? &e.tile_flags[tr * tiles_c + tc] : nullptr;
  const int row0 = tr * BM, col0 = tc * BN;
  if (!OFFGRID || (row0 + BM <= R && col0 + BN <= Cn))
    valu_tile<Op, BM, BN, TM, TN, BK, false, OFFGRID>(R, Cn, K, X, ldx, Y, ldy, O, ldo, e,
                                                             row0, col0, flag, sm);
  else
    valu_tile<Op, BM, BN, TM, TN, BK, true, true, true>(R, Cn, K, X, ldx, Y, ldy, O, ldo, e,
                                                               row0, col0, flag, sm);
}

// The smallest problems (up to one 64x64 tile per CU) on whole tiles and slabs:
// eight waves per 64x64 tile, each on its own range of slabs with 8x8 outputs
// per lane and its own LDS, so that no barrier holds the waves together; their
// partial tiles are combined in wave order, ((p0 (+) p1) (+) p2) ..., before
// the epilogue.  Only where (+) is min or max, which is exact: regrouping the
// terms changes no bit.  Bound: VALU issue at two waves per SIMD; four groups
// of 256 threads with 4x4 outputs per lane (the split kernel below) read LDS
// twice as often per term and meet at 1024-thread barriers: 1024^3 42 us, here
// 38.  With more tiles a second wave per SIMD hides less than those groups do,
// and so do the masked loads off the grid (1000x1000x700 33 us, 36 this way).
constexpr int WT = 64, WTM = 8, WBK = 16;
constexpr int WG = 8;  // waves per tile

struct WaveSmem {
  __attribute__((aligned(16))) float Xs[2][WBK][WT + 4];
  __attribute__((aligned(16))) float Ys[2][WBK][WT];
};

// Between LDS stores and reads of what other lanes of the same wave stored (or
// the reverse).  A wave's LDS instructions execute in order, so this costs no
// instruction: it keeps the compiler from moving one across the other.
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// acc = the slabs [kt0, kt1) of the tile at X's row and Y's column.  The LDS
// slabs are the wave's own and its LDS instructions execute in order, so
// nothing waits at a barrier: the fragments of a k pair are read while the pair
// before it is computed, the next slab is written to the other buffer in the
// middle of this one and the slab after it requested from memory.
template <class Op>
__device__ __forceinline__ void wave_loop(WaveSmem &sm, float (&acc)[WTM][WTM],
                                          const float *__restrict__ X, int64_t ldx,
                                          const float *__restrict__ Y, int64_t ldy, int kt0,
                                          int kt1, int lane) {
  const int tx = lane % 8, ty = lane / 8;
#pragma unroll
  for (int i = 0; i < WTM; ++i)
#pragma unroll
    for (int j = 0; j < WTM; ++j) acc[i][j] = Op::identity;
  if (kt1 <= kt0) return;
  vf4 xv[4], yv[4];
  auto load = [&](int kt) {
#pragma unroll
    for (int h = 0; h < 4; ++h)
      xv[h] = *reinterpret_cast<const vf4u *>(X + (int64_t)(lane / 4 + 16 * h) * ldx + kt * WBK +
                                              lane % 4 * 4);
#pragma unroll
    for (int h = 0; h < 4; ++h)
      yv[h] = *reinterpret_cast<const vf4u *>(Y + (int64_t)(kt * WBK + lane / 16 + 4 * h) * ldy +
                                              lane % 16 * 4);
  };
  auto store = [&](int buf) {
    store_slab<WT, WT, WBK, 64, WT + 4>(sm.Xs[buf], sm.Ys[buf], xv, yv, lane);
  };
  float a[2][2][WTM], b[2][2][WTM];  // [set][k of the pair][...]
  auto read = [&](int set, int buf, int kp) {
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
      for (int g = 0; g < 2; ++g) {
        *reinterpret_cast<vf4 *>(&a[set][k][g * 4]) =
            *reinterpret_cast<const vf4 *>(&sm.Xs[buf][2 * kp + k][g * 32 + ty * 4]);
        *reinterpret_cast<vf4 *>(&b[set][k][g * 4]) =
            *reinterpret_cast<const vf4 *>(&sm.Ys[buf][2 * kp + k][g * 32 + tx * 4]);
      }
  };
  load(kt0);
  store(0);
  wave_lds_fence();
  load(min(kt0 + 1, kt1 - 1));
  read(0, 0, 0);
  for (int kt = kt0; kt < kt1; ++kt) {
    const int buf = (kt - kt0) & 1;
#pragma unroll
    for (int kp = 0; kp < WBK / 2; ++kp) {
      __builtin_amdgcn_sched_barrier(0);
      if (kp == WBK / 4) {
        wave_lds_fence();
        store(buf ^ 1);
        wave_lds_fence();
        load(min(kt + 2, kt1 - 1));
      }
      const int s = kp & 1;
      if (kp + 1 < WBK / 2) read(s ^ 1, buf, kp + 1);
      else read(s ^ 1, buf ^ 1, 0);
#pragma unroll
      for (int i = 0; i < WTM; ++i)
#pragma unroll
        for (int j = 0; j < WTM; ++j)
          acc[i][j] = Op::add3(acc[i][j], Op::mul(a[s][0][i], b[s][0][j]),
                               Op::mul(a[s][1][i], b[s][1][j]));
    }
  }
}

template <class Op>
__global__ __launch_bounds__(64 * WG) __attribute__((amdgpu_waves_per_eu(2))) void
srgemm_wave_kernel(int K, const float *__restrict__ X, int64_t ldx, const float *__restrict__ Y,
                   int64_t ldy, float *O, int64_t ldo, Epilogue e, int tiles_r, int tiles_c) {
  __shared__ WaveSmem sm[WG];
  __shared__ int any_changed;
  if (flag_done(e.flag, e.step)) return;
  int tr, tc;
  map_tile(bid_x(), tiles_r, tiles_c, tr, tc);
  const int row0 = tr * WT, col0 = tc * WT;
  const int lane = tid_x() % 64, w = __builtin_amdgcn_readfirstlane(tid_x() / 64);
  const int slabs = K / WBK, per = (slabs + WG - 1) / WG;
  const int kt0 = min(w * per, slabs), kt1 = min(kt0 + per, slabs);
  if (tid_x() == 0) any_changed = 0;
  float acc[WTM][WTM];
  wave_loop<Op>(sm[w], acc, X + (int64_t)row0 * ldx, ldx, Y + col0, ldy, kt0, kt1, lane);
  // every wave parks its partial tile in its own slabs and finishes one of the
  // register tile's rows
  static_assert(WTM * WTM * 64 * sizeof(float) <= sizeof(WaveSmem), "partial tile");
  static_assert(WTM == WG, "one row of the register tile per wave");
  wave_lds_fence();
  vf4 *part = reinterpret_cast<vf4 *>(&sm[w]);
#pragma unroll
  for (int i = 0; i < WTM; ++i)
#pragma unroll
    for (int g = 0; g < 2; ++g)
      part[(i * 2 + g) * 64 + lane] =
          vf4{acc[i][g * 4], acc[i][g * 4 + 1], acc[i][g * 4 + 2], acc[i][g * 4 + 3]};
  // C and the previous values travel while the partial tiles are combined (a
  // squaring loop passes the same matrix as both)
  const int tx = lane % 8, ty = lane / 8;
  const int r = row0 + w / 4 * 32 + ty * 4 + w % 4;
  vf4 cv[2], pv[2];
#pragma unroll
  for (int g = 0; g < 2; ++g) {
    const int c = col0 + g * 32 + tx * 4;
    cv[g] = pv[g] = vf4{0.f, 0.f, 0.f, 0.f};
    if (e.C) cv[g] = *reinterpret_cast<const vf4u *>(e.C + (int64_t)r * e.ldc + c);
    if (e.P == e.C && e.ldp == e.ldc) pv[g] = cv[g];
    else if (e.P) pv[g] = *reinterpret_cast<const vf4u *>(e.P + (int64_t)r * e.ldp + c);
  }
  __syncthreads();
  bool changed = false;
#pragma unroll
  for (int g = 0; g < 2; ++g) {
    float v[4];
#pragma unroll
    for (int q = 0; q < WG; ++q) {
      const vf4 p = reinterpret_cast<const vf4 *>(&sm[q])[(w * 2 + g) * 64 + lane];
#pragma unroll
      for (int z = 0; z < 4; ++z) v[z] = q == 0 ? p[z] : Op::add(v[z], p[z]);
    }
#pragma unroll
    for (int z = 0; z < 4; ++z) {
      if (e.C) v[z] = Op::add(v[z], cv[g][z]);
      if (e.mode == CHECK_APLP && v[z] > -1.0f && v[z] < 1.0f) v[z] = -FLT_MAX;
      if (e.P) changed |= differs(v[z], pv[g][z], e.mode);
    }
    *reinterpret_cast<vf4u *>(O + (int64_t)r * ldo + col0 + g * 32 + tx * 4) =
        vf4u{v[0], v[1], v[2], v[3]};
  }
  if (e.flag) {  // one atomic per tile at most (valu_epilogue)
    if (__any(changed) && lane == 0) any_changed = 1;
    __syncthreads();
    if (tid_x() == 0 && any_changed) atomicMax(e.flag, e.step);
  }
}

// Small problems (at most four 64x64 tiles per CU): the K
// loop of each tile is split over G groups of 256 threads in one workgroup
// (G: splitk_groups), each over a contiguous range of
// slabs with its own LDS buffers, and the partial tiles are combined in
// group order, ((p0 (+) p1) (+) p2) (+) p3, before the usual epilogue: G
// times the resident waves.  Only for the semirings whose (+) is min or max,
// which is exact: regrouping the terms changes no bit.  RAGGED: any shape, as
// OFFGRID above; every group runs ceil(slabs / G) slabs, the ranges past K
// reading padding, whose terms are the (+)-identity.
template <class Op, int SK_GROUPS, bool RAGGED>
__global__ __launch_bounds__(256 * SK_GROUPS) void srgemm_valu_splitk_kernel(
    int R, int Cn, int K, const float *__restrict__ X, int64_t ldx,
    const float *__restrict__ Y, int64_t ldy, float *O, int64_t ldo, Epilogue e,
    int tiles_r, int tiles_c) {
  using S = CfgS;
  __shared__ ValuSmem<S::BM, S::BN, S::BK> sm[SK_GROUPS];
  if (flag_done(e.flag, e.step)) return;
  int tr, tc;
  map_tile(bid_x(), tiles_r, tiles_c, tr, tc);
  int *flag = e.tile_flags ? &e.tile_flags[tr * tiles_c + tc] : nullptr;
  const int row0 = tr * S::BM, col0 = tc * S::BN;
  const int g = tid_x() / 256, t = tid_x() % 256;
  if (tid_x() == 0) sm[0].changed = 0;  // published by the main loop's barriers
  const int per = ((K + S::BK - 1) / S::BK + SK_GROUPS - 1) / SK_GROUPS;
  float acc[S::TM][S::TN];
  if (!RAGGED || (row0 + S::BM <= R && col0 + S::BN <= Cn))
    valu_mainloop<Op, S::BM, S::BN, S::TM, S::TN, S::BK, false, RAGGED>(
        R, Cn, K, X, ldx, Y, ldy, row0, col0, nullptr, 0, sm[g], acc, t, g * per, (g + 1) * per);
  else
    valu_mainloop<Op, S::BM, S::BN, S::TM, S::TN, S::BK, false, true, true>(
        R, Cn, K, X, ldx, Y, ldy, row0, col0, nullptr, 0, sm[g], acc, t, g * per, (g + 1) * per);
  // The main loop ends with a barrier after every read of the slabs: groups
  // 1.. park their partial tiles in their own LDS (16 KB of its 16.5).
  static_assert(S::TM * S::TN * 256 * sizeof(float) <= sizeof(ValuSmem<S::BM, S::BN, S::BK>) -
                                                           sizeof(int), "partial tile");
  if (g > 0) {
    float *part = reinterpret_cast<float *>(&sm[g]);
#pragma unroll
    for (int i = 0; i < S::TM; ++i)
#pragma unroll
      for (int j = 0; j < S::TN; ++j) part[(i * S::TN + j) * 256 + t] = acc[i][j];
  }
  __syncthreads();
  if (g == 0) {
#pragma unroll
    for (int q = 1; q < SK_GROUPS; ++q) {
      const float *part = reinterpret_cast<const float *>(&sm[q]);
#pragma unroll
      for (int i = 0; i < S::TM; ++i)
#pragma unroll
        for (int j = 0; j < S::TN; ++j)
          acc[i][j] = Op::add(acc[i][j], part[(i * S::TN + j) * 256 + t]);
    }
  }
  valu_epilogue<Op, S::BM, S::BN, S::TM, S::TN, RAGGED>(R, Cn, O, ldo, e, row0, col0,
                                                               flag, &sm[0].changed, acc, t,
                                                               g == 0);
}

// groups 8: the wave kernel; 4 or 2: whole tiles and slab groups; -4 or -2: the
// ragged form of as many groups.
template <class Op>
hipError_t launch_splitk(int R, int Cn, int K, const float *X, int64_t ldx, const float *Y,
                         int64_t ldy, float *O, int64_t ldo, const Epilogue &e, int groups,
                         hipStream_t s) {
  const int tiles_r = (R + CfgS::BM - 1) / CfgS::BM, tiles_c = (Cn + CfgS::BN - 1) / CfgS::BN;
  const dim3 grid(tiles_r * tiles_c);
  if (groups == WG)
    srgemm_wave_kernel<Op><<<grid, dim3(64 * WG), 0, s>>>(K, X, ldx, Y, ldy, O, ldo, e, tiles_r,
                                                          tiles_c);
  else if (groups == 4)
    srgemm_valu_splitk_kernel<Op, 4, false><<<grid, dim3(1024), 0, s>>>(
        R, Cn, K, X, ldx, Y, ldy, O, ldo, e, tiles_r, tiles_c);
  else if (groups == 2)
    srgemm_valu_splitk_kernel<Op, 2, false><<<grid, dim3(512), 0, s>>>(
        R, Cn, K, X, ldx, Y, ldy, O, ldo, e, tiles_r, tiles_c);
  else if (groups == -4)
    srgemm_valu_splitk_kernel<Op, 4, true><<<grid, dim3(1024), 0, s>>>(
        R, Cn, K, X, ldx, Y, ldy, O, ldo, e, tiles_r, tiles_c);
  else
    srgemm_valu_splitk_kernel<Op, 2, true><<<grid, dim3(512), 0, s>>>(
        R, Cn, K, X, ldx, Y, ldy, O, ldo, e, tiles_r, tiles_c);
  return hipGetLastError();
}

template <class Op, class Cfg>
hipError_t launch_cfg(int R, int Cn, int K, const float *X, int64_t ldx,
                      const float *Y, int64_t ldy, float *O, int64_t ldo,
                      const Epilogue &e, hipStream_t s) {
  const int tiles_r = (R + Cfg::BM - 1) / Cfg::BM;
  const int tiles_c = (Cn + Cfg::BN - 1) / Cfg::BN;
  const int nthreads = (Cfg::BM / Cfg::TM) * (Cfg::BN / Cfg::TN);
  const dim3 grid(tiles_r * tiles_c), block(nthreads);
  if (R % Cfg::BM == 0 && Cn % Cfg::BN == 0 && K % Cfg::BK == 0)
    srgemm_valu_kernel<Op, Cfg::BM, Cfg::BN, Cfg::TM, Cfg::TN, Cfg::BK, Cfg::WAVES, false>
        <<<grid, block, 0, s>>>(R, Cn, K, X, ldx, Y, ldy, O, ldo, e, tiles_r, tiles_c);
  else
    srgemm_valu_kernel<Op, Cfg::BM, Cfg::BN, Cfg::TM, Cfg::TN, Cfg::BK, Cfg::WAVES, true>
        <<<grid, block, 0, s>>>(R, Cn, K, X, ldx, Y, ldy, O, ldo, e, tiles_r, tiles_c);
  return hipGetLastError();
}

template <class Op>
hipError_t launch_op(int R, int Cn, int K, const float *X, int64_t ldx,
                     const float *Y, int64_t ldy, float *O, int64_t ldo,
                     const Epilogue &e, hipStream_t s, int cfg) {
  if (cfg == CFG_S64) return launch_cfg<Op, CfgS>(R, Cn, K, X, ldx, Y, ldy, O, ldo, e, s);
  if (cfg == CFG_M128x64) return launch_cfg<Op, CfgM>(R, Cn, K, X, ldx, Y, ldy, O, ldo, e, s);
  return launch_cfg<Op, CfgL>(R, Cn, K, X, ldx, Y, ldy, O, ldo, e, s);
}

}  // namespace

int device_cu_count() {
  static int cus = 0;
  if (cus == 0) {
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) == hipSuccess &&
        hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && n > 0)
      cus = n;
    else
      cus = 256;
  }
  return cus;
}

ValuCfgInfo valu_cfg_info(int cfg) {
  if (cfg == CFG_S64) return {CfgS::BM, CfgS::BN, CfgS::BK, 256};
  if (cfg == CFG_M128x64) return {CfgM::BM, CfgM::BN, CfgM::BK, 256};
  return {CfgL::BM, CfgL::BN, CfgL::BK, 256};
}

// Tile shape choice, measured on MI355X (us in 64x64, 128x64 and 128x128 tiles).
// What a size wastes is its last round over the CUs.  The 64x64 tiles' many
// workgroups waste least (min_plus 3328^3: 965, 1058, 1181; 4608: 2451, 2570,
// 2891; 5120: 3260, 3337, 3663).  The larger tiles read LDS less and win where
// their rounds fill:
//   * minus_square, whose step is one instruction shorter, in 128x128 tiles from
//     more than three per CU up (4096^2 x 1024: 699, 672, 651; 8192x4096x1000
//     1317, 1290, 1244; 5376^2 x 300 358, 350, 340; rounds not full: 4608^2 x 300
//     269, 274, 286; 5120^2 x 300 322, 329, 333).  Below K = 128 the memory is the
//     bound and more workgroups keep it busier with C (8192^2 x 16 108, 140, 165;
//     x 64 215, 223, 237; without C 68, 65, 68 and 198, 196, 192);
//   * the others in 128x128 tiles from 5900^2 up, where three per CU at once fill
//     (6144^3: 5558, 5407, 5479; 8192: 12893, 12620, 12588; not full: 7168: 8788,
//     8782, 9090), and in 128x64 tiles at eight and more full rounds up to 4096^2
//     (max_mul 4096^3 1718, 1699, 1759; min_plus within 1%; not full: 3900^2 x 512
//     208, 225, 236; 4100^2 x 512 235, 245, 281).  Above, those gain 1 to 3% again at
//     some sizes, but the scheduled loop, which asks here too, can halve the work of
//     square tiles only.
// Shapes the autotuner has timed (simd2_autotune) use the recorded winner instead.
namespace {
struct TunedEntry { int op, R, Cn, K, cfg; };
constexpr int TUNED_MAX = 64;
TunedEntry g_tuned[TUNED_MAX];
int g_tuned_n = 0;
std::mutex g_tuned_mu;
}  // namespace

void valu_record_cfg(int op, int R, int Cn, int K, int cfg) {
  std::lock_guard<std::mutex> lock(g_tuned_mu);
  for (int i = 0; i < g_tuned_n; ++i)
    if (g_tuned[i].op == op && g_tuned[i].R == R && g_tuned[i].Cn == Cn && g_tuned[i].K == K) {
      g_tuned[i].cfg = cfg;
      return;
    }
  const int slot = g_tuned_n < TUNED_MAX ? g_tuned_n++ : (op + R + Cn + K) % TUNED_MAX;
  g_tuned[slot] = {op, R, Cn, K, cfg};
}

int valu_pick_cfg(int op, int R, int Cn, int K) {
  {
    std::lock_guard<std::mutex> lock(g_tuned_mu);
    for (int i = 0; i < g_tuned_n; ++i)
      if (g_tuned[i].op == op && g_tuned[i].R == R && g_tuned[i].Cn == Cn && g_tuned[i].K == K)
        return g_tuned[i].cfg;
  }
  const int64_t cus = device_cu_count();
  const double area = (double)R * Cn;
  const double a = area * (256.0 / cus);   // rule is for 256 CUs
  auto tiles = [&](int bm, int bn) {
    return (int64_t)((R + bm - 1) / bm) * ((Cn + bn - 1) / bn);
  };
  // share of the CUs' rounds that ends up as outputs
  auto fill = [&](int bm, int bn) {
    const int64_t rounds = (tiles(bm, bn) + cus - 1) / cus;
    return area / ((double)bm * bn * cus * rounds);
  };
  if (op == 8 && K < 128) return CFG_S64;
  if (op == 8 && tiles(128, 128) > 3 * cus && fill(128, 128) >= 0.91) return CFG_L128;
  if (a <= 4096.0 * 4096.0 * 1.01)
    return tiles(128, 64) >= 8 * cus && fill(128, 64) >= 0.975 ? CFG_M128x64 : CFG_S64;
  const double rounds = (double)tiles(128, 128) / (3 * cus);
  return a >= 5900.0 * 5900.0 && rounds >= 0.85 * ceil(rounds) ? CFG_L128 : CFG_S64;
}

// How a min / max semiring splits K where the 64x64 tiles were chosen and are
// few: 8 -- the wave kernel, on whole tiles and slabs up to one tile per CU with
// at least two slabs a wave (64x64x1024 36.8 us in four groups, 31.7; 512^3 21.5
// and 19.6; 1024x1024x256 15.0 and 14.0; x128 9.8 both); 4 or 2 -- groups of
// 256 threads, negative off the grid; 0 -- unsplit, from four tiles per CU up
// (1999x1801x777 104 us in two, 111 unsplit).  Four groups pay where a CU has
// one workgroup, or two of the form without bounds, and each group some slabs
// (1408^3 87 us in four, 92 in two; 1025x1023x1021 77 and 69; 1100x1000x200 27
// and 21.5; 1024x1024x96 11.0 and 8.5).  Never more groups than slabs
// (16x16x16 7.4 us in four groups, 5.3 unsplit; 16x16x32 8.0, 5.8 in two, 6.2
// unsplit; 1500x1400x32 9.8 in two, 9.1 unsplit).
static int splitk_groups(int op, int R, int Cn, int K, const Epilogue &e) {
  if (op == 1 || op == 8 || op < 0 || op > 6 || e.gate || K <= 0) return 0;
  const int64_t tiles =
      (int64_t)((R + CfgS::BM - 1) / CfgS::BM) * ((Cn + CfgS::BN - 1) / CfgS::BN);
  const int64_t cus = device_cu_count();
  if (R % WT == 0 && Cn % WT == 0 && K % WBK == 0 && K >= 2 * WBK * WG && tiles <= cus &&
      !e.tile_flags)
    return WG;
  if (tiles > 4 * cus || K <= CfgS::BK || (K <= 2 * CfgS::BK && tiles >= 2 * cus)) return 0;
  const bool whole = R % CfgS::BM == 0 && Cn % CfgS::BN == 0;
  const bool whole4 = whole && K % (CfgS::BK * 4) == 0;
  if (K > 8 * CfgS::BK && (tiles <= cus || (tiles < 2 * cus && whole4))) return whole4 ? 4 : -4;
  return whole && K % (CfgS::BK * 2) == 0 ? 2 : -2;
}

hipError_t launch_valu_f32(int op, int R, int Cn, int K, const float *X,
                           int64_t ldx, const float *Y, int64_t ldy, float *O,
                           int64_t ldo, const Epilogue &e, hipStream_t s,
                           int cfg) {
  if (cfg == CFG_AUTO) {
    cfg = valu_pick_cfg(op, R, Cn, K);
    const int g = cfg == CFG_S64 ? splitk_groups(op, R, Cn, K, e) : 0;
    if (g) {
      switch (op) {
      case 0: return launch_splitk<MinPlus>(R, Cn, K, X, ldx, Y, ldy, O, ldo, e, g, s);
      case 2: return launch_splitk<MaxPlus>(R, Cn, K, X, ldx, Y, ldy, O, ldo, e, g, s);
      case 3: return launch_splitk<MaxMin>(R, Cn, K, X, ldx, Y, ldy, O, ldo, e, g, s);
      case 4: return launch_splitk<MaxMul>(R, Cn, K, X, ldx, Y, ldy, O, ldo, e, g, s);
      case 5: return launch_splitk<MinMul>(R, Cn, K, X, ldx, Y, ldy, O, ldo, e, g, s);
      case 6: return launch_splitk<MinMax>(R, Cn, K, X, ldx, Y, ldy, O, ldo, e, g, s);
      default: break;
      }
    }
  }
  switch (op) {
  case 0: return launch_op<MinPlus>(R, Cn, K, X, ldx, Y, ldy, O, ldo, e, s, cfg);
  case 1: return launch_op<PlusMul>(R, Cn, K, X, ldx, Y, ldy, O, ldo, e, s, cfg);
  case 2: return launch_op<MaxPlus>(R, Cn, K, X, ldx, Y, ldy, O, ldo, e, s, cfg);
  case 3: return launch_op<MaxMin>(R, Cn, K, X, ldx, Y, ldy, O, ldo, e, s, cfg);
  case 4: return launch_op<MaxMul>(R, Cn, K, X, ldx, Y, ldy, O, ldo, e, s, cfg);
  case 5: return launch_op<MinMul>(R, Cn, K, X, ldx, Y, ldy, O, ldo, e, s, cfg);
  case 6: return launch_op<MinMax>(R, Cn, K, X, ldx, Y, ldy, O, ldo, e, s, cfg);
  case 8: return launch_op<MinusSquare>(R, Cn, K, X, ldx, Y, ldy, O, ldo, e, s, cfg);
  default: return hipErrorInvalidValue;
  }
}

}  // namespace simd2
