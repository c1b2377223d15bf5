// Launches of the fp16 GEMMs over the MFMA GEMM core: tile shape, K slices and grid per problem.
// Included by one source file per group of kernel instances, which compile side by side.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdlib>

#include "gemm_core.h"
#include "gemm_dtl.h"

namespace mthip {

int gemm_cu_count(int device);
int launch_linear_rows(const GemmArgs& a, int mf, hipStream_t s);

namespace {

// Workgroup tile and wave layout (4 waves): T128x128 = 2x2 waves of 64x64, T128x64w4 = 4x1
// waves of 32x64, T64x128w1 = 1x4 waves of 64x32, T64x64 = 2x2 waves of 32x32.
enum TileKind { T128x128, T128x64w4, T64x128w1, T64x64 };

TileKind pick_tile(int MODE, int64_t M, int64_t N, int64_t batch) {
  // MTHIP_GEMM_TILE=0..3 forces a tile shape (tuning sweeps); unset selects by problem size.
  if (const char* force = std::getenv("MTHIP_GEMM_TILE")) {
    const int t = std::atoi(force);
    if (t >= 0 && t <= 3) return static_cast<TileKind>(t);
  }
  (void)M;
  (void)batch;
  // 64x64 everywhere: in isolation 128x128 tiles ran some large convs 5-20% faster, but inside
  // the UNet step (bias/residual epilogues, split-K interplay) they were 13% slower in total;
  // the four resident 64x64 workgroups per CU also hide the short K loops of the linears.
  (void)MODE;
  (void)N;
  return T64x64;
}

// Tuning switches for sweeps: MTHIP_GEMM_SPLITK=0 disables K splitting, MTHIP_GEMM_PERSIST=0
// launches one workgroup per unit, MTHIP_GEMM_XCD=0/1 forces the plain / XCD-contiguous unit
// order (default: XCD-contiguous), MTHIP_GEMM_MFAST=0/1 forces which tile dimension varies
// fastest (default: the one with fewer tiles), MTHIP_GEMM_SPLIT_TARGET sets the split-K units
// per CU.
int env_flag(const char* name, int dflt) {
  const char* e = std::getenv(name);
  return e ? std::atoi(e) : dflt;
}
bool splitk_enabled() { return env_flag("MTHIP_GEMM_SPLITK", 1) != 0; }
bool persist_enabled() { return env_flag("MTHIP_GEMM_PERSIST", 1) != 0; }
int xcd_mode() { return env_flag("MTHIP_GEMM_XCD", 2); }
int split_target() { return std::max(1, env_flag("MTHIP_GEMM_SPLIT_TARGET", 4)); }

int cu_count(int device) { return gemm_cu_count(device); }

// The kernel instance behind a tile choice: DS > 0 selects the direct-to-LDS fp16 kernel
// with DS stages, DS == 0 the register-staged kernel.
template <typename T, int BM, int BN, int MODE, int EPI, int ACT, bool FAST, int WGM, int DS>
constexpr auto gemm_kernel_ptr() {
  if constexpr (DS > 0) {
    static_assert(sizeof(T) == 2 && (MODE == MODE_NT || (MODE == MODE_CONV && FAST)), "direct-to-LDS: fp16, k-contiguous");
    return &gemm_dtl_kernel<BM, BN, WGM, MODE, EPI, ACT, DS>;
  } else {
    return &gemm_kernel<T, BM, BN, WGM, MODE, EPI, ACT, FAST>;
  }
}

// Resident workgroups per CU of one kernel instance (registers and LDS decide it).
template <typename T, int BM, int BN, int MODE, int EPI, int ACT, bool FAST, int WGM, int DS>
int resident_per_cu() {
  static const int v = [] {
    int n = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, gemm_kernel_ptr<T, BM, BN, MODE, EPI, ACT, FAST, WGM, DS>(),
                                                     256, 0) != hipSuccess ||
        n < 1)
      n = 1;
    return n;
  }();
  return v;
}

// Sizes the persistent grid, splits K when the output tiles cannot fill the chip, launches the
// GEMM (and the slice reduction).
template <typename T, int BM, int BN, int MODE, int EPI, int ACT, bool FAST, int WGM = 2, int DS = 0>
int launch_tile(int device, GemmArgs a, int64_t batch, hipStream_t s) {
  constexpr int BK = Mfma<T>::BK;
  a.tiles_m = ceil_div(a.M, BM);
  a.tiles_n = ceil_div(a.N, BN);
  const int64_t nk = std::max<int64_t>(ceil_div(a.K, BK), 1);
  const int64_t tiles = a.tiles_m * a.tiles_n * batch;
  const int64_t slots = (int64_t)cu_count(device) * resident_per_cu<T, BM, BN, MODE, EPI, ACT, FAST, WGM, DS>();
  int64_t ksplit = 1;
  if (batch == 1 && nk >= 16 && splitk_enabled() && EPI != EPI_GEGLU) {
    if (DS > 0) {
      // Pick the slice count with the shortest modelled makespan: the persistent grid runs
      // ceil(units / slots) rounds of ceil(nk / ksplit) K tiles, and every extra slice adds an
      // fp32 M x N write here plus its read in the reduction kernel.  (640 tiles on 768 slots
      // gain nothing from 2 slices -- 2 rounds of half the K -- and would pay the reduction.)
      constexpr double kStepUs = 0.6, kReduceBytesPerUs = 3.0e6;
      const double kReduceFixedUs = env_flag("MTHIP_GEMM_REDUCE_US", 3);
      double best = 0.0;
      const int64_t max_split = std::min<int64_t>(16, nk / 8);
      for (int64_t ks = 1; ks <= max_split; ++ks) {
        const int64_t rounds = ceil_div(tiles * ks, slots);
        double t = (double)(rounds * ceil_div(nk, ks)) * kStepUs;
        if (ks > 1) t += kReduceFixedUs + (double)((ks + 1) * a.M * a.N * 4) / kReduceBytesPerUs;
        if (ks == 1 || t < best) {
          best = t;
          ksplit = ks;
        }
      }
      if (const char* force = std::getenv("MTHIP_GEMM_KSPLIT")) ksplit = std::max(1, std::min(16, std::atoi(force)));
    } else {
      // Register-staged kernel: split single-batch problems with fewer tiles than about
      // `split_target` units per CU and >= 32 K tiles into enough slices to reach that, each
      // slice keeping >= 16 K tiles.
      const int64_t target = (int64_t)cu_count(device) * split_target();
      if (tiles < target && nk >= 32)
        ksplit = std::max<int64_t>(1, std::min<int64_t>(std::min<int64_t>(ceil_div(target, tiles), nk / 16), 16));
    }
  }
  a.kt_per_split = ceil_div(nk, ksplit);
  a.ksplit = ceil_div(nk, a.kt_per_split);  // no empty slice
  if constexpr (DS > 0 && MODE == MODE_NT && EPI == EPI_LINEAR) {
    if (a.rows_vec) return launch_linear_rows(a, 32, s);  // the same slices and bits
  }
  a.units = tiles * a.ksplit;
  MTHIP_REQUIRE(a.units < (int64_t(1) << 31) && a.N < (int64_t(1) << 31) && a.M < (int64_t(1) << 31),
                "gemm: problem too large (tiles, rows or columns beyond 2^31)");
  a.div_tiles_n = FastDiv((uint32_t)a.tiles_n);
  a.div_tiles_m = FastDiv((uint32_t)a.tiles_m);
  a.div_ksplit = FastDiv((uint32_t)a.ksplit);
  if (MODE == MODE_CONV) {
    a.div_ohw = FastDiv((uint32_t)(a.OH * a.OW));
    a.div_ow = FastDiv((uint32_t)a.OW);
  }
  int64_t g = persist_enabled() ? std::min(a.units, slots) : a.units;
  if (g > 8 && g < a.units) g = g / 8 * 8;  // a multiple of 8 keeps each XCD on its own run of tiles
  // Unit order and L2 reuse: each XCD takes a contiguous band of the operand with more tiles
  // and walks all tiles of the other operand fastest, so it holds 1/8 of the large operand
  // and all of the small one.  (Dealt round-robin instead, a conv's XCD would see every 8th
  // pixel tile and fetch every 3x3 halo row from memory: 2.9x the operand bytes, measured.)
  const int xm = xcd_mode();
  a.xcd_remap = xm == 0 ? 0 : 1;
  a.m_fast = a.tiles_m * batch <= a.tiles_n ? 1 : 0;
  if (const char* f = std::getenv("MTHIP_GEMM_MFAST")) a.m_fast = std::atoi(f) != 0;
  void* ws = nullptr;
  if (a.ksplit > 1) {
    a.ld_partial = ceil_div(a.N, 4) * 4;
    if (int rc = mthip_malloc(device, (size_t)(a.ksplit * a.M * a.ld_partial) * sizeof(float), &ws)) return rc;
    a.partial = static_cast<float*>(ws);
  }
  hipLaunchKernelGGL((gemm_kernel_ptr<T, BM, BN, MODE, EPI, ACT, FAST, WGM, DS>()), dim3((unsigned)g), dim3(256), 0, s, a);
  int rc = check_launch("gemm_kernel");
  if constexpr (EPI == EPI_GEGLU) return rc;
  if (rc == MTHIP_OK && a.ksplit > 1) {
    const int64_t work = a.M * ceil_div(a.N, 4);
    const unsigned rg = (unsigned)std::min<int64_t>(ceil_div(work, 256), 8192);
    hipLaunchKernelGGL((gemm_splitk_reduce_kernel<T, EPI, ACT>), dim3(rg), dim3(256), 0, s, a);
    rc = check_launch("gemm_splitk_reduce_kernel");
  }
  if (ws) mthip_free(device, ws);  // stream-ordered: reused only by later work
  return rc;
}

// Direct-to-LDS tile shapes (fp16, k-contiguous operands): MTHIP_GEMM_DTL=0 turns the kernel
// off, MTHIP_GEMM_DTL_TILE=0..5 forces one of
//   0: 64x64 (2x2 waves of 32x32), 3 stages     1: 64x64, 4 stages
//   2: 128x64 (2x2 waves of 64x32), 3 stages    3: 64x128 (2x2 waves of 32x64), 3 stages
//   4: 128x128 (2x2 waves of 64x64), 3 stages   5: 128x128, 2 stages
bool dtl_enabled() { return env_flag("MTHIP_GEMM_DTL", 1) != 0; }

// Default shape per problem, from sweeps of the SD-1.5 GEMMs and convs (fp16, batch 2):
// convs over more than 128 output pixels with a multiple of 128 output channels take 128x64
// (5-18% over 64x64 at 640 and 1280 channels; at 320 channels the third 128-row tile is half
// empty and 64x64 is 9% faster), the 8x8 convs (long K, split) and every conv with K >= 2048
// 64x64 with 4 stages (the SD stride-2 downsampling convs, graph-replayed with the layout pass:
// 320 @64x64 27.4 -> 26.3 us, 640 @32x32 27.4 -> 24.6 us against 64x64 / 128x64 with 3 stages,
// which date from before the 3x3 stride-1 convs moved to the halo kernel); linears take
// 64x64 (3 stages) up to K = 1280, 4 stages beyond, 64x128 when M*N is large, 128x128 with 2
// stages for the big square problems.
int dtl_tile_for(int MODE, int64_t M, int64_t N, int64_t K) {
  const int forced = env_flag("MTHIP_GEMM_DTL_TILE", -1);
  if (forced >= 0) return forced;
  if (MODE == MODE_CONV) return (N <= 128 || K >= 2048) ? 1 : M % 128 == 0 ? 2 : 0;
  if (M >= 4096 && N >= 4096 && K >= 2048) return 5;
  if (K >= 2048) return 1;
  if (M * N >= (int64_t)2048 * 1920 && K >= 640) return 3;
  return 0;
}

template <int MODE, int EPI, int ACT>
int launch_dtl(int device, const GemmArgs& a, int64_t batch, hipStream_t s) {
  using T = uint16_t;
  constexpr bool F = MODE == MODE_CONV;
  if constexpr (EPI == EPI_GEGLU) {
    // MTHIP_GEMM_GEGLU_TILE: 0 = 128x64 (4x1 waves of 32x64), 1 = 128x128 (2x2 waves of 64x64)
    // with 3 stages, 2 = 128x128 with 2 stages.  By default 128x128 / 2 stages where the 128x64
    // tiles number >= 2560 or, over >= 512 rows, <= 640 (SD feed-forward, graph-replayed:
    // 8192x2560x320 43.7 -> 38.9 us, 512x10240x1280 30.7 -> 29.4; 4096x2560x320 22.7 against
    // 23.6 and 2048x5120x640 even stay on 128x64; 3 stages hold one workgroup per CU and lose
    // everywhere).
    const int64_t t64 = ceil_div(a.M, 128) * ceil_div(a.N, 64) * batch;
    const int dflt = (t64 >= 2560 || (a.M >= 512 && t64 <= 640)) ? 2 : 0;
    switch (env_flag("MTHIP_GEMM_GEGLU_TILE", dflt)) {
      case 1:
        return launch_tile<T, 128, 128, MODE, EPI, ACT, F, 2, 3>(device, a, batch, s);
      case 2:
        return launch_tile<T, 128, 128, MODE, EPI, ACT, F, 2, 2>(device, a, batch, s);
      default:
        return launch_tile<T, 128, 64, MODE, EPI, ACT, F, 4, 3>(device, a, batch, s);
    }
  } else if constexpr (ACT != MTHIP_ACT_NONE) {
    switch (env_flag("MTHIP_GEMM_DTL_TILE", 0)) {
      case 3:
        return launch_tile<T, 64, 128, MODE, EPI, ACT, F, 2, 3>(device, a, batch, s);
      case 5:
        return launch_tile<T, 128, 128, MODE, EPI, ACT, F, 2, 2>(device, a, batch, s);
      default:
        return launch_tile<T, 64, 64, MODE, EPI, ACT, F, 2, 3>(device, a, batch, s);
    }
  } else {
    switch (dtl_tile_for(MODE, a.M, a.N, a.K)) {
      case 1:
        return launch_tile<T, 64, 64, MODE, EPI, ACT, F, 2, 4>(device, a, batch, s);
      case 2:
        return launch_tile<T, 128, 64, MODE, EPI, ACT, F, 2, 3>(device, a, batch, s);
      case 3:
        return launch_tile<T, 64, 128, MODE, EPI, ACT, F, 2, 3>(device, a, batch, s);
      case 4:
        return launch_tile<T, 128, 128, MODE, EPI, ACT, F, 2, 3>(device, a, batch, s);
      case 5:
        return launch_tile<T, 128, 128, MODE, EPI, ACT, F, 2, 2>(device, a, batch, s);
      default:
        return launch_tile<T, 64, 64, MODE, EPI, ACT, F, 2, 3>(device, a, batch, s);
    }
  }
}

template <typename T, int MODE, int EPI, int ACT, bool FAST>
int launch_gemm_tiles(int device, const GemmArgs& a, int64_t batch, hipStream_t s) {
  if constexpr (sizeof(T) == 2 && (MODE == MODE_NT || (MODE == MODE_CONV && FAST))) {
    if (dtl_enabled()) return launch_dtl<MODE, EPI, ACT>(device, a, batch, s);
  }
  switch (pick_tile(MODE, a.M, a.N, batch)) {
    case T128x128:
      return launch_tile<T, 128, 128, MODE, EPI, ACT, FAST>(device, a, batch, s);
    case T128x64w4:
      return launch_tile<T, 128, 64, MODE, EPI, ACT, FAST, 4>(device, a, batch, s);
    case T64x128w1:
      return launch_tile<T, 64, 128, MODE, EPI, ACT, FAST, 1>(device, a, batch, s);
    default:
      return launch_tile<T, 64, 64, MODE, EPI, ACT, FAST>(device, a, batch, s);
  }
}

template <typename T, int MODE, int EPI>
int launch_gemm(int device, const GemmArgs& a, int64_t batch, hipStream_t s) {
  return launch_gemm_tiles<T, MODE, EPI, MTHIP_ACT_NONE, false>(device, a, batch, s);
}

}  // namespace
}  // namespace mthip
