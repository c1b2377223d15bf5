// fp16 linear with few rows: y[M, N] = act(x[M, K] . w[N, K]^T + b) (+ residual), M <= 16 -- the
// timestep MLP and the time projections of an SD UNet (M = 2).
//
// Returns the bits of the tile GEMM it stands in for: the launchers of the direct-to-LDS GEMM
// (gemm_launch.h) and of the streamed GEMM (linear_stream.hip) call it after they have chosen their
// K slices, and a slice runs that kernel's MFMAs (MF = 32: 32x32x16, MF = 16: 16x16x32) over the
// same K positions in the same order; the slices are summed and finished as
// gemm_splitk_reduce_kernel does.  An output's sum does not depend on what the other rows and
// columns of a fragment hold, so a fragment may hold COLS real columns by M real rows.
//
// Bound by one memory round trip and the slice's chain of MFMAs (1280x1280, M = 2: 5.4 us, 3.3 MB of
// weights): a wave owns COLS columns of one slice, so that a layer of SD's sizes has a wave on
// most SIMDs, issues the weight loads of ten K tiles before it waits for the first, and the slices
// meet in LDS instead of in a second launch.
#include <hip/hip_runtime.h>

#include <cstdlib>

#include "gemm_core.h"

namespace mthip {

namespace {

// A workgroup is one wave per K slice (at most MAXW) over COLS output columns.  V: halves per load (8,
// or 2 where rows are only 4-byte aligned); T: 64-deep K tiles whose weight loads are in flight
// together, XT (a divisor of T): tiles whose x is.
template <int MF, int COLS, int V, int T, int XT, int MAXW, int ACT>
__global__ __launch_bounds__(64 * MAXW) void linear_rows_kernel(const GemmArgs args) {
  constexpr int KI = MF == 32 ? 16 : 32, NM = 64 / KI;  // k per MFMA, MFMAs per tile
  constexpr int NR = MF == 32 ? COLS / 2 : 4;           // accumulator registers that hold real columns
  constexpr uint32_t kOOB = 0x80000000u;                // beyond every buffer: reads zeros
  typedef float Acc __attribute__((ext_vector_type(MF == 32 ? 16 : 4)));
  __shared__ float part[MAXW][16][COLS + 4];

  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lr = lane % MF, hc = lane / MF;
  const int M = (int)args.M, K = (int)args.K_rows;
  const int64_t N = args.N, n0 = (int64_t)blockIdx.x * COLS;
  const __amdgpu_buffer_rsrc_t x_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      (void*)args.a, (short)0, (int)(((args.M - 1) * args.lda + K) * 2), 0x00020000);
  const __amdgpu_buffer_rsrc_t w_rsrc = __builtin_amdgcn_make_buffer_rsrc(
      (void*)args.b, (short)0, (int)(((N - 1) * args.ldb + K) * 2), 0x00020000);
  const uint32_t x_off = lr < M ? (uint32_t)(lr * args.lda + hc * 8) * 2u : kOOB;
  const uint32_t w_off = lr < COLS && n0 + lr < N ? (uint32_t)((n0 + lr) * args.ldb + hc * 8) * 2u : kOOB;
  const int kt0 = wave * (int)args.kt_per_split;
  const int nkt = min((int)args.kt_per_split, (int)ceil_div(args.K, 64) - kt0);

  // The 8 halves at element k of the row at byte offset off (zeros past K).
  auto load = [&](const __amdgpu_buffer_rsrc_t& r, uint32_t off, int k) -> halfx8 {
    uint4 u;
    if constexpr (V == 8) {
      const uint32_t o = k < K ? off + (uint32_t)(k - hc * 8) * 2u : kOOB;
      u = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)(off == kOOB ? kOOB : o), 0, 0));
    } else {
      uint32_t d[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t o = k + 2 * i < K ? off + (uint32_t)(k - hc * 8 + 2 * i) * 2u : kOOB;
        d[i] = __builtin_amdgcn_raw_buffer_load_b32(r, (int)(off == kOOB ? kOOB : o), 0, 0);
      }
      u = make_uint4(d[0], d[1], d[2], d[3]);
    }
    return __builtin_bit_cast(halfx8, u);
  };

  // a thread's outputs below lie in one column: its bias arrives under the products
  const uint16_t* bias = reinterpret_cast<const uint16_t*>(args.bias);
  const int64_t n = n0 + threadIdx.x % COLS;
  const uint16_t bias_h = bias && n < N ? bias[n] : 0x8000u;  // (-0 leaves every value as it is)

  Acc acc;
#pragma unroll
  for (int r = 0; r < (MF == 32 ? 16 : 4); ++r) acc[r] = 0.0f;
  for (int t0 = 0; t0 < nkt; t0 += T) {
    halfx8 w[T][NM];
    auto tile_k = [&](int t, int kk) {  // (K: zeros)
      return t0 + t < nkt ? (kt0 + t0 + t) * 64 + kk * KI + hc * 8 : K;
    };
#pragma unroll
    for (int t = 0; t < T; ++t)
#pragma unroll
      for (int kk = 0; kk < NM; ++kk) w[t][kk] = load(w_rsrc, w_off, tile_k(t, kk));
    __builtin_amdgcn_sched_barrier(0);  // every load of the trip in flight before the first is waited for
#pragma unroll
    for (int h = 0; h < T; h += XT) {
      halfx8 x[XT][NM];
#pragma unroll
      for (int t = 0; t < XT; ++t)
#pragma unroll
        for (int kk = 0; kk < NM; ++kk) x[t][kk] = load(x_rsrc, x_off, tile_k(h + t, kk));
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int t = 0; t < XT; ++t) {
        if (t0 + h + t >= nkt) break;
#pragma unroll
        for (int kk = 0; kk < NM; ++kk) {
          if constexpr (MF == 32)
            acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(w[h + t][kk], x[t][kk], acc, 0, 0, 0);
          else
            acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(w[h + t][kk], x[t][kk], acc, 0, 0, 0);
        }
      }
    }
  }
  // lane's accumulator: row lr, columns 8 (r / 4) + 4 hc + r % 4 (MF = 16: 4 hc + r)
  if (lr < M) {
#pragma unroll
    for (int r = 0; r < NR; ++r) part[wave][lr][8 * (r >> 2) + 4 * hc + (r & 3)] = acc[r];
  }
  __syncthreads();
  if (n >= N) return;
  const uint16_t* res = reinterpret_cast<const uint16_t*>(args.residual);
  uint16_t* Y = reinterpret_cast<uint16_t*>(args.c);
  const int c = threadIdx.x % COLS;
  const float b = h2f_bits(bias_h);
  for (int m = threadIdx.x / COLS; m < M; m += blockDim.x / COLS) {
    float v = part[0][m][c];
    for (int k = 1; k < (int)args.ksplit; ++k) v += part[k][m][c];
    NarrowExact narrow;
    const uint32_t h = res ? epi_chain_h<EPI_LINEAR, ACT, false, true>(v, b, 0.0f, h2f_bits(res[m * args.ld_res + n]),
                                                                      args.gelu_tab, narrow)
                           : epi_chain_h<EPI_LINEAR, ACT, false, false>(v, b, 0.0f, 0.0f, args.gelu_tab, narrow);
    Y[m * args.ldc + n] = (uint16_t)h;
  }
}

template <int MF, int COLS, int V, int T, int XT, int MAXW>
int launch(const GemmArgs& a, hipStream_t s) {
  const dim3 grid((unsigned)ceil_div(a.N, COLS)), block((unsigned)(64 * a.ksplit));
  switch (a.act) {
    case MTHIP_ACT_GELU:
      hipLaunchKernelGGL((linear_rows_kernel<MF, COLS, V, T, XT, MAXW, MTHIP_ACT_GELU>), grid, block, 0, s, a);
      break;
    case MTHIP_ACT_GELU_TANH:
      hipLaunchKernelGGL((linear_rows_kernel<MF, COLS, V, T, XT, MAXW, MTHIP_ACT_GELU_TANH>), grid, block, 0, s, a);
      break;
    case MTHIP_ACT_SILU:
      hipLaunchKernelGGL((linear_rows_kernel<MF, COLS, V, T, XT, MAXW, MTHIP_ACT_SILU>), grid, block, 0, s, a);
      break;
    default:
      hipLaunchKernelGGL((linear_rows_kernel<MF, COLS, V, T, XT, MAXW, MTHIP_ACT_NONE>), grid, block, 0, s, a);
  }
  return check_launch("linear_rows_kernel");
}

}  // namespace

// Halves per load with which the kernel takes this problem, or 0: fp16, at most 16 rows, rows and
// bases at 16-byte alignment (8) or at 4-byte alignment (2).  The size rule is where it wins at every
// row count against the GEMM with its reduction launch, weights from memory, us at M = 2 and 16 (SiLU,
// then without an activation): 320x1280 9.1 -> 4.5, 9.4 -> 4.9, 5.4 -> 4.2, 5.5 -> 4.5; 1280x1280
// 10.6 -> 5.4, 10.9 -> 6.1, 8.0 -> 4.7, 8.4 -> 5.5; 2048x2048 10.8 -> 7.4, 11.2 -> 8.5, 8.9 -> 7.0,
// 9.2 -> 8.1; 64x64 6.8 -> 3.7, 7.3 -> 4.2, 3.5 -> 3.4, 3.7 -> 3.6.  Past it (K x N) 16-byte loads of
// eight rows a wave fall behind the GEMM's tile loads: 128x8192 4.8 against 5.4 here, 320x6400 5.5
// against 5.9, 2560x1600 9.1 against 9.3 (M = 16), 4096x4096 12.1 against 18.2.
// MTHIP_GEMM_SKINNY=0 turns it off.
int linear_rows_vec(const GemmArgs& a) {
  if (a.M > 16 || a.K < 1 || a.K > 2048 || a.N > 4096 || a.N * a.K > (int64_t(1) << 22)) return 0;
  if (const char* e = std::getenv("MTHIP_GEMM_SKINNY"))
    if (e[0] == '0') return 0;
  // (operands above 2 GiB are the general path's to refuse)
  if (((a.M - 1) * a.lda + a.K) * 2 >= (int64_t(1) << 31) || ((a.N - 1) * a.ldb + a.K) * 2 >= (int64_t(1) << 31)) return 0;
  auto ok = [&](int bytes) {
    const int v = bytes / 2;
    return ((uintptr_t)a.a % bytes) == 0 && ((uintptr_t)a.b % bytes) == 0 && a.lda % v == 0 && a.ldb % v == 0 && a.K % v == 0;
  };
  return ok(16) ? 8 : ok(4) ? 2 : 0;
}

// The linear over the caller's K slices (a.ksplit of a.kt_per_split tiles) with its MFMA shape; more
// slices than the planners choose at these sizes only when a sweep forces them.
int launch_linear_rows(const GemmArgs& a, int mf, hipStream_t s) {
  if (mf == 16) return launch<16, 16, 8, 10, 5, 8>(a, s);
  if (a.ksplit <= 4) return a.rows_vec == 8 ? launch<32, 8, 8, 10, 5, 4>(a, s) : launch<32, 8, 2, 4, 2, 4>(a, s);
  return a.rows_vec == 8 ? launch<32, 8, 8, 2, 2, 16>(a, s) : launch<32, 8, 2, 2, 2, 16>(a, s);
}

}  // namespace mthip
