// linear / matmul / addmm entry points: argument checks, operand staging and the choice of kernel.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdlib>

#include "gemm_core.h"

namespace mthip {

// The fp32 GEMMs (gemm_f32.hip).
int launch_linear_f32(int device, const GemmArgs& a, hipStream_t s);
int launch_geglu_f32(int device, const GemmArgs& a, hipStream_t s);
int launch_gemm_f32(int device, const GemmArgs& a, int64_t batch, bool b_trans, hipStream_t s);
int launch_conv_f32(int device, const GemmArgs& a, hipStream_t s);
// The fp16 GEMMs (gemm.hip).
int launch_linear_f16(int device, const GemmArgs& a, hipStream_t s);
int launch_geglu_f16(int device, const GemmArgs& a, hipStream_t s);
int launch_gemm_f16(int device, const GemmArgs& a, int64_t batch, bool b_trans, hipStream_t s);
// The streamed-kernel launcher for linears (linear_stream.hip); -1 where it does not apply.
int try_stream_linear(int device, const GemmArgs& a, hipStream_t s);
// How the kernel for few rows may load a linear's operands (linear_skinny.hip).
int linear_rows_vec(const GemmArgs& a);

namespace {

bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }

// dst[b][r][c] = c < cols ? src[b*sbs + r*lds + c] : 0 for c < ldd: stages an operand whose
// rows are not whole 16-byte chunks into a zero-padded, aligned copy.
template <typename T>
__global__ void pad_rows_kernel(const T* __restrict__ src, T* __restrict__ dst, int64_t rows, int64_t cols,
                                int64_t lds, int64_t sbs, int64_t ldd) {
  const int64_t b = blockIdx.y;
  const int64_t n = rows * ldd;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    const int64_t r = i / ldd, c = i - r * ldd;
    dst[b * n + i] = c < cols ? src[b * sbs + r * lds + c] : T(0);
  }
}

// Stages `rows x cols` (row stride lds, batch stride sbs, `batches` copies) into a fresh
// buffer with rows padded to `ldd` elements.  Returns 0 and the buffer (owned by the caller).
template <typename T>
int pad_operand(int device, hipStream_t s, const void* src, int64_t batches, int64_t rows, int64_t cols, int64_t lds,
                int64_t sbs, int64_t ldd, void** out) {
  if (int rc = mthip_malloc(device, (size_t)(batches * rows * ldd) * sizeof(T), out)) return rc;
  const int64_t n = rows * ldd;
  const unsigned g = (unsigned)std::min<int64_t>(std::max<int64_t>(ceil_div(n, 256), 1), 2048);
  hipLaunchKernelGGL(pad_rows_kernel<T>, dim3(g, (unsigned)batches), dim3(256), 0, s, (const T*)src, (T*)*out, rows,
                     cols, lds, sbs, ldd);
  return check_launch("pad_rows_kernel");
}

constexpr int64_t kMaxBufferBytes = (int64_t(1) << 31) - 1;
// c = narrow(beta * c_in) (0 without c_in): addmm / baddbmm at alpha = 0, where the reference
// skips the product (tensor.cpp:25320, 25621), so an inf or NaN in the operands never reaches the
// output while one in c_in does (0 * inf = NaN even at beta = 0, tensor.cpp:25256).
template <typename T>
__global__ __launch_bounds__(256) void gemm_beta_only_kernel(const GemmArgs a, int64_t batch) {
  const int64_t total = batch * a.M * a.N;
  const T* cin = reinterpret_cast<const T*>(a.c_in);
  T* c = reinterpret_cast<T*>(a.c);
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
    const int64_t col = i % a.N, t = i / a.N, row = t % a.M, bz = t / a.M;
    const float v = cin ? a.beta * Elem<T>::load(cin, bz * a.stride_c_in + row * a.c_in_rs + col * a.c_in_cs) : 0.0f;
    Elem<T>::store(c, bz * a.stride_c + row * a.ldc + col, v);
  }
}

}  // namespace
}  // namespace mthip

using namespace mthip;

extern "C" {

int mthip_linear(int device, int dtype, const void* x, int64_t lda, const void* w, int64_t ldw, const void* b,
                 void* y, int64_t ldy, int64_t M, int64_t N, int64_t K, int act, const void* residual,
                 int64_t ld_res) {
  MTHIP_REQUIRE(dtype == MTHIP_F16 || dtype == MTHIP_F32, "mthip_linear: dtype must be F16 or F32");
  MTHIP_REQUIRE(M >= 0 && N >= 0 && K >= 0, "mthip_linear: negative extent");
  MTHIP_REQUIRE(lda >= K && ldw >= K && ldy >= N, "mthip_linear: leading dimension smaller than the row");
  MTHIP_REQUIRE(act >= MTHIP_ACT_NONE && act <= MTHIP_ACT_SILU, "mthip_linear: unknown activation");
  if (M == 0 || N == 0) return MTHIP_OK;
  hipStream_t s = stream_for(device);
  if (!s) return MTHIP_ERR_HIP;
  if (int rc = use_device(device)) return rc;
  GemmArgs a{};
  a.M = M;
  a.N = N;
  a.K = K;
  a.a = x;
  a.lda = lda;
  a.b = w;
  a.ldb = ldw;
  a.c = y;
  a.ldc = ldy;
  a.bias = b;
  a.act = act;
  a.residual = residual;
  a.ld_res = ld_res;
  if (dtype == MTHIP_F16 && act == MTHIP_ACT_GELU) {
    a.gelu_tab = gelu_f16_lookup(device, s);
    if (!a.gelu_tab) return fail(MTHIP_ERR_HIP, "mthip_linear: gelu table setup failed");
  }
  const int vec = dtype == MTHIP_F16 ? 8 : 4;
  const int64_t es = dtype == MTHIP_F16 ? 2 : 4;
  // the fp32 kernel reads rows of any length and alignment in place
  const bool vec_ok =
      dtype == MTHIP_F32 || (aligned16(x) && aligned16(w) && lda % vec == 0 && ldw % vec == 0 && K % vec == 0);
  const int64_t Kp = ceil_div(K, vec) * vec;
  // Few rows: the launchers of the tile GEMM and the streamed GEMM hand the problem on.  Rows of any
  // even length are read in place where the tile GEMM would take their padded copies.
  if (dtype == MTHIP_F16) {
    a.rows_vec = linear_rows_vec(a);
    a.K_rows = K;
    // (not where the padded copies would take the streamed GEMM, or no few-row hand-over exists)
    if (a.rows_vec == 2) {
      const char* dtl = std::getenv("MTHIP_GEMM_DTL");
      if ((Kp % 320 == 0 && (act == MTHIP_ACT_NONE || act == MTHIP_ACT_GELU)) || (dtl && dtl[0] == '0')) a.rows_vec = 0;
    }
  }
  const bool in_place = vec_ok || a.rows_vec == 2;
  void* xp = nullptr;
  void* wp = nullptr;
  if (!in_place) {
    // Zero-padded aligned copies of both operands (K rounded up to a whole chunk).
    int rc = pad_operand<uint16_t>(device, s, x, 1, M, K, lda, 0, Kp, &xp);
    if (rc == MTHIP_OK) rc = pad_operand<uint16_t>(device, s, w, 1, N, K, ldw, 0, Kp, &wp);
    if (rc != MTHIP_OK) {
      mthip_free(device, xp);
      return rc;
    }
    a.a = xp;
    a.b = wp;
    a.lda = a.ldb = Kp;
  }
  if (dtype == MTHIP_F16) a.K = Kp;
  a.a_bytes = ((M - 1) * a.lda + a.K) * es;
  a.b_bytes = ((N - 1) * a.ldb + a.K) * es;
  int rc;
  if (a.a_bytes > kMaxBufferBytes || a.b_bytes > kMaxBufferBytes)
    rc = fail(MTHIP_ERR_UNSUPPORTED, "mthip_linear: operands above 2 GiB are not supported");
  else if (dtype == MTHIP_F16) {
    rc = (act == MTHIP_ACT_NONE || act == MTHIP_ACT_GELU) && a.rows_vec != 2 ? try_stream_linear(device, a, s) : -1;
    if (rc < 0) rc = launch_linear_f16(device, a, s);
  } else {
    rc = launch_linear_f32(device, a, s);
  }
  mthip_free(device, xp);  // stream-ordered: reused only by later work
  mthip_free(device, wp);
  return rc;
}

int mthip_linear_geglu(int device, int dtype, const void* x, int64_t lda, const void* w, const void* b, void* y,
                       int64_t ldy, int64_t M, int64_t N, int64_t K) {
  MTHIP_REQUIRE(dtype == MTHIP_F16 || dtype == MTHIP_F32, "mthip_linear_geglu: dtype must be F16 or F32");
  MTHIP_REQUIRE(M >= 0 && N >= 0 && K >= 0 && N % 32 == 0, "mthip_linear_geglu: N must be a multiple of 32");
  MTHIP_REQUIRE(lda >= K && ldy >= N, "mthip_linear_geglu: leading dimension smaller than the row");
  const int vec = dtype == MTHIP_F16 ? 8 : 4;
  MTHIP_REQUIRE(aligned16(x) && aligned16(w) && lda % vec == 0 && K % vec == 0,
                "mthip_linear_geglu: operands must be 16-byte aligned with K a multiple of 16 bytes");
  if (M == 0 || N == 0) return MTHIP_OK;
  hipStream_t s = stream_for(device);
  if (!s) return MTHIP_ERR_HIP;
  if (int rc = use_device(device)) return rc;
  const int64_t es = dtype == MTHIP_F16 ? 2 : 4;
  GemmArgs a{};
  a.M = M;
  a.N = 2 * N;  // interleaved value/gate columns
  a.K = K;
  a.a = x;
  a.lda = lda;
  a.b = w;
  a.ldb = K;
  a.c = y;
  a.ldc = ldy;
  a.bias = b;
  a.a_bytes = ((M - 1) * lda + K) * es;
  a.b_bytes = (2 * N * K) * es;
  MTHIP_REQUIRE(a.a_bytes <= kMaxBufferBytes && a.b_bytes <= kMaxBufferBytes,
                "mthip_linear_geglu: operands above 2 GiB are not supported");
  if (dtype == MTHIP_F16) {
    a.gelu_tab = gelu_f16_lookup(device, s);
    if (!a.gelu_tab) return fail(MTHIP_ERR_HIP, "mthip_linear_geglu: gelu table setup failed");
    return launch_geglu_f16(device, a, s);
  }
  return launch_geglu_f32(device, a, s);
}

int mthip_gemm(int device, int dtype, int64_t batch, int64_t M, int64_t N, int64_t K, const void* a_ptr, int64_t lda,
               int64_t stride_a, const void* b_ptr, int64_t ldb, int64_t stride_b, int b_trans, void* c, int64_t ldc,
               int64_t stride_c, double alpha, double beta, const void* c_in, int64_t c_in_rs, int64_t c_in_cs,
               int64_t stride_c_in) {
  MTHIP_REQUIRE(dtype == MTHIP_F16 || dtype == MTHIP_F32, "mthip_gemm: dtype must be F16 or F32");
  MTHIP_REQUIRE(batch >= 0 && M >= 0 && N >= 0 && K >= 0, "mthip_gemm: negative extent");
  if (batch == 0 || M == 0 || N == 0) return MTHIP_OK;
  hipStream_t s = stream_for(device);
  if (!s) return MTHIP_ERR_HIP;
  if (int rc = use_device(device)) return rc;
  GemmArgs a{};
  a.M = M;
  a.N = N;
  a.K = K;
  a.a = a_ptr;
  a.lda = lda;
  a.stride_a = stride_a;
  a.b = b_ptr;
  a.ldb = ldb;
  a.stride_b = stride_b;
  a.c = c;
  a.ldc = ldc;
  a.stride_c = stride_c;
  a.alpha = (float)alpha;
  a.beta = (float)beta;
  a.c_in = c_in;
  a.c_in_rs = c_in_rs;
  a.c_in_cs = c_in_cs;
  a.stride_c_in = stride_c_in;
  if (alpha == 0.0) {
    const int64_t total = batch * M * N;
    const unsigned grid = (unsigned)std::min<int64_t>(ceil_div(total, 256), 4096);
    if (dtype == MTHIP_F16)
      hipLaunchKernelGGL(gemm_beta_only_kernel<uint16_t>, dim3(grid), dim3(256), 0, s, a, batch);
    else
      hipLaunchKernelGGL(gemm_beta_only_kernel<float>, dim3(grid), dim3(256), 0, s, a, batch);
    return check_launch("gemm_beta_only_kernel");
  }
  const int vec = dtype == MTHIP_F16 ? 8 : 4;
  const int64_t es = dtype == MTHIP_F16 ? 2 : 4;
  const int64_t b_cols = b_trans ? K : N;   // contiguous extent of a B row
  const int64_t b_rows = b_trans ? N : K;
  // the fp32 kernel reads rows of any length and alignment in place
  const bool f32 = dtype == MTHIP_F32;
  bool a_ok = f32 || (aligned16(a_ptr) && lda % vec == 0 && stride_a % vec == 0 && K % vec == 0);
  bool b_ok = f32 || (aligned16(b_ptr) && ldb % vec == 0 && stride_b % vec == 0 && b_cols % vec == 0);
  void* ap = nullptr;
  void* bp = nullptr;
  int rc = MTHIP_OK;
  if (!a_ok || !b_ok) {
    // Zero-padded aligned copies; K (and, for a [K, N] B, N) rounded up to whole chunks.
    const int64_t Kp = ceil_div(K, vec) * vec;
    const int64_t a_batches = stride_a == 0 ? 1 : batch, b_batches = stride_b == 0 ? 1 : batch;
    rc = pad_operand<uint16_t>(device, s, a_ptr, a_batches, M, K, lda, stride_a, Kp, &ap);
    const int64_t bcp = ceil_div(b_cols, vec) * vec;
    if (rc == MTHIP_OK)
      rc = pad_operand<uint16_t>(device, s, b_ptr, b_batches, b_rows, b_cols, ldb, stride_b, bcp, &bp);
    if (rc == MTHIP_OK) {
      a.a = ap;
      a.lda = Kp;
      a.stride_a = stride_a == 0 ? 0 : M * Kp;
      a.b = bp;
      a.ldb = bcp;
      a.stride_b = stride_b == 0 ? 0 : b_rows * bcp;
      // K-padding of a [K, N] B adds zero rows: extend K only when both operands carry it.
      if (b_trans) a.K = Kp;
    }
  }
  if (rc == MTHIP_OK) {
    // A row is read in whole 16-byte chunks and the buffer range check drops any dword that
    // crosses a_bytes, so the extent covers the last row's final chunk (the padded copy holds
    // zeros there; unpadded rows have K a multiple of the chunk).
    // (fp32 rows end at K, and N: their last chunk may be cut by the range check.)
    a.a_bytes = ((M - 1) * a.lda + (f32 ? K : ceil_div(a.K, vec) * vec)) * es;
    // (K = 0: B has no rows, and an extent of less than nothing would let every read pass the check)
    a.b_bytes = b_trans  ? ((N - 1) * a.ldb + a.K) * es
                : K == 0 ? 0
                         : ((K - 1) * a.ldb + (f32 ? N : ceil_div(N, vec) * vec)) * es;
    if (a.a_bytes > kMaxBufferBytes || a.b_bytes > kMaxBufferBytes) {
      rc = fail(MTHIP_ERR_UNSUPPORTED, "mthip_gemm: operands above 2 GiB per batch are not supported");
    } else {
      rc = f32 ? launch_gemm_f32(device, a, batch, b_trans != 0, s) : launch_gemm_f16(device, a, batch, b_trans != 0, s);
    }
  }
  mthip_free(device, ap);
  mthip_free(device, bp);
  return rc;
}

}  // extern "C"
