// seq_linear.h — product routing shared by the step functions of the sequence models (mingnative.h sections 9 and 10).
//   M <= 8 rows                      mn_skinny_gemm (weight streaming, fp32 FMA)
//   MN_SEQ_ARITH_BF16, 9 .. 64 rows  mn_skinny_gemm's weight-streaming MFMA route on bf16 hi/lo rows (fp32-class products)
//   MN_SEQ_ARITH_BF16, M > 64        mn_gemm_bf16_parts on the bf16 copy the producing kernel wrote (MFMA, fp32 accumulate; the order of K follows the row count)
//   MN_SEQ_ARITH_F32, or a K that is no multiple of 8 / an unaligned weight: mn_gemm_f32_batched (fp32 FMA; more than 2 rows, 8 where rows are not of whole 16 bytes: fp32 matrix cores)
#pragma once
#include <string.h>

#include "common.h"

namespace {

inline size_t al(size_t n) { return (n + 255) & ~(size_t)255; }

inline bool mfma_ok(const uint16_t* W, int K) { return K >= 8 && (K % 8) == 0 && (((uintptr_t)W) & 15) == 0; }

// C fp32 [M, N] = A W^T + bias.  A16 (optional) = bf16 copy of A with row stride lda16; gws / gws_bytes: scratch of the weight-streaming
// MFMA route (mn_skinny_workspace_bytes).
inline int linear(int arith, int M, const float* A, int64_t lda, const uint16_t* A16, int64_t lda16, const uint16_t* W, int N, int K,
           const uint16_t* bias, float* C, int64_t ldc, void* gws, size_t gws_bytes, void* stream) {
  // <= 8 rows: weight streaming on fp32 FMA.  9 .. 64 rows (bf16 arithmetic): the weight-streaming MFMA route on hi/lo rows — every
  // weight byte once over all CUs, where the tiled GEMM would put a 32-row problem on N / 128 workgroups
  const bool stream_mfma = arith == MN_SEQ_ARITH_BF16 && M > 8 && M <= 64 && gws && gws_bytes >= mn_skinny_workspace_bytes(M, N, K, MN_EPI_NONE);
  if ((M <= 8 || stream_mfma) && mfma_ok(W, K)) {
    mn_skinny_args a;
    memset(&a, 0, sizeof(a));
    a.x = A; a.ldx = lda; a.w = W; a.ldw = K; a.bias = bias; a.out = C; a.ldo = ldc;
    a.M = M; a.N = N; a.K = K;
    if (M > 8) { a.ws = gws; a.ws_bytes = gws_bytes; }
    return mn_skinny_gemm(&a, stream);
  }
  if (arith == MN_SEQ_ARITH_BF16 && A16 && mfma_ok(W, K) && (lda16 % 8) == 0 && (((uintptr_t)A16) & 15) == 0)
    return mn_gemm_bf16_parts(A16, lda16, W, K, bias, C, ldc, M, N, K, MN_GEMM_F32, stream);
  return mn_gemm_f32_batched(A, lda, 0, W, K, 0, bias, C, ldc, 0, nullptr, 0, 0, nullptr, 0, 0, M, N, K, 1, 1.0f, stream);
}

// Where the kernel that makes the rows A of linear()'s call may leave them as bf16 hi rows and lo rows ([2, M, K], at the start of gws) for mn_skinny_gemm_presplit to take
// up: a launch less a product (32 rows of 2048: 5.2 us).  NULL: linear() takes another route.  Nothing else may use gws in between.
inline uint16_t* linear_operand(int arith, int M, const float* A, int64_t lda, const uint16_t* W, int N, int K, const uint16_t* bias, float* C, int64_t ldc, void* gws,
                                size_t gws_bytes, mn_skinny_args* a) {
  if (arith != MN_SEQ_ARITH_BF16 || M <= 8 || M > 64 || !mfma_ok(W, K)) return nullptr;
  memset(a, 0, sizeof(*a));
  a->x = A; a->ldx = lda; a->w = W; a->ldw = K; a->bias = bias; a->out = C; a->ldo = ldc;
  a->M = M; a->N = N; a->K = K; a->ws = gws; a->ws_bytes = gws_bytes;
  return mn_skinny_operand(a);
}

// act fp32 [M, N] = gelu_tanh(A Wg^T) * (A Wu^T) with W = [Wg ; Wu] (2N rows) as the EPILOGUE of the weight-streaming product, for steps
// that take that route (<= 8 rows, or 9 .. 64 rows with scratch in the bf16 arithmetic).  *done says whether the step
// took it; if not, the caller runs the plain product and the activation launch.
inline int linear_geglu(int arith, int M, const float* A, int64_t lda, const uint16_t* W, int N, int K, float* act, int64_t ldact, void* gws,
                        size_t gws_bytes, void* stream, bool* done) {
  *done = false;
  const bool stream_mfma = arith == MN_SEQ_ARITH_BF16 && M > 8 && M <= 64 && gws && gws_bytes >= mn_skinny_workspace_bytes(M, N, K, MN_EPI_GEGLU_TANH);
  if (!((M <= 8 || stream_mfma) && mfma_ok(W, K))) return MN_OK;
  mn_skinny_args a;
  memset(&a, 0, sizeof(a));
  a.x = A; a.ldx = lda; a.w = W; a.ldw = K; a.out = act; a.ldo = ldact;
  a.M = M; a.N = N; a.K = K; a.epilogue = MN_EPI_GEGLU_TANH;
  if (M > 8) { a.ws = gws; a.ws_bytes = gws_bytes; }
  *done = true;
  return mn_skinny_gemm(&a, stream);
}

// Prompt rows (M > 64, bf16 arithmetic) whose whole-K-tile products take the LDS-DMA GEMM: is this one of them?  (C2 / C rows: quadruples of columns)
inline bool gemm_epilogue_ok(int arith, int M, const uint16_t* A16, int64_t lda16, const uint16_t* W, int64_t w_rows, int N, int K, const void* C, int64_t ldc) {
  return arith == MN_SEQ_ARITH_BF16 && M > 64 && A16 && (((uintptr_t)A16 | (uintptr_t)W) & 15) == 0 && mn_gemm256_supported(lda16, 0, K, w_rows, M, N, K) &&
         (ldc % 4) == 0 && ((uintptr_t)C & 15) == 0;
}

// C fp32 [M, N] = A W^T except its columns [t0, t1), which go squared-relu'd to C2 as bf16 [M, t1 - t0]: the hidden units' fp32 round trip (2048 x 12288:
// 200 MB, 56 us of its own launch) is not taken.  *done says whether the step took it.
inline int linear_relu2_tail(int arith, int M, const uint16_t* A16, int64_t lda16, const uint16_t* W, int N, int K, float* C, int64_t ldc, int t0, int t1,
                             uint16_t* C2, int64_t ldc2, void* stream, bool* done) {
  *done = false;
  if (!gemm_epilogue_ok(arith, M, A16, lda16, W, N, N, K, C, ldc) || (t0 % 4) != 0 || (t1 % 4) != 0 || (ldc2 % 4) != 0 || ((uintptr_t)C2 & 7) != 0) return MN_OK;
  mn_g256 a;
  memset(&a, 0, sizeof(a));
  a.A = A16; a.lda = lda16; a.W = W; a.ldw = K; a.C = C; a.ldc = ldc; a.C2 = C2; a.ldc2 = ldc2; a.tail0 = t0; a.tail1 = t1; a.M = M; a.N = N; a.K = K;
  const int rc = mn_gemm256_ex(&a, MN_G256_F32_TAIL_RELU2, 1, stream);
  *done = rc >= 0;
  return rc < 0 ? rc : MN_OK;
}

// act bf16 [M, N] = gelu_tanh(A Wg^T) * (A Wu^T), W = [Wg ; Wu], in the epilogue of the product (1409 x 2 x 4096: 16 us of a launch of its own and the
// fp32 round trip).  The caller's next product must read the bf16 rows.
inline int linear_geglu_rows(int arith, int M, const uint16_t* A16, int64_t lda16, const uint16_t* W, int N, int K, uint16_t* act, int64_t ldact,
                             void* stream, bool* done) {
  *done = false;
  if (!gemm_epilogue_ok(arith, M, A16, lda16, W, 2 * (int64_t)N, N, K, act, ldact)) return MN_OK;
  mn_g256 a;
  memset(&a, 0, sizeof(a));
  a.A = A16; a.lda = lda16; a.W = W; a.ldw = K; a.w_pair_rows = N; a.C = act; a.ldc = ldact; a.M = M; a.N = N; a.K = K;
  const int rc = mn_gemm256_ex(&a, MN_G256_GEGLU_BF16, 1, stream);
  *done = rc >= 0;
  return rc < 0 ? rc : MN_OK;
}

// Split-K slices of C fp32 [M, N] = A W^T for prompt rows whose consumer sums the slabs: 1 = one product (2048 x 2048 x 14336: 142 us in one, 93 us in four
// plus 10 us of the norm reading them)
inline int linear_slices(int arith, int M, int N, int K, int most) {
  if (arith != MN_SEQ_ARITH_BF16 || M <= 64 || (K % 64) != 0 || (N % 4) != 0 || N > 8192) return 1;
  const int ks = mn_gemm256_plan_ksplit(M, N, K, 0);
  return ks > most ? (most > 1 ? most : 1) : (ks > 1 ? ks : 1);
}
// C = that many slabs M * N apart (room for linear_slices of them); *nz says how many were written, 0: the caller's plain product serves this shape
inline int linear_slabs(int arith, int M, const uint16_t* A16, int64_t lda16, const uint16_t* W, int N, int K, int ks, float* C, void* stream, int* nz) {
  *nz = 0;
  if (ks <= 1 || !gemm_epilogue_ok(arith, M, A16, lda16, W, N, N, K, C, N)) return MN_OK;
  const int rc = mn_gemm256_splitk(A16, lda16, 0, W, K, nullptr, C, M, N, K, ks, stream);
  if (rc < 0) return rc;
  *nz = rc;
  return MN_OK;
}

// the step's own copy of its input rows (a kernel, not a memcpy node: the step may be captured into a graph)
__global__ void copy_rows_kernel(const float* __restrict__ x, int64_t ldx, float* __restrict__ y, int n) {
  const int c = blockIdx.x * 256 + threadIdx.x;
  if (c < n) y[(int64_t)blockIdx.y * n + c] = x[(int64_t)blockIdx.y * ldx + c];
}

}  // namespace
