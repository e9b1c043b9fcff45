// latent_ops.hip — row operators of sequence models that cache a low-rank latent instead of keys and values (mingnative.h
// section 9).  Everything here works on fp32 rows [M, n] of a step (tokens of one or several cache sequences, each sequence's
// rows consecutive) and bf16 weights; every size is an argument.
//
//   mn_affine_ln_rows        y = (x - mean) / sqrt(var + eps) * w + b                      (optional bf16 copy for an MFMA GEMM)
//   mn_gated_ln_residual     x += LN(sigmoid(g) * y) * w + b                               (gate, norm and residual add of a sublayer)
//   mn_rms_rows              y = x / sqrt(mean(x^2) + eps) * w, rows optionally scattered into a cache arena [n_seq, t_max, n]
//   mn_polynorm_rows         y = a U(z) + b U(z^2) + c U(z^3) + e,  U(v) = v / sqrt(mean(v^2) + eps)
//   mn_tap_filter_rows       y_t = x_t + sum_j w[:, j] x_(t - taps + 1 + j) over each sequence, the taps - 1 rows before a step
//                            taken from a per-sequence state, which mn_tap_state_update then advances
//   mn_gemm_f32_batched      C = alpha * A W^T (+ bias) (* sigmoid(G)), fp32 FMA / fp32 matrix cores on fp32 rows x bf16 weights, batched by strides
//                            (grid.z): the true-32-bit product and the per-head absorb / expand products of latent attention
//   mn_latent_attn           causal softmax attention of per-head absorbed queries [M, H, r] against the cached latents [t, r]
//                            (keys = values = the latent, shared by all heads), online softmax in fp32, key range splittable
//   mn_softcap_rows          z = cap * tanh(z / cap)
#include "common.h"
#include "mfma_f32_tiles.h"

namespace {

__device__ __forceinline__ float sigmoid_f(float x) { return 1.0f / (1.0f + expf(-x)); }

// ---------------------------------------------------------------------------------------------------------------------------
// one wave per row: LayerNorm with weight and bias
__global__ __launch_bounds__(256) void affine_ln_kernel(const float* __restrict__ x, int64_t ldx, const bf16_t* __restrict__ w,
                                                        const bf16_t* __restrict__ b, float eps, float* __restrict__ y, int64_t ldy,
                                                        bf16_t* __restrict__ y16, int64_t ldy16, int M, int n) {
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (row >= M) return;
  const float* xr = x + (int64_t)row * ldx;
  float s = 0.f;
  for (int i = lane; i < n; i += 64) s += xr[i];
  const float mean = wave_sum(s) / (float)n;
  float v = 0.f;
  for (int i = lane; i < n; i += 64) { const float d = xr[i] - mean; v += d * d; }
  const float rstd = 1.0f / sqrtf(wave_sum(v) / (float)n + eps);
  for (int i = lane; i < n; i += 64) {
    const float o = (xr[i] - mean) * rstd * bf16_to_f32(w[i]) + bf16_to_f32(b[i]);
    if (y) y[(int64_t)row * ldy + i] = o;
    if (y16) y16[(int64_t)row * ldy16 + i] = f32_to_bf16(o);
  }
}

// x[row] += LN(sigmoid(g[row]) * y[row]) * w + b
__global__ __launch_bounds__(256) void gated_ln_residual_kernel(float* __restrict__ x, int64_t ldx, const float* __restrict__ g,
                                                                int64_t ldg, const float* __restrict__ yv, int64_t ldy,
                                                                const bf16_t* __restrict__ w, const bf16_t* __restrict__ b, float eps,
                                                                int M, int n) {
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (row >= M) return;
  const float* gr = g + (int64_t)row * ldg;
  const float* yr = yv + (int64_t)row * ldy;
  float s = 0.f;
  for (int i = lane; i < n; i += 64) s += sigmoid_f(gr[i]) * yr[i];
  const float mean = wave_sum(s) / (float)n;
  float v = 0.f;
  for (int i = lane; i < n; i += 64) { const float d = sigmoid_f(gr[i]) * yr[i] - mean; v += d * d; }
  const float rstd = 1.0f / sqrtf(wave_sum(v) / (float)n + eps);
  for (int i = lane; i < n; i += 64) {
    const float t = sigmoid_f(gr[i]) * yr[i];
    x[(int64_t)row * ldx + i] += (t - mean) * rstd * bf16_to_f32(w[i]) + bf16_to_f32(b[i]);
  }
}

// RMS norm with a plain weight; output row index = row, or row_seq[row] * t_max + row_slot[row] (append into a cache arena)
__global__ __launch_bounds__(256) void rms_rows_kernel(const float* __restrict__ x, int64_t ldx, const bf16_t* __restrict__ w, float eps,
                                                       float* __restrict__ y, int64_t ldy, bf16_t* __restrict__ y16, int64_t ldy16,
                                                       const int32_t* __restrict__ row_seq, const int32_t* __restrict__ row_slot,
                                                       int t_max, int M, int n) {
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (row >= M) return;
  const float* xr = x + (int64_t)row * ldx;
  float s = 0.f;
  for (int i = lane; i < n; i += 64) s += xr[i] * xr[i];
  const float r = 1.0f / sqrtf(wave_sum(s) / (float)n + eps);
  const int64_t orow = row_seq ? (int64_t)row_seq[row] * t_max + row_slot[row] : row;
  for (int i = lane; i < n; i += 64) {
    const float o = xr[i] * r * bf16_to_f32(w[i]);
    if (y) y[orow * ldy + i] = o;
    if (y16) y16[(int64_t)row * ldy16 + i] = f32_to_bf16(o);
  }
}

// The same for aligned rows of up to 256 V values: the row in registers, 16 bytes a lane, requested with its weight and its destination in one batch, so
// that a row is one round trip where the loop above is one for every 64 values (32 rows of 512 or 768: 4.6 us, 7.7 before; 4.5 us is what any launch between two others takes).  Two jobs
// of the same rows are one launch (grid.y): a layer's query and key/value latents lie in one product.
struct RmsJob {
  const float* x; int64_t ldx;
  const bf16_t* w;
  float* y; int64_t ldy;
  bf16_t* y16; int64_t ldy16;
  const int32_t *row_seq, *row_slot; int t_max;
  int n;
};
struct RmsJobs { RmsJob job[2]; };

template <int V>
__global__ __launch_bounds__(256) void rms_rows_vec_kernel(RmsJobs jobs, float eps, int M) {
  const RmsJob a = jobs.job[blockIdx.y];
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63, n = a.n;
  if (row >= M) return;
  f32x4 v[V];
  ushort4 w[V];
  const int64_t orow = a.row_seq ? (int64_t)a.row_seq[row] * a.t_max + a.row_slot[row] : row;
#pragma unroll
  for (int i = 0; i < V; ++i) {
    const int c = 4 * (lane + 64 * i), cc = c < n ? c : 0;
    v[i] = *reinterpret_cast<const f32x4*>(a.x + (int64_t)row * a.ldx + cc);
    w[i] = *reinterpret_cast<const ushort4*>(a.w + cc);
  }
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < V; ++i)
    if (4 * (lane + 64 * i) < n) s += (v[i].x * v[i].x + v[i].y * v[i].y) + (v[i].z * v[i].z + v[i].w * v[i].w);
  const float r = 1.0f / sqrtf(wave_sum(s) / (float)n + eps);
#pragma unroll
  for (int i = 0; i < V; ++i) {
    const int c = 4 * (lane + 64 * i);
    if (c >= n) continue;
    const f32x4 o = {v[i].x * r * bf16_to_f32(w[i].x), v[i].y * r * bf16_to_f32(w[i].y), v[i].z * r * bf16_to_f32(w[i].z), v[i].w * r * bf16_to_f32(w[i].w)};
    if (a.y) *reinterpret_cast<f32x4*>(a.y + orow * a.ldy + c) = o;
    if (a.y16) *reinterpret_cast<ushort4*>(a.y16 + (int64_t)row * a.ldy16 + c) = ushort4{f32_to_bf16(o.x), f32_to_bf16(o.y), f32_to_bf16(o.z), f32_to_bf16(o.w)};
  }
}

// 16-byte accesses of the fp32 rows, 8-byte ones of the bf16 rows and the weight; at most 4096 values a row
bool rms_vec_ok(const RmsJob& j) {
  return (j.n % 4) == 0 && j.n <= 4096 && (j.ldx % 4) == 0 && ((uintptr_t)j.x & 15) == 0 && ((uintptr_t)j.w & 7) == 0 &&
         (!j.y || ((j.ldy % 4) == 0 && ((uintptr_t)j.y & 15) == 0)) && (!j.y16 || ((j.ldy16 % 4) == 0 && ((uintptr_t)j.y16 & 7) == 0));
}
void rms_vec_launch(const RmsJobs& jobs, int n_jobs, float eps, int M, hipStream_t st) {
  const int n = n_jobs > 1 && jobs.job[1].n > jobs.job[0].n ? jobs.job[1].n : jobs.job[0].n, v = (n + 255) / 256;
  const dim3 grid((unsigned)mn_cdiv(M, 4), (unsigned)n_jobs);
#define MN_RV(V_) hipLaunchKernelGGL((rms_rows_vec_kernel<V_>), grid, dim3(256), 0, st, jobs, eps, M)
  if (v <= 1) MN_RV(1); else if (v <= 2) MN_RV(2); else if (v <= 4) MN_RV(4); else if (v <= 8) MN_RV(8); else MN_RV(16);
#undef MN_RV
}

// one workgroup per row
__global__ __launch_bounds__(256) void polynorm_kernel(const float* __restrict__ z, int64_t ldz, const bf16_t* __restrict__ coef, float eps,
                                                       float* __restrict__ y, int64_t ldy, bf16_t* __restrict__ y16, int64_t ldy16, int n) {
  __shared__ float red[8];
  const int row = blockIdx.x;
  const float* zr = z + (int64_t)row * ldz;
  float s2 = 0.f, s4 = 0.f, s6 = 0.f;
  for (int i = threadIdx.x; i < n; i += 256) {
    const float v = zr[i], v2 = v * v, v3 = v2 * v;
    s2 += v2; s4 += v2 * v2; s6 += v3 * v3;
  }
  s2 = block_sum(s2, red); s4 = block_sum(s4, red); s6 = block_sum(s6, red);
  const float a = bf16_to_f32(coef[0]) / sqrtf(s2 / (float)n + eps), b = bf16_to_f32(coef[1]) / sqrtf(s4 / (float)n + eps),
              c = bf16_to_f32(coef[2]) / sqrtf(s6 / (float)n + eps), e = bf16_to_f32(coef[3]);
  for (int i = threadIdx.x; i < n; i += 256) {
    const float v = zr[i], v2 = v * v;
    const float o = a * v + b * v2 + c * (v2 * v) + e;
    if (y) y[(int64_t)row * ldy + i] = o;
    if (y16) y16[(int64_t)row * ldy16 + i] = f32_to_bf16(o);
  }
}

// One workgroup per row with the row held in registers (VPT values per thread, n <= 256 VPT): one batch of loads, the reductions,
// one batch of stores — the form for wide rows, where a single wave walking the row three times is a chain of dependent round trips.
enum { ROW_LN = 0, ROW_GATED_LN_RESIDUAL = 1, ROW_POLYNORM = 2 };
struct RowArgs {
  const float* x; int64_t ldx;          // LN / polynorm input; gated: the residual stream (updated in place)
  const float* g; int64_t ldg;          // gated: gate pre-activation
  const float* y; int64_t ldy;          // gated: sublayer result
  const bf16_t* w; const bf16_t* b;     // norm weight / bias; polynorm: w = the four coefficients
  float eps;
  float* out; int64_t ldo;
  bf16_t* out16; int64_t ldo16;
  int n;
  int64_t lo16;                          // polynorm: out16 as hi rows, lo rows lo16 values further (0: plain bf16)
};

template <int VPT, int MODE>
__global__ __launch_bounds__(256) void row_block_kernel(RowArgs a) {
  __shared__ float red[8];
  const int row = blockIdx.x, tid = threadIdx.x, n = a.n;
  float v[VPT];
  if (MODE == ROW_GATED_LN_RESIDUAL) {
    float gv[VPT];
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
      const int c = tid + 256 * i, cc = c < n ? c : 0;
      gv[i] = a.g[(int64_t)row * a.ldg + cc];
      v[i] = a.y[(int64_t)row * a.ldy + cc];
    }
#pragma unroll
    for (int i = 0; i < VPT; ++i) v[i] = (tid + 256 * i < n) ? sigmoid_f(gv[i]) * v[i] : 0.f;
  } else {
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
      const int c = tid + 256 * i;
      const float t = a.x[(int64_t)row * a.ldx + (c < n ? c : 0)];
      v[i] = c < n ? t : 0.f;
    }
  }
  if (MODE == ROW_POLYNORM) {
    float s2 = 0.f, s4 = 0.f, s6 = 0.f;
#pragma unroll
    for (int i = 0; i < VPT; ++i) { const float v2 = v[i] * v[i], v3 = v2 * v[i]; s2 += v2; s4 += v2 * v2; s6 += v3 * v3; }
    s2 = block_sum(s2, red); s4 = block_sum(s4, red); s6 = block_sum(s6, red);
    const float ca = bf16_to_f32(a.w[0]) / sqrtf(s2 / (float)n + a.eps), cb = bf16_to_f32(a.w[1]) / sqrtf(s4 / (float)n + a.eps),
                cc = bf16_to_f32(a.w[2]) / sqrtf(s6 / (float)n + a.eps), ce = bf16_to_f32(a.w[3]);
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
      const int c = tid + 256 * i;
      if (c >= n) continue;
      const float v2 = v[i] * v[i], o = ca * v[i] + cb * v2 + cc * (v2 * v[i]) + ce;
      if (a.out) a.out[(int64_t)row * a.ldo + c] = o;
      if (a.out16) {
        const bf16_t hi = f32_to_bf16(o);
        a.out16[(int64_t)row * a.ldo16 + c] = hi;
        if (a.lo16) a.out16[a.lo16 + (int64_t)row * a.ldo16 + c] = f32_to_bf16(o - bf16_to_f32(hi));
      }
    }
    return;
  }
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < VPT; ++i) s += v[i];
  const float mean = block_sum(s, red) / (float)n;
  float q = 0.f;
#pragma unroll
  for (int i = 0; i < VPT; ++i) { const float d = (tid + 256 * i < n) ? v[i] - mean : 0.f; q += d * d; }
  const float rstd = 1.0f / sqrtf(block_sum(q, red) / (float)n + a.eps);
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    const int c = tid + 256 * i;
    if (c >= n) continue;
    const float o = (v[i] - mean) * rstd * bf16_to_f32(a.w[c]) + bf16_to_f32(a.b[c]);
    if (MODE == ROW_GATED_LN_RESIDUAL) {
      a.out[(int64_t)row * a.ldo + c] += o;
    } else {
      if (a.out) a.out[(int64_t)row * a.ldo + c] = o;
      if (a.out16) a.out16[(int64_t)row * a.ldo16 + c] = f32_to_bf16(o);
    }
  }
}

// rows of 512 .. 8192 values take the register form; launches it and returns true, or false for other widths
template <int MODE>
bool launch_row_block(const RowArgs& a, int M, hipStream_t st) {
  if (a.n < 512 || a.n > 8192) return false;
  const int vpt = (a.n + 255) / 256;
#define MN_RB(V_) hipLaunchKernelGGL((row_block_kernel<V_, MODE>), dim3((unsigned)M), dim3(256), 0, st, a)
  if (vpt <= 2) MN_RB(2); else if (vpt <= 4) MN_RB(4); else if (vpt <= 8) MN_RB(8); else if (vpt <= 16) MN_RB(16); else MN_RB(32);
#undef MN_RB
  return true;
}

// y[m, c] = x[m, c] + sum_k w[c, taps - 1 - k] * (the sequence's input k positions back); grid (ceil(n / 256), M)
__global__ __launch_bounds__(256) void tap_filter_kernel(const float* __restrict__ x, int64_t ldx, const bf16_t* __restrict__ w, int taps,
                                                         const float* __restrict__ state, const int32_t* __restrict__ row_seq,
                                                         const int32_t* __restrict__ row_slot, const int32_t* __restrict__ row_back,
                                                         float* __restrict__ y, int64_t ldy, bf16_t* __restrict__ y16, int64_t ldy16, int n,
                                                         float self_w) {
  const int m = blockIdx.y, c = blockIdx.x * 256 + threadIdx.x;
  if (c >= n) return;
  const int seq = row_seq[m], slot = row_slot[m], back = row_back[m];
  const float cur = x[(int64_t)m * ldx + c];
  float acc = self_w * cur;                         // 1: the input is added to its filter, 0: the filter alone
  for (int k = 0; k < taps; ++k) {
    float v = 0.f;
    if (k <= back) v = x[(int64_t)(m - k) * ldx + c];
    else if (slot - k >= 0) v = state[((int64_t)seq * (taps - 1) + (k - back - 1)) * n + c];
    acc += bf16_to_f32(w[(int64_t)c * taps + (taps - 1 - k)]) * v;
  }
  if (y) y[(int64_t)m * ldy + c] = acc;
  if (y16) y16[(int64_t)m * ldy16 + c] = f32_to_bf16(acc);
}

// state[seq][i] = the sequence's input i positions before its next one; only the LAST row of a sequence in the step works
__global__ __launch_bounds__(256) void tap_state_kernel(const float* __restrict__ x, int64_t ldx, int taps, float* __restrict__ state,
                                                        const int32_t* __restrict__ row_seq, const int32_t* __restrict__ row_back, int M,
                                                        int n) {
  const int m = blockIdx.y, c = blockIdx.x * 256 + threadIdx.x;
  if (c >= n) return;
  if (m + 1 < M && row_back[m + 1] != 0) return;
  const int cnt = row_back[m] + 1;                  // rows of this sequence in the step, ending at m
  float* st = state + (int64_t)row_seq[m] * (taps - 1) * n + c;
  for (int i = taps - 2; i >= 0; --i)               // descending: the old entries that move are read before they are overwritten
    st[(int64_t)i * n] = (i < cnt) ? x[(int64_t)(m - i) * ldx + c] : st[(int64_t)(i - cnt) * n];
}

__global__ void softcap_kernel(float* __restrict__ z, int64_t ld, int n, float cap) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n) { float* p = z + (int64_t)blockIdx.y * ld + i; *p = cap * tanhf(*p / cap); }
}

// ---------------------------------------------------------------------------------------------------------------------------
// fp32 GEMM: C[z][m, n] = alpha * sum_k A[z][m, k] W[z][n, k] (+ bias[n]) (* sigmoid(G[z][m, n])).
struct GemmF32 {
  const float* A; int64_t lda, a_bs;
  const bf16_t* W; int64_t ldw, w_bs;
  const bf16_t* bias;
  float* C; int64_t ldc, c_bs;
  bf16_t* C16; int64_t ldc16, c16_bs;
  const float* G; int64_t ldg, g_bs;
  int M, N, K;
  float alpha;
};

__device__ __forceinline__ void f32_store(const GemmF32& a, int z, int m, int n, float v) {
  if (m >= a.M || n >= a.N) return;
  v *= a.alpha;
  if (a.bias) v += bf16_to_f32(a.bias[n]);
  if (a.G) v *= sigmoid_f(a.G[(int64_t)z * a.g_bs + (int64_t)m * a.ldg + n]);
  if (a.C) a.C[(int64_t)z * a.c_bs + (int64_t)m * a.ldc + n] = v;
  if (a.C16) a.C16[(int64_t)z * a.c16_bs + (int64_t)m * a.ldc16 + n] = f32_to_bf16(v);
}

// outputs n .. n + 3 of row m
__device__ __forceinline__ void f32_store4(const GemmF32& a, int z, int m, int n, f32x4 v) {
  float* c = a.C ? a.C + (int64_t)z * a.c_bs + (int64_t)m * a.ldc + n : nullptr;
  if (n + 4 > a.N || !c || a.C16 || a.G) {
#pragma unroll
    for (int e = 0; e < 4; ++e) f32_store(a, z, m, n + e, v[e]);
    return;
  }
  v *= a.alpha;
  if (a.bias) {
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] += bf16_to_f32(a.bias[n + e]);
  }
  *reinterpret_cast<f32x4u*>(c) = v;                          // (rows may start at any float)
}

// More than 2 rows (8 where accesses go value by value) run on the matrix cores, fp32 rows and bf16 weights: few tiles on the fp32 ones (v_mfma_f32_16x16x4f32: lane l holds row / column l & 15,
// weights widened on the way; lane l takes the values 4 (l >> 4) .. + 3 of every 16 of K, so the four products of a 16-step take one 16-byte read of each operand), many on the bf16 ones.
// Values past K enter as zeros.  V4: rows of A are 16-byte, rows of W 8-byte aligned; else value by value.

// Few tiles: 32 x 16 outputs a workgroup, whose four waves split K; operands straight from memory, the next 32 values in flight during
// the products.  Latency bounds it (32 rows x 16 heads of 512 x 128: 5 us here, 45 us as one wave a column and 8 rows).  A block of 32
// values is summed as a tree of single products and added to the running sum with its rounding error kept (two-sum), so the
// result is as close to the exact sum as the tree over 64 lanes that one or two rows take (0.22e-7 and 0.46e-7 of the summed magnitudes at K 512).
template <bool V4>
__global__ __launch_bounds__(256) void gemm_f32_few_kernel(GemmF32 a) {
  __shared__ float red[4][16][64];
  const int z = blockIdx.z, wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 15, q = lane >> 4;
  const int m0 = blockIdx.y * 32, n0 = blockIdx.x * 16;
  const int per = ((a.K + 63) / 64) * 16, kb = wave * per, ke = min(a.K, kb + per);
  const float* ap[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) ap[i] = a.A + (int64_t)z * a.a_bs + (int64_t)min(m0 + 16 * i + r, a.M - 1) * a.lda;
  const bf16_t* wp = a.W + (int64_t)z * a.w_bs + (int64_t)min(n0 + r, a.N - 1) * a.ldw;
  f32x4 fa[2][2];
  ushort4 fw[2];
  float sum[8], low[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) sum[e] = low[e] = 0.f;
  auto fetch = [&](int k0) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int k = k0 + 16 * u + 4 * q;
      fw[u] = ushort4{0, 0, 0, 0};
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        fa[u][i] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (V4) { if (k < ke) fa[u][i] = *reinterpret_cast<const f32x4*>(ap[i] + k); }
        else
#pragma unroll
          for (int t = 0; t < 4; ++t) if (k + t < ke) fa[u][i][t] = ap[i][k + t];
      }
      if (V4) { if (k < ke) fw[u] = *reinterpret_cast<const ushort4*>(wp + k); }
      else {
        if (k < ke) fw[u].x = wp[k];
        if (k + 1 < ke) fw[u].y = wp[k + 1];
        if (k + 2 < ke) fw[u].z = wp[k + 2];
        if (k + 3 < ke) fw[u].w = wp[k + 3];
      }
    }
  };
  if (kb < ke) fetch(kb);
  for (int k0 = kb; k0 < ke; k0 += 32) {
    f32x4 ca[2][2], cw[2], p[2][4][2];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      ca[u][0] = fa[u][0]; ca[u][1] = fa[u][1];
      cw[u] = f32x4{bf16_to_f32(fw[u].x), bf16_to_f32(fw[u].y), bf16_to_f32(fw[u].z), bf16_to_f32(fw[u].w)};
    }
    if (k0 + 32 < ke) fetch(k0 + 32);
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int i = 0; i < 2; ++i) p[u][t][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(ca[u][i][t], cw[u][t], f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int i = e >> 2, c = e & 3;
      const float v = ((p[0][0][i][c] + p[0][1][i][c]) + (p[0][2][i][c] + p[0][3][i][c])) + ((p[1][0][i][c] + p[1][1][i][c]) + (p[1][2][i][c] + p[1][3][i][c]));
      two_sum(sum[e], low[e], v);
    }
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) { red[wave][e][lane] = sum[e]; red[wave][8 + e][lane] = low[e]; }
  __syncthreads();
#pragma unroll
  for (int t = 0; t < 2; ++t) {                               // the four waves deal the tile's values among themselves
    const int e = 2 * wave + t;
    float s = red[0][e][lane], l = red[0][8 + e][lane];
#pragma unroll
    for (int w = 1; w < 4; ++w) {
      l += red[w][8 + e][lane];
      two_sum(s, l, red[w][e][lane]);
    }
    f32_store(a, z, m0 + 16 * (e >> 2) + 4 * q + (e & 3), n0 + r, s + l == s + l ? s + l : s);   // a sum at infinity has no error term
  }
}

// Many tiles: 64 x 64 outputs a workgroup, 32 x 32 a wave, on the bf16 matrix cores.  An fp32 value is the sum of three bf16 values, its upper, middle and lower 8 bits of mantissa cut off one
// after the other, and a weight is one already: three products a pair, each exact in fp32, take a fifth of the fp32 cores' time for the one.  The rows are split once a workgroup, on their way to
// LDS (7 instructions a value); 64 values of K at a time, rows 144 bytes apart (the 16-byte reads of 16 rows meet all 64 banks), two stages of loads in flight in registers.  The upper products
// and the others have accumulators of their own.  The middle and lower parts enter times 2^24, exact down to the smallest value (as they are, rows below 2^-110 lost their last bits: 2.5e-7 at
// 2^-112, 7e-5 at 2^-120).  Values from 2^112 on overflow there and of an infinite one nothing but NaN is left: an output whose lower parts have no finite sum, while the upper ones do not say
// NaN, is taken over again value by value, and so are all of a workgroup that saw an infinite weight, which would meet a part that is zero.
// NB: buffers of LDS: two (two workgroups a CU), or one and a second barrier (three a CU) where the tiles are more than two a CU: us, two / one: 900 rows of
// 16 x 512 x 128 24.4 / 21.3, 2048 x 4096 x 1024 100 / 94, 8 x 2129 x 1676 x 302 241 / 216; 900 of 1024 x 1024 (240 tiles) 19.7 / 20.6.
// us, fp32 matrix cores (values a lane stored one by one) -> here: 900 rows of 16 x 512 x 128 32 -> 21.5, of 16 x 128 x 512 28 -> 17, 1900 rows 53 -> 35 and 49 -> 30, 2048 x 4096 x 1024 168 -> 87 (197
// TFLOP/s), 200 rows of 16 x 128 x 512 17.5 -> 11.2.  What bounds short K is a workgroup's round trips.  Error against 64 bits, rows of uneven magnitudes: 1.47e-7 -> 0.77e-7 at K = 128, 2.9e-7 -> 1.5e-7 at 512, 5.7e-7 ->
// 2.9e-7 at 2048.
template <bool V4, int NB>
__global__ __launch_bounds__(256, NB == 1 ? 3 : 2) void gemm_f32_tile_kernel(GemmF32 a) {
  typedef short bf16x8 __attribute__((ext_vector_type(8)));
  typedef unsigned short us2 __attribute__((ext_vector_type(2)));
  constexpr int LD = 72, PLANE = 64 * LD;
  constexpr float LOW = 0x1p24f;
  __shared__ __attribute__((aligned(16))) uint16_t lds[NB][4 * PLANE];      // [upper | middle | lower | weights][64][LD]
  const int z = blockIdx.z, tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, r = lane & 15, q = lane >> 4;
  const int m0 = blockIdx.y * 64, n0 = blockIdx.x * 64, wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
  const float* A = a.A + (int64_t)z * a.a_bs;
  const bf16_t* W = a.W + (int64_t)z * a.w_bs;
  const int k4 = 4 * (tid & 15);
  const float* ap[4];
  const bf16_t* wp[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) {                               // rows past the matrix repeat its last one; nothing of them is stored
    const int row = (tid >> 4) + 16 * t;
    ap[t] = A + (int64_t)min(m0 + row, a.M - 1) * a.lda;
    wp[t] = W + (int64_t)min(n0 + row, a.N - 1) * a.ldw;
  }
  f32x4 fa[2][4];
  ushort4 fw[2][4];
  us2 top = {0, 0};                                           // the weights' largest magnitudes, as bits
  auto fetch = [&](int k0, int h) {
    const int k = k0 + k4;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      if (V4) {
        const int kc = min(k, a.K - 4);
        fa[h][t] = *reinterpret_cast<const f32x4*>(ap[t] + kc);
        fw[h][t] = *reinterpret_cast<const ushort4*>(wp[t] + kc);
      } else {
#pragma unroll
        for (int c = 0; c < 4; ++c) fa[h][t][c] = ap[t][min(k + c, a.K - 1)];
        fw[h][t] = ushort4{wp[t][min(k, a.K - 1)], wp[t][min(k + 1, a.K - 1)], wp[t][min(k + 2, a.K - 1)], wp[t][min(k + 3, a.K - 1)]};
      }
    }
  };
  auto put = [&](int b, int k0, int h) {
    const int left = a.K - k0 - k4;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      uint32_t part[3][4], w01 = fw[h][t].x | (uint32_t)fw[h][t].y << 16, w23 = fw[h][t].z | (uint32_t)fw[h][t].w << 16;
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const float v = c < left ? fa[h][t][c] : 0.f;         // what is past K becomes zero here: a branch around the load is a wait
        const float u = __uint_as_float(__float_as_uint(v) & 0xffff0000u), d = (v - u) * LOW;
        const float m = __uint_as_float(__float_as_uint(d) & 0xffff0000u);
        part[0][c] = __float_as_uint(v);
        part[1][c] = __float_as_uint(d);
        part[2][c] = __float_as_uint(d - m);
      }
      if (left < 4) {
        w01 &= left > 1 ? 0xffffffffu : left > 0 ? 0xffffu : 0u;
        w23 &= left > 3 ? 0xffffffffu : left > 2 ? 0xffffu : 0u;
      }
      const uint32_t b01 = w01 & 0x7fff7fffu, b23 = w23 & 0x7fff7fffu;
      top = __builtin_elementwise_max(top, __builtin_elementwise_max(*reinterpret_cast<const us2*>(&b01), *reinterpret_cast<const us2*>(&b23)));
      uint16_t* at = &lds[b % NB][((tid >> 4) + 16 * t) * LD + k4];
#pragma unroll
      for (int x = 0; x < 3; ++x)
        *reinterpret_cast<uint2*>(at + x * PLANE) = uint2{__builtin_amdgcn_perm(part[x][1], part[x][0], 0x07060302u), __builtin_amdgcn_perm(part[x][3], part[x][2], 0x07060302u)};
      *reinterpret_cast<uint2*>(at + 3 * PLANE) = uint2{w01, w23};
    }
  };
  f32x4 acc[2][2][2];
#pragma unroll
  for (int u = 0; u < 2; ++u)
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) acc[u][i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto step = [&](int k0, int b) {                            // buffer b holds K-step k0, registers b ^ 1 the one after it
    if (k0 + 128 < a.K) fetch(k0 + 128, b);
    lds_barrier();
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      bf16x8 fr[3][2], wr[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        wr[i] = *reinterpret_cast<const bf16x8*>(&lds[b % NB][3 * PLANE + (wn + 16 * i + r) * LD + 32 * u + 8 * q]);
#pragma unroll
        for (int x = 0; x < 3; ++x) fr[x][i] = *reinterpret_cast<const bf16x8*>(&lds[b % NB][x * PLANE + (wm + 16 * i + r) * LD + 32 * u + 8 * q]);
      }
#pragma unroll
      for (int x = 2; x >= 0; --x)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j) acc[x == 0][i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wr[j], fr[x][i], acc[x == 0][i][j], 0, 0, 0);
    }
    if (k0 + 64 < a.K) {
      if (NB == 1) lds_barrier();
      put(b ^ 1, k0 + 64, b ^ 1);                             // NB 2: the buffer that every wave left before this step's barrier
    }
  };
  fetch(0, 0);
  if (64 < a.K) fetch(64, 1);
  put(0, 0, 0);
  for (int k0 = 0; k0 < a.K; k0 += 128) {
    step(k0, 0);
    if (k0 + 64 < a.K) step(k0 + 64, 1);
  }
  const bool odd = __syncthreads_or(top.x >= 0x7f80 || top.y >= 0x7f80);
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) {                             // a lane's four outputs are neighbours in a row
      const int m = m0 + wm + 16 * i + r, n = n0 + wn + 16 * j + 4 * q;
      const f32x4 up = acc[1][i][j], low = acc[0][i][j];
      f32x4 v = up + low * (1.0f / LOW);
      const f32x4 lost = low * 0.f;                           // zero, or NaN
      if (odd || (lost[0] + lost[1]) + (lost[2] + lost[3]) != 0.f) {
        const float* x = A + (int64_t)min(m, a.M - 1) * a.lda;
#pragma unroll 1
        for (int e = 0; e < 4; ++e) {
          const float ue = e == 0 ? up[0] : e == 1 ? up[1] : e == 2 ? up[2] : up[3], le = e == 0 ? lost[0] : e == 1 ? lost[1] : e == 2 ? lost[2] : lost[3];
          if (!odd && (le == 0.f || ue != ue)) continue;
          const bf16_t* w = W + (int64_t)min(n + e, a.N - 1) * a.ldw;
          float t[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
          for (int k = 0; k < a.K; k += 8)
#pragma unroll
            for (int c = 0; c < 8; ++c)
              if (k + c < a.K) t[c] = fmaf(x[k + c], bf16_to_f32(w[k + c]), t[c]);
          const float r = ((t[0] + t[1]) + (t[2] + t[3])) + ((t[4] + t[5]) + (t[6] + t[7]));
          v = f32x4{e == 0 ? r : v[0], e == 1 ? r : v[1], e == 2 ? r : v[2], e == 3 ? r : v[3]};
        }
      }
      if (m < a.M) f32_store4(a, z, m, n, v);
    }
}

// Decode rows (every row alone in its sequence), one workgroup per row, the row in registers, up to three stages in one launch:
//   1 (g given)  x += LN(sigmoid(g) * y; wa, ba)          the previous sublayer's gate, norm and residual add
//   2            n  = LN(x; wb, bb)                        this sublayer's input norm
//   3 (h given)  h  = n + taps filter over the sequence's last inputs (from its state), and the state moves on by this row
struct FusedRowArgs {
  float* x; int64_t ldx;
  const float* g; int64_t ldg;
  const float* y; int64_t ldy;
  const bf16_t *wa, *ba, *wb, *bb;
  float eps;
  float* n_out; int64_t ldn;
  const bf16_t* taps_w; int taps;
  float* state; const int32_t* row_seq; const int32_t* row_slot;
  float* h; int64_t ldh;
  int n;
  bf16_t* y16; int64_t y_lo;             // optional: the last of the outputs (h, or n_out without a filter) as dense bf16 hi rows, lo rows y_lo values further
};
__device__ __forceinline__ void store_hilo(bf16_t* y, int64_t lo, float v) {
  const bf16_t hi = f32_to_bf16(v);
  y[0] = hi;
  y[lo] = f32_to_bf16(v - bf16_to_f32(hi));
}

constexpr int FUSED_MAX_TAPS = 8;

template <int VPT, bool FILTER>
__global__ __launch_bounds__(256) void row_fused_kernel(FusedRowArgs a) {
  __shared__ float red[8];
  const int row = blockIdx.x, tid = threadIdx.x, n = a.n;
  float xv[VPT];
  // everything the row needs from memory is requested before the first store: the state is float like the outputs, so a load
  // placed after a store would wait its turn, one round trip per value
  float sv[FILTER ? VPT : 1][FUSED_MAX_TAPS - 1];
  const int seq = FILTER ? a.row_seq[row] : 0, slot = FILTER ? a.row_slot[row] : 0;
  float* const st0 = FILTER ? a.state + (int64_t)seq * (a.taps - 1) * n : nullptr;
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    const int c = tid + 256 * i, cc = c < n ? c : 0;
    const float t = a.x[(int64_t)row * a.ldx + cc];
    xv[i] = c < n ? t : 0.f;
    if (FILTER) {
#pragma unroll
      for (int k = 1; k < FUSED_MAX_TAPS; ++k) sv[i][k - 1] = (k < a.taps) ? st0[(int64_t)(k - 1) * n + cc] : 0.f;
    }
  }
  if (a.g) {
    float t[VPT];
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
      const int c = tid + 256 * i, cc = c < n ? c : 0;
      const float gv = a.g[(int64_t)row * a.ldg + cc], yv = a.y[(int64_t)row * a.ldy + cc];
      t[i] = c < n ? sigmoid_f(gv) * yv : 0.f;
    }
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < VPT; ++i) s += t[i];
    const float mean = block_sum(s, red) / (float)n;
    float q = 0.f;
#pragma unroll
    for (int i = 0; i < VPT; ++i) { const float d = (tid + 256 * i < n) ? t[i] - mean : 0.f; q += d * d; }
    const float rstd = 1.0f / sqrtf(block_sum(q, red) / (float)n + a.eps);
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
      const int c = tid + 256 * i;
      if (c >= n) continue;
      xv[i] += (t[i] - mean) * rstd * bf16_to_f32(a.wa[c]) + bf16_to_f32(a.ba[c]);
      a.x[(int64_t)row * a.ldx + c] = xv[i];
    }
  }
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < VPT; ++i) s += xv[i];
  const float mean = block_sum(s, red) / (float)n;
  float q = 0.f;
#pragma unroll
  for (int i = 0; i < VPT; ++i) { const float d = (tid + 256 * i < n) ? xv[i] - mean : 0.f; q += d * d; }
  const float rstd = 1.0f / sqrtf(block_sum(q, red) / (float)n + a.eps);
#pragma unroll
  for (int i = 0; i < VPT; ++i) {
    const int c = tid + 256 * i;
    if (c >= n) continue;
    const float nv = (xv[i] - mean) * rstd * bf16_to_f32(a.wb[c]) + bf16_to_f32(a.bb[c]);
    a.n_out[(int64_t)row * a.ldn + c] = nv;
    if (!FILTER && a.y16) store_hilo(a.y16 + (int64_t)row * n + c, a.y_lo, nv);
    if (FILTER) {
      const bf16_t* tw = a.taps_w + (int64_t)c * a.taps;
      float acc = nv + bf16_to_f32(tw[a.taps - 1]) * nv;
#pragma unroll
      for (int k = 1; k < FUSED_MAX_TAPS; ++k)
        if (k < a.taps && slot - k >= 0) acc += bf16_to_f32(tw[a.taps - 1 - k]) * sv[i][k - 1];
      a.h[(int64_t)row * a.ldh + c] = acc;
      if (a.y16) store_hilo(a.y16 + (int64_t)row * n + c, a.y_lo, acc);
      float* st = st0 + c;
#pragma unroll
      for (int k = FUSED_MAX_TAPS - 2; k >= 1; --k)
        if (k < a.taps - 1) st[(int64_t)k * n] = sv[i][k - 1];
      if (a.taps > 1) st[0] = nv;
    }
  }
}

// The same for aligned rows: 4 consecutive values a thread, n / 4 threads, and everything the row and its norms need from memory requested in one
// batch of 16- and 8-byte loads.  A row is then one round trip and four sums over the workgroup; above, the weights of either norm and the filter's
// taps each wait behind the sums before them (32 rows of 2048 with three tap rows: 5.3 us, 16.0 there; without the filter 4.8, 11.7).  TAPS 0: no filter.
template <int TAPS>
__global__ __launch_bounds__(1024) void row_fused_vec_kernel(FusedRowArgs a) {
  __shared__ float red[16];
  const int row = blockIdx.x, n = a.n, c = 4 * threadIdx.x;
  const bool on = c < n;
  const int cc = on ? c : 0;
  auto row4 = [&](const float* p, int64_t ld) { return *reinterpret_cast<const f32x4*>(p + (int64_t)row * ld + cc); };
  auto par4 = [&](const bf16_t* p) { return *reinterpret_cast<const ushort4*>(p + cc); };
  auto wide = [](ushort4 v) { return f32x4{bf16_to_f32(v.x), bf16_to_f32(v.y), bf16_to_f32(v.z), bf16_to_f32(v.w)}; };
  constexpr int TS = TAPS > 1 ? TAPS - 1 : 1, TW = TAPS > 0 ? TAPS : 1;
  f32x4 sv[TS];
  ushort4 tw[TW];                                      // taps of 4 columns: value j * TAPS + t
  int slot = 0;
  float* st0 = nullptr;
  if (TAPS > 0) {
    slot = a.row_slot[row];
    if (TAPS > 1) {
      st0 = a.state + (int64_t)a.row_seq[row] * (TAPS - 1) * n + cc;
#pragma unroll
      for (int k = 0; k < TAPS - 1; ++k) sv[k] = *reinterpret_cast<const f32x4*>(st0 + (int64_t)k * n);
    }
#pragma unroll
    for (int k = 0; k < TAPS; ++k) tw[k] = *reinterpret_cast<const ushort4*>(a.taps_w + (int64_t)cc * TAPS + 4 * k);
  }
  f32x4 x = row4(a.x, a.ldx);
  const ushort4 wb = par4(a.wb), bb = par4(a.bb);
  auto norm = [&](const f32x4& v, ushort4 w, ushort4 b) {
    const float mean = block_sum(on ? (v.x + v.y) + (v.z + v.w) : 0.f, red) / (float)n;
    const f32x4 d = v - mean;
    const float q = block_sum(on ? (d.x * d.x + d.y * d.y) + (d.z * d.z + d.w * d.w) : 0.f, red);
    return d * (1.0f / sqrtf(q / (float)n + a.eps)) * wide(w) + wide(b);
  };
  if (a.g) {
    const f32x4 g = row4(a.g, a.ldg);
    f32x4 y = row4(a.y, a.ldy);
    const ushort4 wa = par4(a.wa), ba = par4(a.ba);
    y = f32x4{sigmoid_f(g.x) * y.x, sigmoid_f(g.y) * y.y, sigmoid_f(g.z) * y.z, sigmoid_f(g.w) * y.w};
    x += norm(y, wa, ba);
    if (on) *reinterpret_cast<f32x4*>(a.x + (int64_t)row * a.ldx + c) = x;
  }
  const f32x4 nv = norm(x, wb, bb);
  if (!on) return;
  auto split = [&](const f32x4& v) {
    ushort4 hi = {f32_to_bf16(v.x), f32_to_bf16(v.y), f32_to_bf16(v.z), f32_to_bf16(v.w)};
    const f32x4 r = v - wide(hi);
    bf16_t* y = a.y16 + (int64_t)row * n + c;
    *reinterpret_cast<ushort4*>(y) = hi;
    *reinterpret_cast<ushort4*>(y + a.y_lo) = ushort4{f32_to_bf16(r.x), f32_to_bf16(r.y), f32_to_bf16(r.z), f32_to_bf16(r.w)};
  };
  *reinterpret_cast<f32x4*>(a.n_out + (int64_t)row * a.ldn + c) = nv;
  if (TAPS == 0 && a.y16) split(nv);
  if (TAPS > 0) {
    float t[4 * TW];
#pragma unroll
    for (int k = 0; k < TW; ++k) { t[4 * k] = bf16_to_f32(tw[k].x); t[4 * k + 1] = bf16_to_f32(tw[k].y); t[4 * k + 2] = bf16_to_f32(tw[k].z); t[4 * k + 3] = bf16_to_f32(tw[k].w); }
    f32x4 h;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      h[j] = nv[j] + t[j * TW + TW - 1] * nv[j];
#pragma unroll
      for (int k = 1; k < TAPS; ++k)
        if (slot - k >= 0) h[j] += t[j * TW + TW - 1 - k] * sv[k - 1][j];
    }
    *reinterpret_cast<f32x4*>(a.h + (int64_t)row * a.ldh + c) = h;
    if (a.y16) split(h);
#pragma unroll
    for (int k = TAPS - 2; k >= 1; --k) *reinterpret_cast<f32x4*>(st0 + (int64_t)k * n) = sv[k - 1];
    if (TAPS > 1) *reinterpret_cast<f32x4*>(st0) = nv;
  }
}

// the vector form's accesses: 16 bytes of fp32 rows, 8 bytes of bf16 parameters
bool row_fused_vec_ok(const FusedRowArgs& a) {
  auto f = [](const float* p, int64_t ld) { return !p || (((uintptr_t)p & 15) == 0 && (ld % 4) == 0); };
  auto h = [](const bf16_t* p) { return ((uintptr_t)p & 7) == 0; };
  return (a.n % 4) == 0 && f(a.x, a.ldx) && f(a.g, a.ldg) && f(a.y, a.ldy) && f(a.n_out, a.ldn) && f(a.h, a.ldh) && f(a.state, 0) && h(a.wa) && h(a.ba) && h(a.wb) &&
         h(a.bb) && h(a.taps_w) && h(a.y16) && (a.y_lo % 4) == 0;
}

// C[z][m, n] = alpha * A[z][m, :] . W[z][n, :] (+ bias) (* sigmoid(G)) for at most MM rows: one wave per output column, lanes over K
template <int MM>
__global__ __launch_bounds__(256) void gemv_f32_kernel(GemmF32 a) {
  const int z = blockIdx.z, n = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (n >= a.N) return;
  const float* A = a.A + (int64_t)z * a.a_bs;
  const bf16_t* Wr = a.W + (int64_t)z * a.w_bs + (int64_t)n * a.ldw;
  float acc[MM];
#pragma unroll
  for (int m = 0; m < MM; ++m) acc[m] = 0.f;
#pragma unroll 4
  for (int k = lane; k < a.K; k += 64) {
    const float w = bf16_to_f32(Wr[k]);
#pragma unroll
    for (int m = 0; m < MM; ++m)
      if (m < a.M) acc[m] = fmaf(A[(int64_t)m * a.lda + k], w, acc[m]);
  }
#pragma unroll
  for (int m = 0; m < MM; ++m) {
    if (m >= a.M) break;
    float v = wave_sum(acc[m]) * a.alpha;
    if (lane != 0) continue;
    if (a.bias) v += bf16_to_f32(a.bias[n]);
    if (a.G) v *= sigmoid_f(a.G[(int64_t)z * a.g_bs + (int64_t)m * a.ldg + n]);
    if (a.C) a.C[(int64_t)z * a.c_bs + (int64_t)m * a.ldc + n] = v;
    if (a.C16) a.C16[(int64_t)z * a.c16_bs + (int64_t)m * a.ldc16 + n] = f32_to_bf16(v);
  }
}

// ---------------------------------------------------------------------------------------------------------------------------
// Latent attention.  One wave per query vector (row, head); the waves of a workgroup share the staged latent tile (all heads and up
// to 4 consecutive rows of one sequence see the same keys).  Phase A: lane = key, dot over r; phase B: lane = latent component,
// sum over keys.  Running maximum / sum / accumulator in fp32 registers.
template <int RCH>
__global__ __launch_bounds__(1024) void latent_attn_kernel(const float* __restrict__ qabs, const float* __restrict__ arena,
                                                           const int32_t* __restrict__ row_seq, const int32_t* __restrict__ row_len,
                                                           const int32_t* __restrict__ blk_tab, int H, int r, int t_max, int KT,
                                                           int tiles_per_split, float* __restrict__ lat, float* __restrict__ part_acc,
                                                           float* __restrict__ part_ml, int KS, int M) {
  extern __shared__ float lds_c[];                 // [KT][r + 1]
  const int row0 = blk_tab[2 * blockIdx.x], nrows = blk_tab[2 * blockIdx.x + 1];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, NW = blockDim.x >> 6;
  const int qv = blockIdx.y * NW + wave;
  const bool active = qv < nrows * H;
  const int ri = active ? qv / H : 0, h = active ? qv % H : 0, m = row0 + ri;
  const int64_t seq = row_seq[row0];
  const int len_max = row_len[row0 + nrows - 1];
  const int my_len = active ? row_len[m] : 0;
  float q[RCH], acc[RCH];
#pragma unroll
  for (int i = 0; i < RCH; ++i) {
    const int d = lane + 64 * i;
    q[i] = (active && d < r) ? qabs[((int64_t)m * H + h) * r + d] : 0.f;
    acc[i] = 0.f;
  }
  float mrun = -INFINITY, l = 0.f;
  const int n_tiles = (len_max + KT - 1) / KT;
  const int t0 = blockIdx.z * tiles_per_split, t1 = min(t0 + tiles_per_split, n_tiles);
  const int ldc = r + 1;
  for (int tile = t0; tile < t1; ++tile) {
    const int key0 = tile * KT;
    __syncthreads();
    for (int j = wave; j < KT; j += NW) {            // a wave copies whole latent rows: consecutive lanes, consecutive components
      const bool in = key0 + j < len_max;
      const float* src = arena + (seq * t_max + key0 + j) * r;
      for (int d = lane; d < r; d += 64) lds_c[j * ldc + d] = in ? src[d] : 0.f;
    }
    __syncthreads();
    if (!active || key0 >= my_len) continue;
    // every lane runs the dot product (lanes beyond the tile or the row's length on a clamped key, masked afterwards): the
    // cross-lane reads of q below then never sit in divergent control flow
    float dot = 0.f;
    {
      const float* cj = lds_c + min(lane, KT - 1) * ldc;
#pragma unroll
      for (int i = 0; i < RCH; ++i) {
        const int dn = min(64, r - 64 * i);
        for (int dd = 0; dd < dn; ++dd) dot = fmaf(lane_f(q[i], dd), cj[64 * i + dd], dot);
      }
    }
    const float s = (lane < KT && key0 + lane < my_len) ? dot : -INFINITY;
    const float mnew = fmaxf(mrun, wave_max(s));       // finite: key0 < my_len
    const float p = (s == -INFINITY) ? 0.f : expf(s - mnew);
    const float corr = (mrun == -INFINITY) ? 0.f : expf(mrun - mnew);
    l = l * corr + wave_sum(p);
#pragma unroll
    for (int i = 0; i < RCH; ++i) acc[i] *= corr;
    const int jn = min(KT, my_len - key0);
    for (int j = 0; j < jn; ++j) {
      const float pj = lane_f(p, j);
#pragma unroll
      for (int i = 0; i < RCH; ++i) {
        const int d = lane + 64 * i;
        if (d < r) acc[i] = fmaf(pj, lds_c[j * ldc + d], acc[i]);
      }
    }
    mrun = mnew;
  }
  if (!active) return;
  const int64_t o = ((int64_t)m * H + h);
  if (KS == 1) {
    const float inv = 1.0f / l;
#pragma unroll
    for (int i = 0; i < RCH; ++i) {
      const int d = lane + 64 * i;
      if (d < r) lat[o * r + d] = acc[i] * inv;
    }
  } else {
    const int64_t po = (int64_t)blockIdx.z * M * H + o;
#pragma unroll
    for (int i = 0; i < RCH; ++i) {
      const int d = lane + 64 * i;
      if (d < r) part_acc[po * r + d] = acc[i];
    }
    if (lane == 0) { part_ml[po * 2] = mrun; part_ml[po * 2 + 1] = l; }
  }
}

// ---------------------------------------------------------------------------------------------------------------------------
// Latent attention on the fp32 matrix cores (v_mfma_f32_16x16x4_f32: fp32 operands, fp32 accumulate — scores and weights stay
// 32-bit).  A workgroup of 4 waves owns 16 query vectors (row, head) of one run of rows and walks its share of the sequence's latents
// (LatentWalk, mfma_f32_tiles.h).
// For few keys a workgroup and for latents of any size; long walks over latents of 128, 256, 384 or 512 are the form below's.
struct PlainScore { __device__ __forceinline__ float operator()(float s) const { return s; } };
template <int NB, int KF, bool VEC>
__global__ __launch_bounds__(256, VEC && NB <= 8 ? 2 : 1) void latent_attn_mfma_kernel(const float* __restrict__ qabs, const float* __restrict__ arena,
                                                               const int32_t* __restrict__ row_seq, const int32_t* __restrict__ row_len,
                                                               const int32_t* __restrict__ blk_tab, int H, int r_, int t_max,
                                                               int tiles_per_split, float* __restrict__ lat, float* __restrict__ part_acc,
                                                               float* __restrict__ part_ml, int KS, int M) {
  using Walk = LatentWalk<NB, KF, VEC, PlainScore>;
  __shared__ __attribute__((aligned(16))) float lds[Walk::LDS_FLOATS];
  const int row0 = blk_tab[2 * blockIdx.x], nrows = blk_tab[2 * blockIdx.x + 1];
  const int nqv = nrows * H, tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, c = lane & 15, g4 = lane >> 4;
  // (one pass unless the grid was cut for runs of one row and this one is longer)
  for (int qv0 = blockIdx.y * 16; qv0 < nqv; qv0 += 16 * gridDim.y) {
    int r = r_;
    asm("" : "+s"(r));                     // (what depends on it is not held over the passes: it would cost half the waves)
    const int64_t seq = row_seq[row0];
    const int len = row_len[row0 + nrows - 1];
    const bool on = qv0 + c < nqv;
    const int qv = on ? qv0 + c : nqv - 1;
    const int64_t o = (int64_t)(row0 + qv / H) * H + qv % H;
    f32x4 q[NB], acc[NB];
#pragma unroll
    for (int it = 0; it < NB; ++it) q[it] = load4<VEC>(qabs + o * r, wave * 16 * NB + 16 * it + 4 * g4, r, on);
    const int n_tiles = (len + Walk::KT - 1) / Walk::KT;
    const int t0 = blockIdx.z * tiles_per_split, t1 = min(t0 + tiles_per_split, n_tiles);
    float mrun, lrun;
    Walk::run(lds, arena + seq * t_max * r, r, r, len, on ? row_len[row0 + qv / H] : len, t0, t1, q, PlainScore{}, mrun, lrun, acc);
    if (!on) continue;
    const float inv = KS == 1 ? 1.0f / lrun : 1.0f;
    float* dst = KS == 1 ? lat + o * r : part_acc + ((int64_t)blockIdx.z * M * H + o) * r;
#pragma unroll
    for (int x = 0; x < NB; ++x) {
      const int d = 16 * (wave + 4 * x) + 4 * g4;
      if (VEC) {
        if (d < r) *reinterpret_cast<f32x4u*>(dst + d) = acc[x] * inv;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (d + e < r) dst[d + e] = acc[x][e] * inv;
      }
    }
    if (KS > 1 && wave == 0 && g4 == 0) {
      const int64_t po = (int64_t)blockIdx.z * M * H + o;
      part_ml[po * 2] = mrun;
      part_ml[po * 2 + 1] = lrun;
    }
  }
}

// The same for latents of 16 NT values, up to 512: a wave takes whole tiles of 16 keys for itself, a running maximum and sum and the 16 NT x 16 sums of its own, and the four waves of a
// workgroup meet once, at the end.  Nothing is exchanged between waves and no barrier stands in the walk.  The loads lie as the scores' A operand (lane: key l % 16, values 4 (l / 16) .. + 3
// of every 16), so a tile goes from memory into registers and from there into the scores; the value products want it turned, which a tile of LDS that only this wave touches does.
// A register that has been multiplied is asked for what follows half a tile further on: loads are in flight all the time.  What bounds it is memory in the walk (5.2 TB/s) and the ends, 5 us until
// the first tile is there and 3 from the last one to the split's results.  us, the form above -> this, the splits' join with it: 32 rows of 16 heads over 2049 latents of 512 54.5 -> 44.4 (the walk alone
// 41.7 -> 36.3; 134 MB, 23 us at the rate of a plain read), 64 rows over 1000 47.0 -> 40.7, 64 rows of 8 heads over 2048 of 256 39.1 -> 37.8; prompts of 2048, 1000, 300, 130 tokens, 16 heads over
// latents of 512, 909 -> 760, 270 -> 240, 48.5 -> 43, 24.6 -> 22.7, 2048 tokens of 8 heads over 256 273 -> 222.  With long walks taken first (prompts, us): 16 heads over 512 2048 tokens 715 -> 635, 900
// 190 -> 155, 300 42.5 -> 32.7, five of 282 133 -> 117, 8 heads over 256 2048 tokens 206 -> 167.
// The sums are taken against a maximum that is raised only where a score is above it by more than 8 (weights up to e^8, which fp32 holds as well as 1): scaling sums that live in the
// matrix cores' half of the registers would cost every tile a copy of them.  Error against 64 bits 1.4 .. 2.0e-7, the form above 1.7 .. 2.9e-7.
__device__ __forceinline__ void wave_order() {         // what the lanes of a wave hand each other through LDS: the hardware keeps its order, this the compiler's
  asm volatile("" ::: "memory");
  __builtin_amdgcn_wave_barrier();
}
template <int NT>
__global__ __launch_bounds__(256, NT <= 16 ? 2 : 1) void latent_attn_wave_kernel(const float* __restrict__ qabs, const float* __restrict__ arena, const int32_t* __restrict__ row_seq,
                                                                                 const int32_t* __restrict__ row_len, const int32_t* __restrict__ blk_tab, int H, int t_max,
                                                                                 float* __restrict__ lat, float* __restrict__ part_acc, float* __restrict__ part_ml, int KS, int M) {
  constexpr int R = 16 * NT, LDK = R + 4, TILE = 16 * LDK, RG = NT % 16 == 0 ? 16 : 8;      // RG: loads of a lane in flight
  static_assert(NT % RG == 0, "a ring slot keeps its place from tile to tile");
  __shared__ __attribute__((aligned(16))) float lds[4 * TILE];
  __shared__ float wm[4][16], wl[4][16];
  __shared__ __attribute__((aligned(16))) float scale[NT > 16 ? 4 : 1][NT > 16 ? 1024 : 4];
  // long walks (a prompt's late rows) first, the query vectors of a run side by side: what is taken last is short
  const int order = blockIdx.y * gridDim.x + blockIdx.x, run = gridDim.x - 1 - order / gridDim.y, row0 = blk_tab[2 * run], nrows = blk_tab[2 * run + 1];
  const int nqv = nrows * H, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  float* K = lds + wave * TILE;
  // (one pass unless the grid was cut for runs of one row and this one is longer)
  for (int qv0 = order % gridDim.y * 16; qv0 < nqv; qv0 += 16 * gridDim.y) {
    int lane = threadIdx.x & 63;
    asm("" : "+v"(lane));                              // (what depends on it is not held over the passes: registers)
    const int c = lane & 15, g4 = lane >> 4;
    const int len = row_len[row0 + nrows - 1];
    const bool on = qv0 + c < nqv;
    const int qv = on ? qv0 + c : nqv - 1, mine = row_len[row0 + qv / H];
    const int64_t o = (int64_t)(row0 + qv / H) * H + qv % H;
    const float* kb = arena + (int64_t)row_seq[row0] * t_max * R + 4 * g4;
    auto keys = [&](int tile) { return kb + (int64_t)min(16 * tile + c, len - 1) * R; };
    // the run's own tiles in equal parts, a part's tiles to its waves in turn
    const uint32_t n = (uint32_t)((len + 15) >> 4);
    const int t1 = (int)((blockIdx.z + 1) * n / (uint32_t)KS);
    int tile = (int)(blockIdx.z * n / (uint32_t)KS) + wave;
    f32x4 k[RG], q[NT], acc[NT];
    const float* p = keys(min(tile, (int)n - 1));
    if (tile < t1) {
#pragma unroll
      for (int it = 0; it < RG; ++it) k[it] = *reinterpret_cast<const f32x4*>(p + 16 * it);
    }
    __builtin_amdgcn_sched_barrier(0);
    {
      const float* qr = qabs + o * R + 4 * g4;
#pragma unroll
      for (int it = 0; it < NT; ++it) q[it] = *reinterpret_cast<const f32x4*>(qr + 16 * it);
    }
#pragma unroll
    for (int it = 0; it < NT; ++it) acc[it] = f32x4{0.f, 0.f, 0.f, 0.f};
    float mrun = -INFINITY, lrun = 0.f;
    __builtin_amdgcn_s_waitcnt(0x0f70);                // (all of them, once: in the walk a wait for one register of the ring is then no wait for the others)
    float* kw = K + c * LDK + 4 * g4;
    const float* kr = K + 4 * g4 * LDK + c;
    for (; tile < t1; tile += 4) {
      const float* pn = keys(min(tile + 4, t1 - 1));      // (behind the last tile: something of this workgroup's, not used)
      f32x4 s[8];                                      // eight chains of sums: no longer ones than those of four waves that split a key's values
#pragma unroll
      for (int e = 0; e < 8; ++e) s[e] = f32x4{0.f, 0.f, 0.f, 0.f};
      wave_order();                                    // the tile before has been read
#pragma unroll
      for (int it = 0; it < NT; ++it) {
        *reinterpret_cast<f32x4*>(kw + 16 * it) = k[it % RG];
#pragma unroll
        for (int e = 0; e < 4; ++e) s[it / (NT / 2) * 4 + e] = __builtin_amdgcn_mfma_f32_16x16x4f32(k[it % RG][e], q[it][e], s[it / (NT / 2) * 4 + e], 0, 0, 0);
        if (it + RG < NT) k[it % RG] = *reinterpret_cast<const f32x4*>(p + 16 * (it + RG));
        else k[it % RG] = *reinterpret_cast<const f32x4*>(pn + 16 * (it + RG - NT));
        __builtin_amdgcn_sched_barrier(0);
      }
      p = pn;
      wave_order();
      f32x4 w = ((s[0] + s[1]) + (s[2] + s[3])) + ((s[4] + s[5]) + (s[6] + s[7]));
      const int key0 = 16 * tile + 4 * g4;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (key0 + i >= mine) w[i] = -INFINITY;
      float mx = fmaxf(fmaxf(w[0], w[1]), fmaxf(w[2], w[3]));
      mx = fmaxf(mx, __shfl_xor(mx, 16));
      mx = fmaxf(mx, __shfl_xor(mx, 32));
      if (__ballot(mx > mrun + 8.0f)) {
        const float mnew = mx > mrun + 8.0f ? mx : mrun, corr = mrun == -INFINITY ? 0.f : fast_exp(mrun - mnew);
        lrun *= corr;
        const bool fresh = __ballot(mrun != -INFINITY) == 0;
        mrun = mnew;
        if (NT <= 16) {
#pragma unroll
          for (int x = 0; x < NT; ++x) acc[x] *= corr;
        } else if (!fresh) {                           // the sums live in the matrix cores' half of the registers: scaled by way of LDS, or every tile would hold a copy of them
          f32x4* z = reinterpret_cast<f32x4*>(scale[wave]) + lane;
#pragma unroll
          for (int x = 0; x < NT; x += 4) {
#pragma unroll
            for (int u = 0; u < 4; ++u) z[u * 64] = acc[x + u];
            wave_order();
#pragma unroll
            for (int u = 0; u < 4; ++u) z[u * 64] *= corr;
            wave_order();
#pragma unroll
            for (int u = 0; u < 4; ++u) acc[x + u] = z[u * 64];
            wave_order();
          }
        }
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) w[i] = w[i] == -INFINITY ? 0.f : fast_exp(w[i] - mrun);
      lrun += (w[0] + w[1]) + (w[2] + w[3]);
      float v[2][8];                                   // a group of eight products, the next one's values on their way
      auto read = [&](int u) {
#pragma unroll
        for (int x = 0; x < 8; ++x) v[u & 1][x] = kr[(u / (NT / 8)) * LDK + 16 * (u % (NT / 8) * 8 + x)];
      };
      read(0);
#pragma unroll
      for (int u = 0; u < NT / 2; ++u) {
        if (u + 1 < NT / 2) read(u + 1);
#pragma unroll
        for (int x = 0; x < 8; ++x) {
          f32x4& a = acc[u % (NT / 8) * 8 + x];
          a = __builtin_amdgcn_mfma_f32_16x16x4f32(v[u & 1][x], w[u / (NT / 8)], a, 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    lrun += __shfl_xor(lrun, 16);
    lrun += __shfl_xor(lrun, 32);
    // ---- the waves' results meet: wave w sums the column blocks w, w + 4, .. ----
    if (g4 == 0) { wm[wave][c] = mrun; wl[wave][c] = lrun; }
    wave_order();
#pragma unroll
    for (int x = 0; x < NT; ++x) *reinterpret_cast<f32x4*>(K + lane * 4 + x * 256) = acc[x];
    __syncthreads();
    float top = -INFINITY, l = 0.f, f[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) top = fmaxf(top, wm[u][c]);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      f[u] = wm[u][c] == -INFINITY ? 0.f : fast_exp(wm[u][c] - top);
      l = fmaf(f[u], wl[u][c], l);
    }
    const float inv = KS == 1 ? 1.0f / l : 1.0f;
    float* dst = (KS == 1 ? lat + o * R : part_acc + ((int64_t)blockIdx.z * M * H + o) * R) + 16 * wave + 4 * g4;
    const float* from = lds + wave * 256 + lane * 4;
#pragma unroll
    for (int y = 0; y < NT / 4; ++y) {
      f32x4 a = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int u = 0; u < 4; ++u) a += f[u] * *reinterpret_cast<const f32x4*>(from + u * TILE + y * 1024);
      if (on) *reinterpret_cast<f32x4*>(dst + 64 * y) = a * inv;
    }
    if (KS > 1 && on && wave == 0 && g4 == 0) {
      const int64_t po = (int64_t)blockIdx.z * M * H + o;
      part_ml[po * 2] = top;
      part_ml[po * 2 + 1] = l;
    }
    __syncthreads();                                   // (another pass writes here)
  }
}

// one wave per (row, head) and 64 latent components: combine the key splits (lane s holds split s's maximum and sum; KS <= 64)
__global__ __launch_bounds__(256) void latent_merge_kernel(const float* __restrict__ part_acc, const float* __restrict__ part_ml, int KS,
                                                           int MH, int r, float* __restrict__ lat) {
  const int o = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63, d = blockIdx.y * 64 + lane;
  if (o >= MH) return;
  const float ms = lane < KS ? part_ml[((int64_t)lane * MH + o) * 2] : -INFINITY;
  const float ls = lane < KS ? part_ml[((int64_t)lane * MH + o) * 2 + 1] : 0.f;
  const float mx = wave_max(ms);
  const float w = (ms == -INFINITY) ? 0.f : expf(ms - mx);
  const float inv = 1.0f / wave_sum(w * ls);
  const int dc = d < r ? d : r - 1;
  float a = 0.f;
#pragma unroll 16
  for (int s = 0; s < KS; ++s) a = fmaf(lane_f(w, s), part_acc[((int64_t)s * MH + o) * r + dc], a);
  if (d < r) lat[(int64_t)o * r + d] = a * inv;
}

}  // namespace

// ---- C entry points ----------------------------------------------------------------------------------------------------------
extern "C" int mn_affine_ln_rows(const float* x, int64_t ldx, const uint16_t* w, const uint16_t* b, float eps, float* y, int64_t ldy,
                                 uint16_t* y16, int64_t ldy16, int M, int n, void* stream) {
  MN_CHECK_ARG(x && w && b && (y || y16) && M >= 1 && n >= 1, "mn_affine_ln_rows: bad args");
  const RowArgs ra{x, ldx, nullptr, 0, nullptr, 0, w, b, eps, y, ldy, y16, ldy16, n, 0};
  if (!launch_row_block<ROW_LN>(ra, M, mn_stream(stream)))
    hipLaunchKernelGGL(affine_ln_kernel, dim3((unsigned)mn_cdiv(M, 4)), dim3(256), 0, mn_stream(stream), x, ldx, w, b, eps, y, ldy, y16, ldy16,
                       M, n);
  MN_CHECK_LAUNCH("mn_affine_ln_rows");
  return MN_OK;
}

extern "C" int mn_gated_ln_residual(float* x, int64_t ldx, const float* g, int64_t ldg, const float* y, int64_t ldy, const uint16_t* w,
                                    const uint16_t* b, float eps, int M, int n, void* stream) {
  MN_CHECK_ARG(x && g && y && w && b && M >= 1 && n >= 1, "mn_gated_ln_residual: bad args");
  const RowArgs ra{nullptr, 0, g, ldg, y, ldy, w, b, eps, x, ldx, nullptr, 0, n, 0};
  if (!launch_row_block<ROW_GATED_LN_RESIDUAL>(ra, M, mn_stream(stream)))
    hipLaunchKernelGGL(gated_ln_residual_kernel, dim3((unsigned)mn_cdiv(M, 4)), dim3(256), 0, mn_stream(stream), x, ldx, g, ldg, y, ldy, w, b,
                       eps, M, n);
  MN_CHECK_LAUNCH("mn_gated_ln_residual");
  return MN_OK;
}

extern "C" int mn_rms_rows(const float* x, int64_t ldx, const uint16_t* w, float eps, float* y, int64_t ldy, uint16_t* y16, int64_t ldy16,
                           const int32_t* row_seq, const int32_t* row_slot, int t_max, int M, int n, void* stream) {
  MN_CHECK_ARG(x && w && (y || y16) && M >= 1 && n >= 1 && (!row_seq || (row_slot && t_max >= 1)), "mn_rms_rows: bad args");
  const RmsJobs jobs{{RmsJob{x, ldx, w, y, ldy, y16, ldy16, row_seq, row_slot, t_max, n}, RmsJob{}}};
  if (rms_vec_ok(jobs.job[0])) {
    rms_vec_launch(jobs, 1, eps, M, mn_stream(stream));
    MN_CHECK_LAUNCH("mn_rms_rows");
    return MN_OK;
  }
  hipLaunchKernelGGL(rms_rows_kernel, dim3((unsigned)mn_cdiv(M, 4)), dim3(256), 0, mn_stream(stream), x, ldx, w, eps, y, ldy, y16, ldy16,
                     row_seq, row_slot, t_max, M, n);
  MN_CHECK_LAUNCH("mn_rms_rows");
  return MN_OK;
}

// two norms of the same M rows, the second into a cache arena (rows of either that the vector form does not take: one launch each)
extern "C" int mn_rms_rows_pair(const float* xa, const uint16_t* wa, float* ya, int64_t ldya, uint16_t* ya16, int64_t ldya16, int na, const float* xb, const uint16_t* wb,
                                float* yb, const int32_t* row_seq, const int32_t* row_slot, int t_max, int nb, int64_t ldx, float eps, int M, void* stream) {
  MN_CHECK_ARG(xa && wa && (ya || ya16) && xb && wb && yb && row_seq && row_slot && t_max >= 1 && M >= 1 && na >= 1 && nb >= 1, "mn_rms_rows_pair: bad args");
  const RmsJobs jobs{{RmsJob{xa, ldx, wa, ya, ldya, ya16, ldya16, nullptr, nullptr, 0, na}, RmsJob{xb, ldx, wb, yb, nb, nullptr, 0, row_seq, row_slot, t_max, nb}}};
  if (rms_vec_ok(jobs.job[0]) && rms_vec_ok(jobs.job[1])) {
    rms_vec_launch(jobs, 2, eps, M, mn_stream(stream));
    MN_CHECK_LAUNCH("mn_rms_rows_pair");
    return MN_OK;
  }
  const int rc = mn_rms_rows(xa, ldx, wa, eps, ya, ldya, ya16, ldya16, nullptr, nullptr, 0, M, na, stream);
  return rc != MN_OK ? rc : mn_rms_rows(xb, ldx, wb, eps, yb, nb, nullptr, 0, row_seq, row_slot, t_max, M, nb, stream);
}

extern "C" int mn_polynorm_rows(const float* z, int64_t ldz, const uint16_t* coef, float eps, float* y, int64_t ldy, uint16_t* y16,
                                int64_t ldy16, int M, int n, void* stream) {
  MN_CHECK_ARG(z && coef && (y || y16) && M >= 1 && n >= 1, "mn_polynorm_rows: bad args");
  const RowArgs ra{z, ldz, nullptr, 0, nullptr, 0, coef, nullptr, eps, y, ldy, y16, ldy16, n, 0};
  if (!launch_row_block<ROW_POLYNORM>(ra, M, mn_stream(stream)))
    hipLaunchKernelGGL(polynorm_kernel, dim3((unsigned)M), dim3(256), 0, mn_stream(stream), z, ldz, coef, eps, y, ldy, y16, ldy16, n);
  MN_CHECK_LAUNCH("mn_polynorm_rows");
  return MN_OK;
}

// The same with its rows as bf16 hi rows, then lo rows (y16 [2, M, n] dense): the operand of a product on such rows; rows of 512 .. 8192 values
extern "C" int mn_polynorm_rows_split(const float* z, int64_t ldz, const uint16_t* coef, float eps, uint16_t* y16, int M, int n, void* stream) {
  MN_CHECK_ARG(z && coef && y16 && M >= 1 && n >= 512 && n <= 8192, "mn_polynorm_rows_split: bad args");
  const RowArgs ra{z, ldz, nullptr, 0, nullptr, 0, coef, nullptr, eps, nullptr, 0, y16, n, n, (int64_t)M * n};
  launch_row_block<ROW_POLYNORM>(ra, M, mn_stream(stream));
  MN_CHECK_LAUNCH("mn_polynorm_rows_split");
  return MN_OK;
}

extern "C" int mn_tap_filter_rows(const float* x, int64_t ldx, const uint16_t* w, int taps, const float* state, const int32_t* row_seq,
                                  const int32_t* row_slot, const int32_t* row_back, float* y, int64_t ldy, uint16_t* y16, int64_t ldy16,
                                  int M, int n, void* stream) {
  MN_CHECK_ARG(x && w && taps >= 1 && (state || taps == 1) && row_seq && row_slot && row_back && (y || y16) && M >= 1 && n >= 1,
               "mn_tap_filter_rows: bad args");
  MN_CHECK_ARG(M <= 65535, "mn_tap_filter_rows: at most 65535 rows per call");
  hipLaunchKernelGGL(tap_filter_kernel, dim3((unsigned)mn_cdiv(n, 256), (unsigned)M), dim3(256), 0, mn_stream(stream), x, ldx, w, taps, state,
                     row_seq, row_slot, row_back, y, ldy, y16, ldy16, n, 1.0f);
  MN_CHECK_LAUNCH("mn_tap_filter_rows");
  return MN_OK;
}

extern "C" int mn_tap_conv_rows(const float* x, int64_t ldx, const uint16_t* w, int taps, const float* state, const int32_t* row_seq,
                                const int32_t* row_slot, const int32_t* row_back, float* y, int64_t ldy, int M, int n, void* stream) {
  MN_CHECK_ARG(x && w && taps >= 1 && (state || taps == 1) && row_seq && row_slot && row_back && y && M >= 1 && M <= 65535 && n >= 1,
               "mn_tap_conv_rows: bad args");
  hipLaunchKernelGGL(tap_filter_kernel, dim3((unsigned)mn_cdiv(n, 256), (unsigned)M), dim3(256), 0, mn_stream(stream), x, ldx, w, taps, state,
                     row_seq, row_slot, row_back, y, ldy, (bf16_t*)nullptr, (int64_t)0, n, 0.0f);
  MN_CHECK_LAUNCH("mn_tap_conv_rows");
  return MN_OK;
}

extern "C" int mn_tap_state_update(const float* x, int64_t ldx, int taps, float* state, const int32_t* row_seq, const int32_t* row_back,
                                   int M, int n, void* stream) {
  MN_CHECK_ARG(x && taps >= 1 && row_seq && row_back && M >= 1 && M <= 65535 && n >= 1, "mn_tap_state_update: bad args");
  if (taps == 1) return MN_OK;
  MN_CHECK_ARG(state, "mn_tap_state_update: null state");
  hipLaunchKernelGGL(tap_state_kernel, dim3((unsigned)mn_cdiv(n, 256), (unsigned)M), dim3(256), 0, mn_stream(stream), x, ldx, taps, state,
                     row_seq, row_back, M, n);
  MN_CHECK_LAUNCH("mn_tap_state_update");
  return MN_OK;
}

// y16 (optional): mn_gated_norm_filter_rows with its last output also as bf16 hi rows, then lo rows ([2, M, n] dense)
extern "C" int mn_gated_norm_filter_rows_split(float* x, int64_t ldx, const float* g, int64_t ldg, const float* y, int64_t ldy, const uint16_t* wa,
                                         const uint16_t* ba, const uint16_t* wb, const uint16_t* bb, float eps, float* n_out, int64_t ldn,
                                         const uint16_t* taps_w, int taps, float* state, const int32_t* row_seq, const int32_t* row_slot,
                                         float* h, int64_t ldh, uint16_t* y16, int M, int n, void* stream) {
  MN_CHECK_ARG(x && wb && bb && n_out && M >= 1 && n >= 1 && n <= 4096, "mn_gated_norm_filter_rows: bad args (rows of at most 4096 values)");
  MN_CHECK_ARG(!g || (y && wa && ba), "mn_gated_norm_filter_rows: the gated stage needs y and its norm");
  MN_CHECK_ARG(!h || (taps_w && taps >= 1 && taps <= FUSED_MAX_TAPS && (state || taps == 1) && row_seq && row_slot),
               "mn_gated_norm_filter_rows: the filter stage needs its state and at most %d taps", FUSED_MAX_TAPS);
  const FusedRowArgs a{x, ldx, g, ldg, y, ldy, wa, ba, wb, bb, eps, n_out, ldn, taps_w, taps, state, row_seq, row_slot, h, ldh, n, y16, (int64_t)M * n};
  const int vpt = (n + 255) / 256;
  hipStream_t st = mn_stream(stream);
  if (row_fused_vec_ok(a)) {
    const dim3 grid((unsigned)M), block((unsigned)mn_cdiv(n / 4, 64) * 64);
#define MN_RFV(T_) case T_: hipLaunchKernelGGL((row_fused_vec_kernel<T_>), grid, block, 0, st, a); break
    switch (h ? taps : 0) { MN_RFV(0); MN_RFV(1); MN_RFV(2); MN_RFV(3); MN_RFV(4); MN_RFV(5); MN_RFV(6); MN_RFV(7); default: hipLaunchKernelGGL((row_fused_vec_kernel<8>), grid, block, 0, st, a); }
#undef MN_RFV
    MN_CHECK_LAUNCH("mn_gated_norm_filter_rows");
    return MN_OK;
  }
#define MN_RF(V_)                                                                                                    \
  do {                                                                                                               \
    if (h) hipLaunchKernelGGL((row_fused_kernel<V_, true>), dim3((unsigned)M), dim3(256), 0, st, a);                 \
    else hipLaunchKernelGGL((row_fused_kernel<V_, false>), dim3((unsigned)M), dim3(256), 0, st, a);                  \
  } while (0)
  if (vpt <= 1) MN_RF(1); else if (vpt <= 2) MN_RF(2); else if (vpt <= 4) MN_RF(4); else if (vpt <= 8) MN_RF(8); else MN_RF(16);
#undef MN_RF
  MN_CHECK_LAUNCH("mn_gated_norm_filter_rows");
  return MN_OK;
}

extern "C" int mn_gated_norm_filter_rows(float* x, int64_t ldx, const float* g, int64_t ldg, const float* y, int64_t ldy, const uint16_t* wa,
                                         const uint16_t* ba, const uint16_t* wb, const uint16_t* bb, float eps, float* n_out, int64_t ldn,
                                         const uint16_t* taps_w, int taps, float* state, const int32_t* row_seq, const int32_t* row_slot,
                                         float* h, int64_t ldh, int M, int n, void* stream) {
  return mn_gated_norm_filter_rows_split(x, ldx, g, ldg, y, ldy, wa, ba, wb, bb, eps, n_out, ldn, taps_w, taps, state, row_seq, row_slot, h, ldh, nullptr, M, n, stream);
}

extern "C" int mn_softcap_rows(float* z, int64_t ld, int M, int n, float cap, void* stream) {
  MN_CHECK_ARG(z && M >= 1 && M <= 65535 && n >= 1 && cap > 0.f, "mn_softcap_rows: bad args");
  hipLaunchKernelGGL(softcap_kernel, dim3((unsigned)mn_cdiv(n, 256), (unsigned)M), dim3(256), 0, mn_stream(stream), z, ld, n, cap);
  MN_CHECK_LAUNCH("mn_softcap_rows");
  return MN_OK;
}

extern "C" int mn_gemm_f32_batched(const float* A, int64_t lda, int64_t a_bs, const uint16_t* W, int64_t ldw, int64_t w_bs,
                                   const uint16_t* bias, float* C, int64_t ldc, int64_t c_bs, uint16_t* C16, int64_t ldc16, int64_t c16_bs,
                                   const float* G, int64_t ldg, int64_t g_bs, int M, int N, int K, int batch, float alpha, void* stream) {
  MN_CHECK_ARG(A && W && (C || C16) && M >= 1 && N >= 1 && K >= 1 && batch >= 1 && batch <= 65535, "mn_gemm_f32_batched: bad args");
  GemmF32 a{A, lda, a_bs, W, ldw, w_bs, bias, C, ldc, c_bs, C16, ldc16, c16_bs, G, ldg, g_bs, M, N, K, alpha};
  hipStream_t st = mn_stream(stream);
  const bool v4 = (K % 4) == 0 && (lda % 4) == 0 && (a_bs % 4) == 0 && ((uintptr_t)A & 15) == 0 && (ldw % 4) == 0 && (w_bs % 4) == 0 && ((uintptr_t)W & 7) == 0;
  // One wave a column, lanes over K: one or two rows, and up to 8 value by value.  Its time grows with the rows, the matrix cores' does not.  us, this / those: 16 x 128 x 512 2 rows 4.4 / 5.9,
  // 3 6.0 / 6.0, 6 8.3 / 6.0, 8 10.0 / 6.0; 16 x 512 x 128 2 rows 3.5 / 4.1, 3 4.5 / 4.1, 8 6.4 / 4.2; 2048 x 1024 3 rows 12.3 / 10.1, 8 19.6 / 10.1; value by value 64 x 4096 8 rows 57 / 73.  Error 0.8 .. 1.8e-7 / 0.7e-7.
  if (M <= (v4 ? 2 : 8)) {
    if (M <= 2) hipLaunchKernelGGL((gemv_f32_kernel<2>), dim3((unsigned)mn_cdiv(N, 4), 1, (unsigned)batch), dim3(256), 0, st, a);
    else hipLaunchKernelGGL((gemv_f32_kernel<8>), dim3((unsigned)mn_cdiv(N, 4), 1, (unsigned)batch), dim3(256), 0, st, a);
    MN_CHECK_LAUNCH("mn_gemm_f32_batched");
    return MN_OK;
  }
  MN_CHECK_ARG(mn_cdiv(M, 64) <= 65535, "mn_gemm_f32_batched: too many rows");
  const int64_t tiles = mn_cdiv(M, 64) * mn_cdiv(N, 64) * batch;
  // up to 64 rows always take the kernel that keeps its roundings (they are decode rows: error against 64 bits 0.2 .. 0.6e-7 of the summed
  // magnitudes).  More rows, from 128 tiles on (us, few / tiles: 200 rows of 16 x 128 x 512, 128 tiles, 17.5 / 11.2; 128 rows, 64 tiles, 10.3 / as many K-steps as those 11.2;
  // 2048 rows x 4096 x 1024 354 / 87)
  if (M <= 64 || 2 * tiles < mn_num_cus()) {
    const dim3 grid((unsigned)mn_cdiv(N, 16), (unsigned)mn_cdiv(M, 32), (unsigned)batch);
    if (v4) hipLaunchKernelGGL(gemm_f32_few_kernel<true>, grid, dim3(256), 0, st, a);
    else hipLaunchKernelGGL(gemm_f32_few_kernel<false>, grid, dim3(256), 0, st, a);
  } else {
    const dim3 grid((unsigned)mn_cdiv(N, 64), (unsigned)mn_cdiv(M, 64), (unsigned)batch);
    const bool many = tiles > 2 * (int64_t)mn_num_cus();
    if (v4 && many) hipLaunchKernelGGL((gemm_f32_tile_kernel<true, 1>), grid, dim3(256), 0, st, a);
    else if (v4) hipLaunchKernelGGL((gemm_f32_tile_kernel<true, 2>), grid, dim3(256), 0, st, a);
    else if (many) hipLaunchKernelGGL((gemm_f32_tile_kernel<false, 1>), grid, dim3(256), 0, st, a);
    else hipLaunchKernelGGL((gemm_f32_tile_kernel<false, 2>), grid, dim3(256), 0, st, a);
  }
  MN_CHECK_LAUNCH("mn_gemm_f32_batched");
  return MN_OK;
}

// rows of a workgroup (consecutive rows of one sequence) and the key-tile length for latent size r
extern "C" int mn_latent_attn_block_rows(void) { return 4; }
static inline int latent_kt(int r, int variant) {
  // VALU: the tile [KT][r + 1] fp32 stays below 66 KiB; MFMA: 32 keys while two such tiles fit a CU's LDS
  return variant == MN_LATENT_ATTN_VALU ? (r <= 256 ? 64 : r <= 512 ? 32 : 16) : (r <= 512 ? 32 : 16);
}

// Two workgroups a CU, at least 64 keys a split.  Never fewer for longer sequences or for fewer runs: scratch sized by it for the longest serves every shorter step.
extern "C" int mn_latent_attn_splits(int n_blk, int max_len, int r) {
  const int tiles = (int)mn_cdiv(max_len > 0 ? max_len : 1, 16);
  int ks = (int)mn_cdiv(2 * (int64_t)mn_num_cus(), n_blk > 0 ? n_blk : 1);
  const int cap = (int)mn_cdiv(tiles, 4);
  if (ks > cap) ks = cap;
  if (ks > 64) ks = 64;
  (void)r;
  return ks < 1 ? 1 : ks;
}

// Whole tiles a wave (0: not that form): where a wave has two of them or more in one round of its workgroups, which is then all the splits there are, of the `ks` that the caller has scratch for;
// wgs: workgroups a split.  With fewer tiles the form whose waves share one is the faster one (us, shared / whole: 64 rows over 300 of 512 27.3 / 25.9 .. 28, 8 rows over 2049
// 27.8 / 29.5, one 22.5 / 24.8, 64 over 64 11.6 / 14.1, 40 rows over 1111 of 256 22.4 / 27.9).  A prompt's rows see half of max_len on average: with more workgroups than one round (above 256 values: three) the
// short walks are the time, and from 160 (320) keys on whole tiles are worth it (16 heads, of 512: 4 prompts of 128 24.0 / 28.6, 5 of 200 68 / 75, 15 of 200 160 / 203, 6 of 300 143 / 153, 4 of 512 272 / 226, one of
// 300 48 / 33; 32 heads, 10 of 200 204 / 264; of 256, 16 heads: 16 of 128 55 / 59, 5 of 11 .. 140 23.8 / 18.4, 8 of 256 86 / 77).
static inline int latent_wave_splits(int r, int max_len, int64_t wgs, int ks, bool runs) {
  if (r != 128 && r != 256 && r != 384 && r != 512) return 0;
  const int cus = mn_num_cus();
  int64_t kw = (r <= 256 ? 2 : 1) * cus / wgs;
  if (kw < 1) kw = 1;
  if (kw > ks) kw = ks;
  if (runs && max_len < 160 && (r <= 256 ? wgs >= 2 * cus : wgs > cus)) return 0;
  if (runs && max_len < 320 && r > 256 && wgs > 3 * cus) return 0;
  return max_len >= 128 * kw ? (int)kw : 0;
}

extern "C" size_t mn_latent_attn_workspace_bytes(int M, int H, int r, int ks) {
  return ks <= 1 ? 0 : (size_t)ks * M * H * (r + 2) * sizeof(float);
}

extern "C" int mn_latent_attn_ex(const float* qabs, const float* arena, const int32_t* row_seq, const int32_t* row_len,
                                 const int32_t* blk_tab, int n_blk, int M, int H, int r, int t_max, int max_len, int ks, float* lat, void* ws,
                                 size_t ws_bytes, int variant, void* stream) {
  MN_CHECK_ARG(qabs && arena && row_seq && row_len && blk_tab && lat && n_blk >= 1 && M >= 1 && H >= 1 && r >= 1 && t_max >= 1,
               "mn_latent_attn: bad args");
  MN_CHECK_ARG(r <= 1024, "mn_latent_attn: latent size %d above 1024 is not supported", r);
  MN_CHECK_ARG(max_len >= 1 && max_len <= t_max && ks >= 1 && ks <= 64, "mn_latent_attn: bad max_len=%d / ks=%d (1 .. 64 key splits)", max_len, ks);
  MN_CHECK_ARG(ws_bytes >= mn_latent_attn_workspace_bytes(M, H, r, ks) && (ks == 1 || ws), "mn_latent_attn: workspace too small");
  MN_CHECK_ARG(variant == MN_LATENT_ATTN_MFMA || variant == MN_LATENT_ATTN_VALU, "mn_latent_attn: unknown variant %d", variant);
  const int KT = latent_kt(r, variant), RB = mn_latent_attn_block_rows();
  const int gy = (int)mn_cdiv((n_blk == M ? 1 : RB) * (int64_t)H, 16);
  float* pacc = reinterpret_cast<float*>(ws);
  const bool aligned = (((uintptr_t)qabs | (uintptr_t)arena | (uintptr_t)lat | (uintptr_t)pacc) & 15) == 0;
  const int kw = variant == MN_LATENT_ATTN_MFMA && aligned ? latent_wave_splits(r, max_len, (int64_t)n_blk * gy, ks, n_blk < M) : 0;
  if (kw) ks = kw;
  const int tiles = (int)mn_cdiv(max_len, KT), tps = (int)mn_cdiv(tiles, ks);
  float* pml = pacc ? pacc + (size_t)ks * M * H * r : nullptr;
  hipStream_t st = mn_stream(stream);
  if (variant == MN_LATENT_ATTN_MFMA) {
    const int nbw = (int)mn_cdiv(r, 64);
    // as many runs as rows: one row each, or longer ones beside empty ones, whose workgroups go round again (workgroups for the rows a run does not have
    // still wait for their LDS: 3 of 4 in a decode step)
    const dim3 grid((unsigned)n_blk, (unsigned)gy, (unsigned)ks);
    MN_CHECK_ARG(mn_cdiv(RB * H, 16) <= 65535 && ks <= 64, "mn_latent_attn: too many heads or key splits");
#define MN_LM(N_, F_, V_)                                                                                                           \
  hipLaunchKernelGGL((latent_attn_mfma_kernel<N_, F_, V_>), grid, dim3(256), 0, st, qabs, arena, row_seq, row_len, blk_tab, H, r, t_max, tps, lat, pacc, \
                     pml, ks, M)
    if (kw) {
#define MN_LW(N_)                                                                                                                              \
  hipLaunchKernelGGL((latent_attn_wave_kernel<N_>), grid, dim3(256), 0, st, qabs, arena, row_seq, row_len, blk_tab, H, t_max, lat, pacc, pml, ks, M)
      if (r == 128) MN_LW(8); else if (r == 256) MN_LW(16); else if (r == 384) MN_LW(24); else MN_LW(32);
#undef MN_LW
    } else if (r & 3) {                                         // (latents of any size but a multiple of 4 go value by value)
      if (nbw <= 2) MN_LM(2, 2, false); else if (nbw <= 8) MN_LM(8, 2, false); else MN_LM(16, 1, false);
    } else {                                             // instantiated paddings: 64 .. 256, 384, 512, 768, 1024
      if (nbw == 1) MN_LM(1, 2, true); else if (nbw == 2) MN_LM(2, 2, true); else if (nbw == 3) MN_LM(3, 2, true); else if (nbw == 4) MN_LM(4, 2, true);
      else if (nbw <= 6) MN_LM(6, 2, true); else if (nbw <= 8) MN_LM(8, 2, true); else if (nbw <= 12) MN_LM(12, 1, true); else MN_LM(16, 1, true);
    }
#undef MN_LM
  } else {
    const int nw = RB * H < 16 ? RB * H : 16;
    const dim3 grid((unsigned)n_blk, (unsigned)mn_cdiv(RB * H, nw), (unsigned)ks), block((unsigned)(64 * nw));
    MN_CHECK_ARG(grid.y <= 65535, "mn_latent_attn: too many heads");
    const size_t lds = (size_t)KT * (r + 1) * sizeof(float);
#define MN_LA(R_)                                                                                                                   \
  do {                                                                                                                              \
    static bool attr_set = false;                                                                                                   \
    if (!attr_set) {                                                                                                                \
      (void)hipFuncSetAttribute(reinterpret_cast<const void*>(latent_attn_kernel<R_>), hipFuncAttributeMaxDynamicSharedMemorySize, 80 * 1024); \
      attr_set = true;                                                                                                              \
    }                                                                                                                               \
    hipLaunchKernelGGL((latent_attn_kernel<R_>), grid, block, lds, st, qabs, arena, row_seq, row_len, blk_tab, H, r, t_max, KT, tps, lat, \
                       pacc, pml, ks, M);                                                                                           \
  } while (0)
    if (r <= 64) MN_LA(1); else if (r <= 128) MN_LA(2); else if (r <= 256) MN_LA(4); else if (r <= 512) MN_LA(8); else MN_LA(16);
#undef MN_LA
  }
  MN_CHECK_LAUNCH("mn_latent_attn");
  if (ks > 1) {
    hipLaunchKernelGGL(latent_merge_kernel, dim3((unsigned)mn_cdiv((int64_t)M * H, 4), (unsigned)mn_cdiv(r, 64)), dim3(256), 0, st, pacc, pml, ks, M * H, r,
                       lat);
    MN_CHECK_LAUNCH("mn_latent_attn(merge)");
  }
  return MN_OK;
}

extern "C" int mn_latent_attn(const float* qabs, const float* arena, const int32_t* row_seq, const int32_t* row_len, const int32_t* blk_tab,
                              int n_blk, int M, int H, int r, int t_max, int max_len, int ks, float* lat, void* ws, size_t ws_bytes,
                              void* stream) {
  return mn_latent_attn_ex(qabs, arena, row_seq, row_len, blk_tab, n_blk, M, H, r, t_max, max_len, ks, lat, ws, ws_bytes,
                           MN_LATENT_ATTN_MFMA, stream);
}
