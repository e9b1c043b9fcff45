// rows_gemm.hip — bf16 products whose tiles are one round of the CUs at most (gfx950): a vision block's on few rows (a picture's 65 encoder tokens, its 256 pixel-decoder tokens),
// with LayerNorm in front or the residual behind in the same launch, so that a block is five launches and not seven (block.py:80-105, mlp.py:34-40, swiglu_ffn.py:27-34), and the
// sequence models' prompts of a few hundred rows.
//
//   mn_ln_gemm_rows      C = act(bf16(LayerNorm(x)) W^T + b)      x fp32, act: none, exact GELU, SwiGLU; C bf16
//   mn_resid_gemm_rows   x += A W^T + b                           A bf16, x fp32
//   mn_rows_gemm         gemm256.hip's dense products of plain or hi/lo rows, where it estimates these forms faster than its tiles
//
// What bounds such a launch is latency, a launch boundary (1.5 us) and then one memory round trip after another, and what a CU can take in (64 B a cycle), not HBM (6 MB of weights are
// 1.3 us) and not the matrix cores.  So:
//   * a workgroup asks for all it needs at once: its rows' LayerNorm input into registers, rows and weights by global_load_lds into up to 160 KiB of LDS, bias and residual;
//   * tiles of 16 .. 64 rows by 16 .. 128 columns, the ones that bring a workgroup the fewest bytes while all of them are one round of the CUs;
//   * LayerNorm is done again by every workgroup of a row tile (32 rows x 4 KB from its XCD's L2): that costs less than a launch of its own with its round trips, and
//     no split-K slabs have to be summed by anyone: the eight waves split K inside the workgroup (in wide tiles four ways, and the columns two) and meet in LDS once.
// us a launch with cold weights, these against a 64 x 64 tile launch and the launch that norms its rows or sums its slabs: 65 rows, 1024 -> 3072 7.5 / 7.7 + 4.6,
// 1024 -> 1024 3.6 / 4.9 + 4.6, 2752 -> 1024 6.6 / 5.6 + 4.6, 1024 -> 2 x 2752 9.9 / 8.0 + 4.6; 256 rows, 1024 -> 4096 with GELU 12.2 / 10.5 + 5.2, 4096 -> 1024 10.8 / 8.8 + 5.2.
// Of the 7.5: 0.7 until the first load (32-bit offsets, one multiply for the tile: 64-bit ones and a division took 1.1), 1.2 until all are issued (64 B a cycle), 1.4 for
// the norm of two rows a wave (five vector instructions a value), 0.8 for the last weights, 0.5 + 0.6 for products, partial sums and stores, 1.5 for the launch itself.
#include <math.h>

#include "common.h"

typedef short bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

namespace {

typedef __attribute__((address_space(3))) void lds_void;
typedef const __attribute__((address_space(1))) void glb_void;

struct RowsGemm {
  const float* x; int64_t ldx; const bf16_t* g; const bf16_t* b; float eps;      // NORM: A = bf16(LayerNorm(x))
  const bf16_t* A; int64_t lda;                                                  // else
  const bf16_t* W; int64_t ldw; const bf16_t* bias; int64_t pair;                // pair: row distance from a unit's gate to its up
  void* C; int64_t ldc; int M, N, K;
  int64_t a_lo, c_lo;                                                            // HILO: elements from a row's hi part to its lo part; split results likewise
  int once;                                                                      // HILO: the weights are read past the caches (below)
  uint32_t tiles_m, magic;                                                       // magic: ceil(2^32 / tiles_m)
};
enum { R_BF16, R_GELU, R_SWIGLU, R_RESID, R_F32, R_SPLIT, R_SWIGLU_SPLIT };

__device__ __forceinline__ f32x4 bf16x4(u32x2 b) { return f32x4{bf16lo_to_f32(b.x), bf16hi_to_f32(b.x), bf16lo_to_f32(b.y), bf16hi_to_f32(b.y)}; }

template <int N>
__device__ __forceinline__ void wait_vm_n() { asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N) : "memory"); }
// all but the `rem` last stages of L loads each have landed (rem <= MAX, uniform)
template <int L, int MAX>
__device__ __forceinline__ void wait_stages(int rem) {
  if constexpr (MAX == 0) {
    wait_vm_n<0>();
  } else {
    if (rem >= MAX) wait_vm_n<L * MAX>();
    else wait_stages<L, MAX - 1>(rem);
  }
}

constexpr int KMAX = 1024;

// HILO: A is a bf16 hi row and, a_lo elements further, the same row's lo part, both multiplied.  NJ: fragments of 16 weight rows a tile; KW: waves along K (a stage is KW k-steps of 32), 8 / KW waves along the columns; S: stages of LDS
template <int EPI, bool NORM, bool HILO, int BM, int NJ, int KW, int S>
__global__ __launch_bounds__(512) void rows_gemm_kernel(const RowsGemm p) {
  constexpr int MI = BM / 16, RW = BM / 8, BN = 16 * NJ, WN = 8 / KW, NW = NJ / WN, ROWB = KW * 64, SLOTS = ROWB / 16, RPI = 1024 / ROWB;
  constexpr bool paired = EPI == R_SWIGLU || EPI == R_SWIGLU_SPLIT, resid = EPI == R_RESID, f32 = resid || EPI == R_F32, split = EPI == R_SPLIT || EPI == R_SWIGLU_SPLIT;
  constexpr int AB = NORM ? BM * KMAX * 2 : 0, AR = NORM ? 0 : HILO ? 2 * BM : BM, ROWS = BN + AR, STAGE = ROWS * ROWB, Q = STAGE / 1024 / 8;
  constexpr int OC = paired ? BN / 2 : BN, RS = BN + 4, RED = KW * BM * RS * 4, GROUPS = BM * OC / 4, T = (GROUPS + 511) / 512;
  constexpr int LDS = AB + S * STAGE > RED ? AB + S * STAGE : RED;
  static_assert(!(NORM && HILO) && NJ % WN == 0 && Q * 1024 * 8 == STAGE && Q * (S - 1) < 64 && LDS <= 160 * 1024, "whole fragments and instructions a wave, vmcnt range, LDS");
  __shared__ __attribute__((aligned(1024))) char lds[LDS];
  const bool once = HILO && p.once;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kw = wave % KW, wn = wave / KW, fr = lane & 15, fq = lane >> 4;
  // an XCD's tiles are consecutive, row tiles fastest: it reads its own part of the weights, and all of the rows
  int bid = blockIdx.x;
  {
    const int nt = gridDim.x, q = nt / 8, r = nt % 8, xcd = bid % 8, idx = bid / 8;
    bid = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + idx;
  }
  const int tn = p.tiles_m == 1 ? bid : (int)__umulhi((uint32_t)bid, p.magic), m0 = (bid - tn * (int)p.tiles_m) * BM, n0 = tn * OC;
  const int nk = (p.K + KW * 32 - 1) / (KW * 32);

  // ---- everything from memory, in the order it is needed ----
  f32x4 v[RW][4];                                       // NORM: 4 rows a wave, 16 columns a lane
  u32x2 lg[4], lb[4];
  const int nx = p.K >> 8;
  if constexpr (NORM) {
#pragma unroll
    for (int i = 0; i < RW; ++i) {
      const float* xr = p.x + (int64_t)min(m0 + wave * RW + i, p.M - 1) * p.ldx + lane * 4;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        v[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (j < nx) v[i][j] = *reinterpret_cast<const f32x4*>(xr + j * 256);
      }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (j < nx) {
        lg[j] = *reinterpret_cast<const u32x2*>(p.g + j * 256 + lane * 4);
        lb[j] = *reinterpret_cast<const u32x2*>(p.b + j * 256 + lane * 4);
      }
  }
  uint32_t src[Q], kin[Q];                             // byte offset of the row and k offset (16-byte slot, swizzled) behind each instruction of this lane
  const int rin = lane / SLOTS, slot = lane % SLOTS;
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    const int L = (wave * Q + q) * RPI + rin;
    kin[q] = (uint32_t)((slot ^ (L & 15)) << 4);
    if (!NORM && L >= BN) {
      src[q] = (uint32_t)min(m0 + (L - BN) % BM, p.M - 1) * ((uint32_t)p.lda * 2u) + (HILO && L - BN >= BM ? (uint32_t)p.a_lo * 2u : 0u);
    } else if (paired) {
      src[q] = (uint32_t)(min(n0 + L % OC, p.N - 1) + (L >= OC ? (int)p.pair : 0)) * ((uint32_t)p.ldw * 2u);
    } else {
      src[q] = (uint32_t)min(n0 + L, p.N - 1) * ((uint32_t)p.ldw * 2u);
    }
  }
  const char* Ab = reinterpret_cast<const char*>(p.A);
  const char* Wb = reinterpret_cast<const char*>(p.W);
  const uint32_t klast = (uint32_t)p.K * 2 - 16;
  auto stage = [&](int kt, int buf) {
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const int L0 = (wave * Q + q) * RPI;             // (an instruction's rows are all of A or all of W: 16 divides BN, RPI divides 16)
      const uint32_t k = min((uint32_t)kt * ROWB + kin[q], klast);      // past K: any value, the k-step is not multiplied
      const char* s = (!NORM && L0 >= BN ? Ab : Wb) + (src[q] + k);
      lds_void* d = (lds_void*)(lds + AB + buf * STAGE + (wave * Q + q) * 1024);
      if (once && L0 < BN) __builtin_amdgcn_global_load_lds((glb_void*)s, d, 16, 0, 2);       // non-temporal
      else __builtin_amdgcn_global_load_lds((glb_void*)s, d, 16, 0, 0);
    }
  };
  // bias and residual of this thread's 4 outputs of a group
  u32x2 bv[T], bu[T];
  f32x4 rv[T];
  int64_t om[T];
  int on[T];
#pragma unroll
  for (int t = 0; t < T; ++t) {
    const int idx = tid + t * 512, m = m0 + idx / (OC / 4), n = n0 + idx % (OC / 4) * 4;
    const bool ok = idx < GROUPS && m < p.M && n < p.N;  // (N % 4 == 0)
    om[t] = ok ? m : -1;
    on[t] = n;
    const int nc = min(n, p.N - 4);
    bv[t] = bu[t] = u32x2{0u, 0u};
    if (p.bias) {
      bv[t] = *reinterpret_cast<const u32x2*>(p.bias + nc);
      if (paired) bu[t] = *reinterpret_cast<const u32x2*>(p.bias + p.pair + nc);
    }
    if (resid) rv[t] = *reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(p.C) + (int64_t)min(m, p.M - 1) * p.ldc + nc);
  }
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int t = 0; t < S; ++t)
    if (t < nk) stage(t, t);
  __builtin_amdgcn_sched_barrier(0);

  // ---- LayerNorm of this wave's rows into LDS: 16-byte slots of a row swizzled by row & 15 ----
  if constexpr (NORM) {
    const float inv = 1.0f / (float)p.K;
#pragma unroll
    for (int i = 0; i < RW; ++i) {
      float s = 0.f, q2 = 0.f;
#pragma unroll
      for (int j = 0; j < 4; ++j) s += (v[i][j].x + v[i][j].y) + (v[i][j].z + v[i][j].w);
      const float mean = wave_sum(s) * inv;
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (j < nx) {
          v[i][j] -= mean;
          q2 += (v[i][j].x * v[i][j].x + v[i][j].y * v[i][j].y) + (v[i][j].z * v[i][j].z + v[i][j].w * v[i][j].w);
        }
      const float rstd = rsqrtf(wave_sum(q2) * inv + p.eps);
      const int r = wave * RW + i;
      char* row = lds + (int64_t)r * p.K * 2;
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (j < nx) {
          const f32x4 o = f32x4{v[i][j].x * rstd * bf16lo_to_f32(lg[j].x) + bf16lo_to_f32(lb[j].x), v[i][j].y * rstd * bf16hi_to_f32(lg[j].x) + bf16hi_to_f32(lb[j].x),
                                v[i][j].z * rstd * bf16lo_to_f32(lg[j].y) + bf16lo_to_f32(lb[j].y), v[i][j].w * rstd * bf16hi_to_f32(lg[j].y) + bf16hi_to_f32(lb[j].y)};
          *reinterpret_cast<u32x2*>(row + (((j * 32 + (lane >> 1)) ^ (r & 15)) << 4) + (lane & 1) * 8) = u32x2{cvt_pk_bf16(o.x, o.y), cvt_pk_bf16(o.z, o.w)};
        }
    }
  }

  // ---- K loop: a stage is one k-step of 32 for each of the KW waves ----
  f32x4 acc[MI][NW];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NW; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int sl = ((kw * 4 + fq) ^ fr) << 4;
  auto mul = [&](int t, int buf) {
    const char* w = lds + AB + buf * STAGE;
    bf16x8 af[MI], wf[NW];
#pragma unroll
    for (int j = 0; j < NW; ++j) wf[j] = *reinterpret_cast<const bf16x8*>(w + ((wn * NW + j) * 16 + fr) * ROWB + sl);
#pragma unroll
    for (int i = 0; i < MI; ++i)
      af[i] = *reinterpret_cast<const bf16x8*>(NORM ? lds + (i * 16 + fr) * p.K * 2 + (((t * KW + kw) * 4 + fq) ^ fr) * 16 : w + (BN + i * 16 + fr) * ROWB + sl);
    if constexpr (HILO) {
      bf16x8 al[MI];
#pragma unroll
      for (int i = 0; i < MI; ++i) al[i] = *reinterpret_cast<const bf16x8*>(w + (BN + BM + i * 16 + fr) * ROWB + sl);
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NW; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[j], al[i], acc[i][j], 0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NW; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[j], af[i], acc[i][j], 0, 0, 0);
  };
  if (nk <= S) {                                       // all of K is on its way: one wait
    wait_vm_n<0>();
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int t = 0; t < S; ++t)
      if (t * (KW * 32) + kw * 32 < p.K) mul(t, t);
  } else {
    int buf = 0;
    for (int t = 0; t < nk; ++t) {
      if (t == 0) wait_stages<Q, S - 1>(min(nk, S) - 1);
      else wait_stages<Q, (S > 2 ? S - 2 : 0)>(min(nk - 1 - t, S - 2));
      __builtin_amdgcn_s_barrier();                    // stage t (and, the first time, the normed rows) are everyone's; stage t - 1 has been read
      __builtin_amdgcn_sched_barrier(0);
      if (t > 0 && t - 1 + S < nk) stage(t - 1 + S, buf == 0 ? S - 1 : buf - 1);
      if (t * (KW * 32) + kw * 32 < p.K) mul(t, buf);
      buf = buf + 1 == S ? 0 : buf + 1;
    }
  }

  // ---- the KW waves' parts meet in LDS ----
  __syncthreads();
  float* red = reinterpret_cast<float*>(lds);
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NW; ++j) *reinterpret_cast<f32x4*>(red + (kw * BM + i * 16 + fr) * RS + (wn * NW + j) * 16 + fq * 4) = acc[i][j];
  __syncthreads();
#pragma unroll
  for (int t = 0; t < T; ++t) {
    if (om[t] < 0) continue;
    const int idx = tid + t * 512;
    const float* r = red + (idx / (OC / 4)) * RS + idx % (OC / 4) * 4;
    f32x4 a = bf16x4(bv[t]), u;
    f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int z = 0; z < KW; ++z) s += *reinterpret_cast<const f32x4*>(r + z * BM * RS);
    a += s;
    if (paired) {
      s = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int z = 0; z < KW; ++z) s += *reinterpret_cast<const f32x4*>(r + OC + z * BM * RS);
      u = bf16x4(bu[t]) + s;
      a = f32x4{silu_f(a.x) * u.x, silu_f(a.y) * u.y, silu_f(a.z) * u.z, silu_f(a.w) * u.w};
    }
    if (EPI == R_GELU) a = f32x4{gelu_erf_f(a.x), gelu_erf_f(a.y), gelu_erf_f(a.z), gelu_erf_f(a.w)};
    if (f32) {
      if (resid) a += rv[t];
      *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(p.C) + om[t] * p.ldc + on[t]) = a;
    } else {
      bf16_t* c = reinterpret_cast<bf16_t*>(p.C) + om[t] * p.ldc + on[t];
      if (split) {
        uint32_t h0, h1, l0, l1;
        split_pk_bf16(a.x, a.y, h0, l0);
        split_pk_bf16(a.z, a.w, h1, l1);
        *reinterpret_cast<u32x2*>(c) = u32x2{h0, h1};
        *reinterpret_cast<u32x2*>(c + p.c_lo) = u32x2{l0, l1};
      } else {
        *reinterpret_cast<u32x2*>(c) = u32x2{cvt_pk_bf16(a.x, a.y), cvt_pk_bf16(a.z, a.w)};
      }
    }
  }
}

template <int EPI, bool NORM, bool HILO, int BM, int NJ, int KW, int S>
void go(RowsGemm p, hipStream_t st) {
  p.tiles_m = (uint32_t)mn_cdiv(p.M, BM);
  p.magic = (uint32_t)mn_cdiv((int64_t)1 << 32, p.tiles_m);
  const int64_t tiles = p.tiles_m * mn_cdiv(p.N, EPI == R_SWIGLU || EPI == R_SWIGLU_SPLIT ? NJ * 8 : NJ * 16);
  hipLaunchKernelGGL((rows_gemm_kernel<EPI, NORM, HILO, BM, NJ, KW, S>), dim3((unsigned)tiles), dim3(512), 0, st, p);
}

struct Form { int bm, nj; };
int64_t form_tiles(const Form& f, int M, int64_t wrows) { return mn_cdiv(M, f.bm) * mn_cdiv(wrows, 16 * f.nj); }
template <int N, class Time>
int best_form(const Form (&forms)[N], Time time, double* us) {
  int best = 0;
  double tb = 1e30;
  for (int i = 0; i < N; ++i) {
    const double t = time(forms[i]);
    if (t < tb) { tb = t; best = i; }
  }
  if (us) *us = tb;
  return best;
}
// What a workgroup takes, us.  Behind a LayerNorm: a launch and its prologue, the norm of its rows (five vector instructions a value), its bytes, rows from its L2 and
// weights from HBM (45 KB/us); more rounds than one where there is nothing else.
constexpr Form ln_forms[] = {{16, 4}, {16, 8}, {32, 3}, {32, 6}, {32, 8}};
double ln_time(const Form& f, int M, int64_t wrows, int K) {
  const double rounds = (double)mn_cdiv(form_tiles(f, M, wrows), mn_num_cus());
  return 1.9 + rounds * ((0.25 + 0.05 * f.bm) * K / 1024 + (f.bm * 4 + 32.0 * f.nj) * K / 45e3);
}
// Plain: 2.3 us, and 68 KB/us of its own or 5.3 TB/s of all weights (6.2 past the caches), whichever is longer, and somewhat more where they are near
// each other; one round or nothing.  us, measured / this: 32 x 16 tiles of K = 1024 3.7 / 3.7, 32 x 32 of 1024 4.2 / 4.2, of 4096 9.7 / 10.0, of 8192 15.6 / 17.7, 64 x 32 of 1024 5.0 / 5.2, 64 x 64 of 4096
// 16.6 / 17.7, 64 x 128 of 2048 15.9 / 13.9, of 8192 46.7 / 48.5; hi/lo, 16384 weight rows of 3072 (100 MB): 16 x 64 17.7 .. 18.2 / 19.4, 32 x 64 19.8 .. 20.9 / 20.3, 48 x 64 22.1 .. 23.8 / 21.7.
constexpr Form forms[] = {{32, 1}, {16, 2}, {32, 2}, {32, 4}, {64, 2}, {64, 4}, {64, 8}}, hilo_forms[] = {{16, 2}, {32, 1}, {32, 2}, {32, 4}, {32, 6}, {32, 8}, {64, 4}, {16, 4}, {48, 4}, {48, 6}};
// (hi/lo 48 x 96, the one form whose waves' LDS reads take longer than its bytes, is 1025 rows by 1024 columns in one round: K = 1024 10.3 us, 2752 22.2, 4096 29.0; 64 x 64 tiles, 272 of them, 11.3, 24.2, 32.9)
double own_time(const Form& f, bool hilo, int K) { return (f.bm * (hilo ? 2 : 1) + 16 * f.nj) * (double)K / (hilo && f.bm * f.nj > 256 ? 31e3 : 34e3); }
// One row tile's weights nobody reads again, and where they take longer than all else they stream faster as non-temporal loads (16384 x 3072: 16 rows 20.0 -> 18.2 us, 36 rows 23.3 -> 22.1); smaller
// ones, whose round trips count, do not: 8 rows 1024 x 4096 8.2 -> 9.9, 2304 x 768 3.9 -> 4.5, 26 of 15952 x 320 5.3 -> 6.0.
bool read_once(const Form& f, bool hilo, int M, int64_t wrows, int K) { return hilo && f.bm >= M && wrows * K >= (int64_t)32 << 20 && (double)wrows * K / 2.65e6 > own_time(f, hilo, K); }
double rows_time(const Form& f, bool hilo, int M, int64_t wrows, int K) {
  if (form_tiles(f, M, wrows) > mn_num_cus()) return 1e30;
  const double own = own_time(f, hilo, K), all = (double)wrows * K / (read_once(f, hilo, M, wrows, K) ? 3.1e6 : 2.65e6), hi = fmax(own, all), lo = fmin(own, all);
  return 2.3 + hi + 0.3 * lo * lo * lo / (hi * hi);
}
template <int EPI>
void go_plain(int form, const RowsGemm& p, hipStream_t st) {
  switch (form) {
    case 0: go<EPI, false, false, 32, 1, 8, 6>(p, st); break;
    case 1: go<EPI, false, false, 16, 2, 8, 6>(p, st); break;
    case 2: go<EPI, false, false, 32, 2, 8, 5>(p, st); break;
    case 3: go<EPI, false, false, 32, 4, 8, 3>(p, st); break;
    case 4: go<EPI, false, false, 64, 2, 8, 3>(p, st); break;
    case 5: go<EPI, false, false, 64, 4, 4, 5>(p, st); break;
    default: go<EPI, false, false, 64, 8, 4, 3>(p, st); break;
  }
}
template <int EPI>
void go_hilo(int form, const RowsGemm& p, hipStream_t st) {
  switch (form) {
    case 0: go<EPI, false, true, 16, 2, 8, 5>(p, st); break;
    case 1: go<EPI, false, true, 32, (EPI == R_SWIGLU_SPLIT ? 2 : 1), 8, 3>(p, st); break;
    case 2: go<EPI, false, true, 32, 2, 8, 3>(p, st); break;
    case 3: go<EPI, false, true, 32, 4, 4, 5>(p, st); break;
    case 4: go<EPI, false, true, 32, 6, 4, 4>(p, st); break;
    case 5: go<EPI, false, true, 32, 8, 4, 3>(p, st); break;
    case 6: go<EPI, false, true, 64, 4, 4, 3>(p, st); break;
    case 7: go<EPI, false, true, 16, 4, 8, 3>(p, st); break;
    case 8: go<EPI, false, true, 48, 4, 4, 4>(p, st); break;
    default: go<EPI, false, true, 48, 6, 4, 3>(p, st); break;
  }
}

bool shape_ok(const void* A, int64_t lda, const void* W, int64_t ldw, int64_t wrows, const void* bias, const void* C, int64_t ldc, int M, int N, int K) {
  return M >= 1 && N >= 4 && N % 4 == 0 && K >= 64 && K % 64 == 0 && lda % 8 == 0 && ldw % 8 == 0 && ldc % 4 == 0 && (((uintptr_t)A | (uintptr_t)W | (uintptr_t)C) & 15) == 0 &&
         ((uintptr_t)bias & 7) == 0 && lda >= 0 && ldw >= 0 && ((int64_t)M * lda + K) * 2 < ((int64_t)1 << 32) && (wrows * ldw + K) * 2 < ((int64_t)1 << 32);      // (offsets of 32 bits)
}

}  // namespace

// Whether the two products below take the rows of a block stack: where the widest tiles make one round of the CUs, for 256 rows at most.  us a block, the 64 x 64 tiles and
// the launches between them / these (bf16, cold weights): dim 768, hidden 2048 SwiGLU: 5 rows 30.9 / 24.2, 65 34.7 / 27.8, 130 36.9 / 31.5, 256 39.9 / 36.8, in two rounds
// 260 40.5 / 42.4; 1024, 2752 SwiGLU: 65 40.8 / 34.5, 130 43.9 / 40.9, in two rounds 196 48.3 / 52.1; 1024, 4096 GELU: 65 43.0 / 36.2, 256 50.4 / 48.8, 260 54.3 / 60.8.
extern "C" int mn_vit_rows_ok(int M, int dim, int hidden, int gelu) {
  if (M < 1 || M > 256 || dim < 256 || dim > KMAX || dim % 256 || hidden < 64 || hidden % 64) return 0;
  const int64_t up = (int64_t)hidden * (gelu ? 1 : 2), wide = up > 3 * (int64_t)dim ? up : 3 * (int64_t)dim;
  return mn_cdiv(M, 32) * mn_cdiv(wide, 128) <= mn_num_cus();
}

extern "C" int mn_ln_gemm_rows(const float* x, int64_t ldx, const uint16_t* g, const uint16_t* b, float eps, const uint16_t* W, int64_t ldw, const uint16_t* bias, int gelu, int pair,
                               uint16_t* C, int64_t ldc, int M, int N, int K, void* stream) {
  MN_CHECK_ARG(x && g && b && W && C && K <= KMAX && K % 256 == 0 && ldx % 4 == 0 && shape_ok(x, 0, W, ldw, pair ? 2 * (int64_t)N : N, bias, C, ldc, M, N, K) &&
                   (((uintptr_t)g | (uintptr_t)b) & 7) == 0 && !(gelu && pair), "mn_ln_gemm_rows: bad args");
  RowsGemm p{};
  p.x = x; p.ldx = ldx; p.g = g; p.b = b; p.eps = eps; p.W = W; p.ldw = ldw; p.bias = bias; p.pair = pair ? N : 0; p.C = C; p.ldc = ldc; p.M = M; p.N = N; p.K = K;
  hipStream_t st = mn_stream(stream);
#define GO(E)                                                                              \
  switch (best_form(ln_forms, [&](const Form& f) { return ln_time(f, M, pair ? 2 * (int64_t)N : N, K); }, nullptr)) {          \
    case 0: go<E, true, false, 16, 4, 8, 4>(p, st); break;                                        \
    case 1: go<E, true, false, 16, 8, 4, 4>(p, st); break;                                        \
    case 2: go<E, true, false, 32, 3, 8, 4>(p, st); break;                                        \
    case 3: go<E, true, false, 32, 6, 4, 4>(p, st); break;                                        \
    default: go<E, true, false, 32, 8, 4, 3>(p, st); break;                                       \
  }
  if (pair) { GO(R_SWIGLU) } else if (gelu) { GO(R_GELU) } else { GO(R_BF16) }
#undef GO
  MN_CHECK_LAUNCH("mn_ln_gemm_rows");
  return MN_OK;
}

extern "C" int mn_resid_gemm_rows(const uint16_t* A, int64_t lda, const uint16_t* W, int64_t ldw, const uint16_t* bias, float* x, int64_t ldx, int M, int N, int K, void* stream) {
  MN_CHECK_ARG(A && W && x && shape_ok(A, lda, W, ldw, N, bias, x, ldx, M, N, K), "mn_resid_gemm_rows: bad args");
  RowsGemm p{};
  p.A = A; p.lda = lda; p.W = W; p.ldw = ldw; p.bias = bias; p.C = x; p.ldc = ldx; p.M = M; p.N = N; p.K = K;
  double us;
  int form = best_form(forms, [&](const Form& f) { return rows_time(f, false, M, N, K); }, &us);
  if (us >= 1e30) form = 6;                              // more than one round of the largest
  go_plain<R_RESID>(form, p, mn_stream(stream));
  MN_CHECK_LAUNCH("mn_resid_gemm_rows");
  return MN_OK;
}

// One dense product of gemm256.hip, of tile_us on its tiles by its estimate: taken (1) where a form here is estimated a tenth faster (3 % where it reads weights past the caches, which the tiles'
// estimate takes them not to), else 0 and nothing is launched.
// us, the tiles / these, cold weights, 40, 101, 256 and 600 rows: hi/lo 768 -> 768 7.5 / 3.8, 7.8 / 3.9, 7.9 / 4.7, 8.1 / 6.0; 2048 -> 768 15.3 / 5.9, 15.5 / 6.0, 15.7 / 7.1, 15.9 / 10.6;
// 768 -> 2304 7.7 / 4.1, 7.9 / 5.8, 8.4 / 6.8, tiles; 4096 -> 1024 27.3 / 8.5, 27.9 / 8.8, 27.6 / 11.8, 28.4 / 21.8; 1024 -> 2 x 2752 gated 10.4 / 8.1, 10.5 / 9.4, tiles (14.1).  Plain rows, 70, 250, 450 and
// 1000: 1024 -> 1024 6.9 / 3.8, 6.9 / 4.5, 7.1 / 5.6, tiles (7.4); 2048 -> 2048 10.5 / 6.1, 10.9 / 7.7, 11.2 / 10.5, 17.4 / 16.0; 8192 -> 2048 34.0 / 16.3, 36.7 / 25.9, 36.7 / 31.7, 57.9 / 51.4; 1024 -> 4096
// 7.0 / 5.5, tiles (7.4).  Gated products of fewer than 512 values stay (26 rows 320 -> 2 x 7976 5.3 / 5.7).  The error is smaller throughout (eight sums of K / 8, or four of K / 4: 1.0e-7 for 1.9e-7 of 64 bits at K = 2048).
extern "C" int mn_rows_gemm(const mn_g256* a, int epi, double tile_us, void* stream) {
  const bool hilo = a->a_lo_off != 0, paired = epi == MN_G256_SWIGLU_SPLIT;
  const bool known = epi == MN_G256_F32 || epi == MN_G256_F32_RESID || (hilo ? epi == MN_G256_BF16_SPLIT || paired : epi == MN_G256_BF16);
  const int64_t wrows = paired ? a->w_pair_rows + a->N : a->N, rows = paired ? 2 * (int64_t)a->N : a->N;
  if (!known || !(hilo || a->k_parts) || (paired && a->K < 512) || a->g_off || a->a_rows || a->f8 || (a->w_pair_rows != 0) != paired ||
      ((uintptr_t)a->C & (epi == MN_G256_F32 || epi == MN_G256_F32_RESID ? 15 : 7)) || a->c_lo_off % 4 || a->w_pair_rows % 4 ||
      !shape_ok(a->A, a->lda, a->W, a->ldw, wrows, a->bias, nullptr, a->ldc, a->M, a->N, a->K) || ((int64_t)a->M * a->lda + a->a_lo_off + a->K) * 2 >= ((int64_t)1 << 32) || a->a_lo_off < 0 || a->a_lo_off % 8)
    return 0;
  double us;
  const auto time = [&](const Form& f) { return (paired && f.nj == 1) ? 1e30 : rows_time(f, hilo, a->M, rows, a->K); };
  const int form = hilo ? best_form(hilo_forms, time, &us) : best_form(forms, time, &us);
  const bool once = hilo && read_once(hilo_forms[form], true, a->M, rows, a->K);
  if (us >= (once ? 0.97 : 0.9) * tile_us) return 0;
  RowsGemm p{};
  p.once = once;
  p.A = a->A; p.lda = a->lda; p.a_lo = a->a_lo_off; p.W = a->W; p.ldw = a->ldw; p.bias = a->bias; p.pair = a->w_pair_rows; p.C = a->C; p.ldc = a->ldc; p.c_lo = a->c_lo_off;
  p.M = a->M; p.N = a->N; p.K = a->K;
  hipStream_t st = mn_stream(stream);
  switch (epi) {
    case MN_G256_F32: hilo ? go_hilo<R_F32>(form, p, st) : go_plain<R_F32>(form, p, st); break;
    case MN_G256_F32_RESID: hilo ? go_hilo<R_RESID>(form, p, st) : go_plain<R_RESID>(form, p, st); break;
    case MN_G256_BF16: go_plain<R_BF16>(form, p, st); break;
    case MN_G256_BF16_SPLIT: go_hilo<R_SPLIT>(form, p, st); break;
    default: go_hilo<R_SWIGLU_SPLIT>(form, p, st); break;
  }
  return 1;
}
