// decode_ops.hip — small-row (decode) operators around the skinny GEMM (gfx950):
//   mn_moe_router       RMSNorm + gate GEMV + softmax + top-k (+ image-gate override)
//   mn_rope_kv_append   neox-style rotary on q/k, append k/v to the fp32 KV cache
//   mn_attn_decode      masked GQA/MHA attention of <= 8 query rows against the cache
//                       (split over the key range = flash-decoding, then a combine pass)
// All of these are HBM/latency-bound index-and-reduce work: coalesced loads, wave shuffles,
// no MFMA.
#include <string.h>

#include "common.h"

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// -------------------------------------------------------------------------------------------
// MoE router = gate logits (skinny GEMV with a fused RMSNorm prologue, all CUs) + this kernel:
// one 256-thread block per row writes the normalised row (input of the experts) and wave 0 does
// the fp32 softmax + iterative arg-max top-k + renormalisation.
//
// TIE RULE (topk_round in common.h, which every router of this library goes by: this kernel, moe_router_row_kernel below, moe_gate_up.hip,
// moe_topk_logits_kernel in prefill_ops.hip and the wide route's top-k in wide_llm.inl): expert e lives in lane e; a round takes the
// wave maximum and `__ffsll(__ballot(cur == best))`, i.e. among EQUAL scores the LOWEST expert id wins, and the picked slots are in
// descending score / ascending id order; a row of NaN scores gets experts 0 .. top_k - 1 with NaN weights.  The reference calls `torch.topk` (modeling_bailing_moe.py:512), whose order among equal
// values is unspecified; exact ties need two identical gate rows (fp32 scores of real weights tie with probability zero).
// Pinned by tests/test_gpu_router_ties.py.
// -------------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void moe_topk_kernel(
    const float* __restrict__ x, int64_t ldx, const bf16_t* __restrict__ norm_w, float eps,
    const float* __restrict__ logits_text, const float* __restrict__ logits_image,
    const uint8_t* __restrict__ image_mask, int H, int E, int top_k, int norm_topk_prob, int n_shared,
    float* __restrict__ x_norm, int32_t* __restrict__ topk_idx, float* __restrict__ topk_w) {
  __shared__ float red[8];
  const int m = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const float* xr = x + (int64_t)m * ldx;
  float ss = 0.f;
  for (int k = tid; k < H; k += 256) { float v = xr[k]; ss += v * v; }
  ss = block_sum(ss, red);
  const float rstd = rsqrtf(ss / (float)H + eps);
  for (int k = tid; k < H; k += 256) x_norm[(int64_t)m * H + k] = xr[k] * rstd * bf16_to_f32(norm_w[k]);
  if (wave == 0) {
    const float* lg = (image_mask && logits_image && image_mask[m]) ? logits_image : logits_text;
    // softmax over E (fp32) then iterative arg-max; ties -> lowest expert index
    float s = lane < E ? lg[(int64_t)m * E + lane] : -INFINITY;
    const float mx = wave_max(s);
    float p = lane < E ? __expf(s - mx) : 0.f;
    const float denom = wave_sum(p);
    p = p / denom;
    float cur = lane < E ? p : -1.f;
    float wsum = 0.f;
    float myw = 0.f;
    int myidx = 0;
    const int n_slot = top_k + n_shared;
    for (int k = 0; k < top_k; ++k) {
      float best;
      const int sel = topk_round(cur, E, k, best);
      if (lane == k) { myw = best; myidx = sel; }
      wsum += best;
    }
    if (lane < top_k) {
      topk_idx[(int64_t)m * n_slot + lane] = myidx;
      topk_w[(int64_t)m * n_slot + lane] = (norm_topk_prob && top_k > 1) ? myw / wsum : myw;
    } else if (lane < n_slot) {
      topk_idx[(int64_t)m * n_slot + lane] = E + (lane - top_k);
      topk_w[(int64_t)m * n_slot + lane] = 1.0f;
    }
  }
}

// Few rows (text decode, one image): the whole router in ONE launch — a 1024-thread workgroup per row does the RMSNorm, the gate
// GEMV of that row's own gate (image rows read image_gate only; 64 x H bf16 = 256 KB from L2, four experts per wave), and wave 0
// the softmax / top-k.  Replaces a 16-workgroup GEMV launch (9 us) + moe_topk_kernel (5 us) per layer.
__global__ __launch_bounds__(1024) void moe_router_row_kernel(
    const float* __restrict__ x, int64_t ldx, const bf16_t* __restrict__ norm_w, float eps, const bf16_t* __restrict__ gate_w,
    const bf16_t* __restrict__ image_gate_w, const uint8_t* __restrict__ image_mask, int M, int H, int E, int top_k,
    int norm_topk_prob, int n_shared, float* __restrict__ x_norm, int32_t* __restrict__ topk_idx, float* __restrict__ topk_w,
    float* __restrict__ logits_out, const float* __restrict__ P, int nz, int64_t slab, float* __restrict__ h_out, bf16_t* __restrict__ Y) {
  __shared__ __attribute__((aligned(16))) float xs[4096];
  __shared__ float red[16];
  __shared__ float lg[64];
  typedef uint32_t u4 __attribute__((ext_vector_type(4)));
  const int m = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const float* xr = x + (int64_t)m * ldx;
  const bool img = image_mask && image_gate_w && image_mask[m];
  const bf16_t* G = img ? image_gate_w : gate_w;
  typedef float f4 __attribute__((ext_vector_type(4)));
  typedef float f2 __attribute__((ext_vector_type(2)));
  float acc[4] = {0.f, 0.f, 0.f, 0.f};          // experts wave, wave + 16, wave + 32, wave + 48: four weight rows in flight per lane
  // H <= 2048 (the 16B-A3B width): this lane's 16 weight slots do not depend on x — requested FIRST, so the launch is one memory round
  // trip (x and the gate rows together) + the reductions, not two dependent ones
  const bool pre = H <= 2048 && (H % 512) == 0;
  u4 gw[4][4];
  if (pre) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int e = wave + 16 * j, k = lane * 8 + 512 * i;
        gw[i][j] = u4{0u, 0u, 0u, 0u};
        if (e < E && k < H) gw[i][j] = *reinterpret_cast<const u4*>(G + (int64_t)e * H + k);
      }
  }
  // P != NULL (the decoder chain, up to 64 rows): the row is h + the sum of the nz K-slice partial slabs of the attention output projection (the slabs first, in slab order, as
  // llm_glue_kernel does), written back to h_out — the residual glue launch and the gate launch fold into this one.  Two columns a thread, the norm's weights with them: all that
  // the row needs is asked for before the first of it is waited for (sixteen slabs at once, one round trip).
  f2 xv[2] = {{0.f, 0.f}, {0.f, 0.f}}, add[2] = {{0.f, 0.f}, {0.f, 0.f}};     // H <= 4096: columns 2 tid, 2 tid + 2048
  uint32_t nw[2] = {0u, 0u};
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int k = 2 * tid + 2048 * i;
    if (k >= H) continue;
    xv[i] = f2{xr[k], xr[k + 1]};
    nw[i] = (uint32_t)norm_w[k] | (uint32_t)norm_w[k + 1] << 16;
  }
  if (P) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int k = 2 * tid + 2048 * i;
      if (k >= H) continue;
      const float* pp = P + (int64_t)m * H + k;
      for (int z0 = 0; z0 < nz; z0 += 16) {
        f2 t[16];
#pragma unroll
        for (int j = 0; j < 16; ++j) t[j] = z0 + j < nz ? *reinterpret_cast<const f2*>(pp + (int64_t)(z0 + j) * slab) : f2{0.f, 0.f};
#pragma unroll
        for (int j = 0; j < 16; ++j) add[i] += t[j];
      }
    }
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int k = 2 * tid + 2048 * i;
    if (k >= H) continue;
    xv[i] += add[i];                              // (the small sum first: the stream is rounded once)
    if (P) *reinterpret_cast<f2*>(h_out + (int64_t)m * H + k) = xv[i];
    ss += xv[i].x * xv[i].x + xv[i].y * xv[i].y;
  }
  ss = block_sum(ss, red);
  const float rstd = rsqrtf(ss / (float)H + eps);
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int k = 2 * tid + 2048 * i;
    if (k >= H) continue;
    const f2 v = f2{xv[i].x * rstd * bf16lo_to_f32(nw[i]), xv[i].y * rstd * bf16hi_to_f32(nw[i])};
    *reinterpret_cast<f2*>(&xs[k]) = v;
    if (x_norm) *reinterpret_cast<f2*>(x_norm + (int64_t)m * H + k) = v;
    if (Y) {                                      // the grouped experts' operand: hi rows, then lo rows
      uint32_t hi, lo;
      split_pk_bf16(v.x, v.y, hi, lo);
      *reinterpret_cast<uint32_t*>(Y + (int64_t)m * H + k) = hi;
      *reinterpret_cast<uint32_t*>(Y + (int64_t)(M + m) * H + k) = lo;
    }
  }
  __syncthreads();
  if (pre) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int k = lane * 8 + 512 * i;
      if (k < H) {
        const f4 xa = *reinterpret_cast<const f4*>(&xs[k]), xb = *reinterpret_cast<const f4*>(&xs[k + 4]);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const u4 wv = gw[i][j];
          float a = acc[j];
          a = fmaf(bf16lo_to_f32(wv.x), xa.x, a); a = fmaf(bf16hi_to_f32(wv.x), xa.y, a);
          a = fmaf(bf16lo_to_f32(wv.y), xa.z, a); a = fmaf(bf16hi_to_f32(wv.y), xa.w, a);
          a = fmaf(bf16lo_to_f32(wv.z), xb.x, a); a = fmaf(bf16hi_to_f32(wv.z), xb.y, a);
          a = fmaf(bf16lo_to_f32(wv.w), xb.z, a); a = fmaf(bf16hi_to_f32(wv.w), xb.w, a);
          acc[j] = a;
        }
      }
    }
  } else
  for (int k = lane * 8; k < H; k += 512) {
    const f4 xa = *reinterpret_cast<const f4*>(&xs[k]), xb = *reinterpret_cast<const f4*>(&xs[k + 4]);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int e = wave + 16 * j;
      if (e < E) {
        const u4 wv = *reinterpret_cast<const u4*>(G + (int64_t)e * H + k);
        float a = acc[j];
        a = fmaf(bf16lo_to_f32(wv.x), xa.x, a); a = fmaf(bf16hi_to_f32(wv.x), xa.y, a);
        a = fmaf(bf16lo_to_f32(wv.y), xa.z, a); a = fmaf(bf16hi_to_f32(wv.y), xa.w, a);
        a = fmaf(bf16lo_to_f32(wv.z), xb.x, a); a = fmaf(bf16hi_to_f32(wv.z), xb.y, a);
        a = fmaf(bf16lo_to_f32(wv.w), xb.z, a); a = fmaf(bf16hi_to_f32(wv.w), xb.w, a);
        acc[j] = a;
      }
    }
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float t = wave_sum(acc[j]);
    if (lane == 0 && wave + 16 * j < E) lg[wave + 16 * j] = t;
  }
  __syncthreads();
  if (wave == 0) {
    // softmax over E (fp32) then iterative arg-max; ties -> lowest expert index  (BailingMoeGate.forward :505-520)
    float s = lane < E ? lg[lane] : -INFINITY;
    if (lane < E) logits_out[((int64_t)(img ? 1 : 0) * M + m) * E + lane] = s;
    const float mx = wave_max(s);
    float p = lane < E ? __expf(s - mx) : 0.f;
    const float denom = wave_sum(p);
    p = p / denom;
    float cur = lane < E ? p : -1.f, wsum = 0.f, myw = 0.f;
    int myidx = 0;
    const int n_slot = top_k + n_shared;
    for (int k = 0; k < top_k; ++k) {
      float best;
      const int sel = topk_round(cur, E, k, best);
      if (lane == k) { myw = best; myidx = sel; }
      wsum += best;
    }
    if (lane < top_k) {
      topk_idx[(int64_t)m * n_slot + lane] = myidx;
      topk_w[(int64_t)m * n_slot + lane] = (norm_topk_prob && top_k > 1) ? myw / wsum : myw;
    } else if (lane < n_slot) {
      topk_idx[(int64_t)m * n_slot + lane] = E + (lane - top_k);
      topk_w[(int64_t)m * n_slot + lane] = 1.0f;
    }
  }
}

static int g_router_rows = 4;      // rows up to which mn_moe_router runs as one launch (A/B hook: mn_moe_router_tune)
#ifdef MN_DEV_HOOKS
extern "C" MN_DEV_API void mn_moe_router_tune(int max_rows) { g_router_rows = max_rows; }
#endif

// The decoder chain's form (engine.hip): h[m] += sum of the nz partial slabs P [nz][M][H]; RMSNorm -> x_norm and / or Y (bf16 hi rows, lo rows); gate;
// top-k — one launch.  A row is a workgroup, which reads the gate (256 KB at 64 x 2048) and its slabs (131 KB) from its XCD's L2: 10.7 us at 64 rows (11.8 with eight slabs a round
// trip and the norm's weights behind the sum; 2 rows 11.0 -> 9.9), where the norm, the gate's product and a one-workgroup top-k and sort took 6 + 5 + 13.
bool moe_router_rows_ok(int M, int H, int E) { return M >= 1 && M <= 64 && H <= 4096 && (H % 8) == 0 && E <= 64; }
int moe_router_rows(float* h, const float* P, int nz, const uint16_t* norm_w, float eps, const uint16_t* gate_w, const uint16_t* image_gate_w, const uint8_t* image_mask, int M,
                    int H, int E, int top_k, int norm_topk_prob, int n_shared_slots, float* x_norm, uint16_t* y, int32_t* topk_idx, float* topk_w, float* logits_ws, void* stream) {
  MN_CHECK_ARG(h && P && norm_w && gate_w && (x_norm || y) && topk_idx && topk_w && logits_ws && moe_router_rows_ok(M, H, E) && top_k >= 1 && top_k <= E &&
               top_k + n_shared_slots <= 64, "moe_router_rows: bad args");
  hipLaunchKernelGGL(moe_router_row_kernel, dim3(M), dim3(1024), 0, mn_stream(stream), (const float*)h, (int64_t)H, norm_w, eps, gate_w,
                     image_gate_w, image_mask, M, H, E, top_k, norm_topk_prob, n_shared_slots, x_norm, topk_idx, topk_w, logits_ws, P, nz, (int64_t)M * H, h, y);
  MN_CHECK_LAUNCH("moe_router_rows");
  return MN_OK;
}

extern "C" int mn_moe_router(const float* x, int64_t ldx, const uint16_t* norm_w, float eps,
                             const uint16_t* gate_w, const uint16_t* image_gate_w, const uint8_t* image_mask,
                             int M, int H, int E, int top_k, int norm_topk_prob, int n_shared_slots,
                             float* x_norm, int32_t* topk_idx, float* topk_w, float* logits_ws, void* ws, size_t ws_bytes,
                             void* stream) {
  MN_CHECK_ARG(M >= 1 && M <= 64 && H >= 8 && (H % 8) == 0, "mn_moe_router: bad M=%d H=%d", M, H);
  MN_CHECK_ARG(E >= 1 && E <= 64 && top_k >= 1 && top_k <= E && top_k + n_shared_slots <= 64,
               "mn_moe_router: bad E=%d top_k=%d", E, top_k);
  MN_CHECK_ARG(x && norm_w && gate_w && x_norm && topk_idx && topk_w && logits_ws, "mn_moe_router: null pointer");
  const bool both = image_mask && image_gate_w;
  if (M <= g_router_rows && H <= 4096) {
    hipLaunchKernelGGL(moe_router_row_kernel, dim3(M), dim3(1024), 0, mn_stream(stream), x, ldx, norm_w, eps, gate_w, image_gate_w,
                       image_mask, M, H, E, top_k, norm_topk_prob, n_shared_slots, x_norm, topk_idx, topk_w, logits_ws,
                       (const float*)nullptr, 0, (int64_t)0, (float*)nullptr, (bf16_t*)nullptr);
    MN_CHECK_LAUNCH("mn_moe_router");
    return MN_OK;
  }
  // >= 5 rows with scratch: one launch on the matrix-core route; otherwise the fp32 path, 8 rows at a time
  const bool mfma = M <= 64 && ws != nullptr && ws_bytes >= mn_skinny_workspace_bytes(M, E, H, 0) && mn_skinny_workspace_bytes(M, E, H, 0) > 0;
  const int mstep = mfma ? M : 8;
  for (int gsel = 0; gsel < (both ? 2 : 1); ++gsel)
    for (int m0 = 0; m0 < M; m0 += mstep) {
      mn_skinny_args a;
      memset(&a, 0, sizeof(a));
      a.x = x + (int64_t)m0 * ldx; a.ldx = ldx; a.w = gsel ? image_gate_w : gate_w; a.ldw = H;
      a.out = logits_ws + (int64_t)gsel * M * E + (int64_t)m0 * E; a.ldo = E;
      a.M = (M - m0) < mstep ? (M - m0) : mstep; a.N = E; a.K = H;
      a.prologue = MN_PRO_RMSNORM; a.ln_g = norm_w; a.eps = eps;
      if (mfma) { a.ws = ws; a.ws_bytes = ws_bytes; }
      const int rc = mn_skinny_gemm(&a, stream);
      if (rc != MN_OK) return rc;
    }
  hipLaunchKernelGGL(moe_topk_kernel, dim3(M), dim3(256), 0, mn_stream(stream), x, ldx, norm_w, eps, logits_ws,
                     both ? logits_ws + (int64_t)M * E : nullptr, image_mask, H, E, top_k, norm_topk_prob,
                     n_shared_slots, x_norm, topk_idx, topk_w);
  MN_CHECK_LAUNCH("mn_moe_router");
  return MN_OK;
}

// One rotary pair.  The products are rounded before they are added (no contraction), like the rotation they stand for: what a fused form
// would round once less depends on which of the two products the compiler folds in.
__device__ __forceinline__ void rotate_pair(float& x1, float& x2, float c, float s) {
#pragma clang fp contract(off)
  const float a = x1 * c, b = x2 * s, d = x2 * c, e = x1 * s;
  x1 = a - b;
  x2 = d + e;
}

// -------------------------------------------------------------------------------------------
// RoPE + KV append. grid (M, n_q + 2*n_kv), block hd/2 threads.
// -------------------------------------------------------------------------------------------
// nz > 1: qkv is a stack of nz K-slice partial slabs (slab elements apart) of the QKV projection, summed here — the
// reduction of the streaming GEMM folded into the consumer (no bias: use_qkv_bias is false on this path).
__global__ void rope_kv_append_kernel(const float* __restrict__ qkv, int64_t ldqkv, int nz, int64_t slab, int n_q, int n_kv, int hd,
                                      int rope, const float* __restrict__ cos_tab, const float* __restrict__ sin_tab,
                                      const int32_t* __restrict__ row_seq, const int32_t* __restrict__ row_slot,
                                      const int32_t* __restrict__ row_pos, int M, int sec_t, int sec_h, float q_scale,
                                      float* __restrict__ q_out, float* __restrict__ kv_cache, int64_t t_max, int round_kv) {
  const int m = blockIdx.x, h = blockIdx.y, i = threadIdx.x, half = hd >> 1;
  const float* src = qkv + (int64_t)m * ldqkv + (int64_t)h * hd;
  float x1 = 0.f, x2 = 0.f;
  for (int z0 = 0; z0 < nz; z0 += 8) {              // eight slabs' loads in flight (one by one: nz dependent round trips)
    float a1[8], a2[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      a1[j] = z0 + j < nz ? src[(int64_t)(z0 + j) * slab + i] : 0.f;
      a2[j] = z0 + j < nz ? src[(int64_t)(z0 + j) * slab + i + half] : 0.f;
    }
    for (int j = 0; j < 8; ++j) x1 += a1[j];                    // (the one-by-one loop's order: same bits)
    for (int j = 0; j < 8; ++j) x2 += a2[j];
  }
  const bool is_q = h < n_q, is_k = !is_q && h < n_q + n_kv;
  if (rope && (is_q || is_k)) {
    // 3D rotary (sec_t > 0): row_pos is [3][M] = t, h, w positions; frequency i of each half follows the t stream for
    // i < sec_t, the h stream for the next sec_h, the w stream for the rest (apply_multimodal_rotary_pos_emb, :463-469)
    const int stream = sec_t <= 0 ? 0 : (i < sec_t ? 0 : (i < sec_t + sec_h ? 1 : 2));
    const int pos = row_pos[stream * M + m];
    const float c = cos_tab[(int64_t)pos * half + i], s = sin_tab[(int64_t)pos * half + i];
    rotate_pair(x1, x2, c, s);
  }
  if (is_q) {
    float* dst = q_out + (int64_t)m * n_q * hd + (int64_t)h * hd;
    dst[i] = x1 * q_scale;
    dst[i + half] = x2 * q_scale;
  } else {
    const int kvh = is_k ? h - n_q : h - n_q - n_kv;
    const int64_t seq = row_seq[m], slot = row_slot[m];
    if ((uint64_t)slot >= (uint64_t)t_max) return;      // never write outside the sequence's arena rows (the host raises before a cache fills up)
    float* dst = kv_cache + (((seq * 2 + (is_k ? 0 : 1)) * n_kv + kvh) * t_max + slot) * hd;
    if (round_kv) {     // measurement only (dev library, tests/measure/kv_bf16_error.py): what a bf16 KV cache would hold
      x1 = bf16_to_f32(f32_to_bf16(x1));
      x2 = bf16_to_f32(f32_to_bf16(x2));
    }
    dst[i] = x1;
    dst[i + half] = x2;
  }
}

static int g_kv_round_bf16 = 0;
#ifdef MN_DEV_HOOKS
extern "C" MN_DEV_API void mn_kv_round_bf16(int on) { g_kv_round_bf16 = on; }
#endif

// Internal (engine.hip): as mn_rope_kv_append_3d, reading the QKV projection as nz partial slabs.
extern "C" int mn_rope_kv_from_partials(const float* qkv, int64_t ldqkv, int nz, int64_t slab, int M, int n_q, int n_kv, int hd,
                                        int rope, const float* cos_tab, const float* sin_tab, const int32_t* row_seq,
                                        const int32_t* row_slot, const int32_t* row_pos, int sec_t, int sec_h, float q_scale,
                                        float* q_out, float* kv_cache, int64_t t_max, void* stream) {
  MN_CHECK_ARG(M >= 1 && n_q >= 1 && n_kv >= 1 && (hd == 64 || hd == 128) && nz >= 1, "mn_rope_kv_append: bad shape");
  MN_CHECK_ARG(qkv && row_seq && row_slot && q_out && kv_cache, "mn_rope_kv_append: null pointer");
  MN_CHECK_ARG(!rope || (cos_tab && sin_tab && row_pos), "mn_rope_kv_append: rope needs tables and positions");
  MN_CHECK_ARG(sec_t >= 0 && sec_h >= 0 && sec_t + sec_h <= hd / 2, "mn_rope_kv_append: bad rotary sections %d/%d", sec_t, sec_h);
  hipLaunchKernelGGL(rope_kv_append_kernel, dim3(M, n_q + 2 * n_kv), dim3(hd / 2), 0, mn_stream(stream), qkv, ldqkv, nz, slab,
                     n_q, n_kv, hd, rope, cos_tab, sin_tab, row_seq, row_slot, row_pos, M, sec_t, sec_h, q_scale, q_out,
                     kv_cache, t_max, g_kv_round_bf16);
  MN_CHECK_LAUNCH("mn_rope_kv_append");
  return MN_OK;
}

extern "C" int mn_rope_kv_append_3d(const float* qkv, int64_t ldqkv, int M, int n_q, int n_kv, int hd, int rope,
                                    const float* cos_tab, const float* sin_tab, const int32_t* row_seq,
                                    const int32_t* row_slot, const int32_t* row_pos, int sec_t, int sec_h, float q_scale,
                                    float* q_out, float* kv_cache, int64_t t_max, void* stream) {
  return mn_rope_kv_from_partials(qkv, ldqkv, 1, 0, M, n_q, n_kv, hd, rope, cos_tab, sin_tab, row_seq, row_slot, row_pos, sec_t,
                                  sec_h, q_scale, q_out, kv_cache, t_max, stream);
}

extern "C" int mn_rope_kv_append(const float* qkv, int64_t ldqkv, int M, int n_q, int n_kv, int hd, int rope,
                                 const float* cos_tab, const float* sin_tab, const int32_t* row_seq,
                                 const int32_t* row_slot, const int32_t* row_pos, float q_scale, float* q_out,
                                 float* kv_cache, int64_t t_max, void* stream) {
  return mn_rope_kv_append_3d(qkv, ldqkv, M, n_q, n_kv, hd, rope, cos_tab, sin_tab, row_seq, row_slot, row_pos, 0, 0, q_scale,
                              q_out, kv_cache, t_max, stream);
}

// -------------------------------------------------------------------------------------------
// Decode attention, split over keys. One wave per (row, q head, split); 4 waves per block
// cover 4 consecutive q heads (= one GQA group when n_q/n_kv == 4, so K/V lines are shared in L1).
// partial layout: [M][n_q][S][HD + 2]  (acc[HD], m, l)
// -------------------------------------------------------------------------------------------
// A row of up to 16 splits' keys is split that finely; a longer one into 16 or splits of four times the keys, 31 at most (with the counters they fit the scratch of 32 splits): us a layer of a
// step of one row, 16 splits at most / these: 4000 keys 34.0 / 34.0, 16000 55.9 / 47.2, 31000 77.5 / 58.9.
constexpr int JOIN_SHORT = 16, JOIN_LONG = 4, JOIN_MOST = 31, JOIN_ROWS = 128;
static_assert(JOIN_MOST <= 64, "a lane a split");
// What mn_attn_decode_fused's launch takes instead of q: the RAW QKV projection; the rotary embedding of the row's q and new k, the q scale and the K / V append of the new token
// happen in the attention launch.
struct AttnFuse {
  const float* qkv; int64_t ldqkv; int nz; int64_t slab;        // raw QKV rows [(n_q + 2 n_kv) * HD], optionally nz K-slice partial slabs
  int rope; const float* cos_tab; const float* sin_tab;          // [n_pos, HD / 2]
  const int32_t* row_slot; const int32_t* row_pos; int sec_t, sec_h; float q_scale; int M;
  float* kv_cache_w;                                              // the arena, writable
};

template <int HD>
__global__ __launch_bounds__(256) void attn_decode_split_kernel(
    const float* __restrict__ q, int n_q, int n_kv, const float* __restrict__ kv_cache, int64_t t_max,
    const int32_t* __restrict__ row_seq, const int32_t* __restrict__ row_len, const uint8_t* __restrict__ key_mask,
    int64_t ld_mask, int S, int chunk_cap, float* __restrict__ partial) {
  extern __shared__ __attribute__((aligned(16))) float sm[];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int m = blockIdx.x, s = blockIdx.z;
  const int h_raw = blockIdx.y * 4 + wave;
  const bool active = h_raw < n_q;          // inactive waves shadow the last head, store nothing
  const int h = active ? h_raw : n_q - 1;
  float* sc = sm + wave * chunk_cap;
  const int len = row_len[m];
  int chunk = (len + S - 1) / S;
  chunk = (chunk + 3) & ~3;
  const int j0 = s * chunk, j1 = min(len, j0 + chunk);
  const int kvh = h / (n_q / n_kv);
  const int64_t seq = row_seq[m];
  const float* Kb = kv_cache + ((seq * 2 + 0) * n_kv + kvh) * t_max * HD;
  const float* Vb = kv_cache + ((seq * 2 + 1) * n_kv + kvh) * t_max * HD;
  const float* qr = q + ((int64_t)m * n_q + h) * HD;
  const uint8_t* mk = key_mask ? key_mask + (int64_t)m * ld_mask : nullptr;
  float* out = partial + (((int64_t)m * n_q + h) * S + s) * (HD + 2);

  // ---- scores: 16 lanes per key, 4 keys per wave-iteration
  constexpr int PER = HD / 16;  // floats per lane (8 for 128, 4 for 64)
  const int sub = lane & 15, kq = lane >> 4;
  float qv[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) qv[i] = qr[sub * PER + i];
  float mx = -INFINITY;
  for (int j = j0 + kq; j < j0 + chunk; j += 4) {
    float d = 0.f;
    const bool ok = j < j1;
    if (ok) {
      const float* kr = Kb + (int64_t)j * HD + sub * PER;
#pragma unroll
      for (int i = 0; i < PER; i += 4) {
        const f32x4 kv = *reinterpret_cast<const f32x4*>(kr + i);
        d = fmaf(kv.x, qv[i], d); d = fmaf(kv.y, qv[i + 1], d); d = fmaf(kv.z, qv[i + 2], d); d = fmaf(kv.w, qv[i + 3], d);
      }
    }
    d = row16_sum(d);           // the 16 lanes of a key are one DPP row
    const bool keep = ok && (!mk || mk[j] != 0);
    const float sv = keep ? d : -INFINITY;
    if (sub == 0 && (j - j0) < chunk_cap) sc[j - j0] = sv;
    mx = fmaxf(mx, sv);
  }
  mx = wave_max(mx);
  // ---- softmax numerators
  __syncthreads();
  float l = 0.f;
  const int n = max(0, j1 - j0);
  for (int j = lane; j < n; j += 64) {
    const float p = (mx == -INFINITY) ? 0.f : __expf(sc[j] - mx);
    sc[j] = p;
    l += p;
  }
  l = wave_sum(l);
  __syncthreads();
  // ---- PV: lane owns HD/64 dims
  constexpr int DPL = HD / 64;  // 2 or 1
  float acc[DPL];
#pragma unroll
  for (int i = 0; i < DPL; ++i) acc[i] = 0.f;
  const float* vr = Vb + (int64_t)j0 * HD + lane * DPL;
  int j = 0;
  for (; j + 4 <= n; j += 4) {
    float v[4][DPL];
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int i = 0; i < DPL; ++i) v[u][i] = vr[(int64_t)(j + u) * HD + i];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const float p = sc[j + u];
#pragma unroll
      for (int i = 0; i < DPL; ++i) acc[i] = fmaf(p, v[u][i], acc[i]);
    }
  }
  for (; j < n; ++j) {
    const float p = sc[j];
#pragma unroll
    for (int i = 0; i < DPL; ++i) acc[i] = fmaf(p, vr[(int64_t)j * HD + i], acc[i]);
  }
  if (active) {
#pragma unroll
    for (int i = 0; i < DPL; ++i) out[lane * DPL + i] = acc[i];
    if (lane == 0) { out[HD] = mx; out[HD + 1] = l; }
  }
}

// GQA form from some 40 (row, KV head) pairs on: one wave per (row, KV head, split) serves all G = n_q / n_kv query heads of its group, so every
// K / V line is loaded ONCE per group instead of once per query head (the per-head kernel above re-reads them through L1:
// 4x the load instructions at G = 4).  Same partial layout, same combine kernel.  Block = 4 waves = 4 KV heads of one row.
template <int HD, int G>
__global__ __launch_bounds__(256) void attn_decode_gqa_kernel(
    const float* __restrict__ q, int n_q, int n_kv, const float* __restrict__ kv_cache, int64_t t_max,
    const int32_t* __restrict__ row_seq, const int32_t* __restrict__ row_len, const uint8_t* __restrict__ key_mask,
    int64_t ld_mask, int S, int chunk_cap, float* __restrict__ partial) {
  extern __shared__ __attribute__((aligned(16))) float sm[];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int m = blockIdx.x, s = blockIdx.z;
  const int kvh_raw = blockIdx.y * 4 + wave;
  const bool active = kvh_raw < n_kv;          // inactive waves shadow the last KV head, store nothing
  const int kvh = active ? kvh_raw : n_kv - 1;
  float* sc = sm + (size_t)wave * G * chunk_cap;            // [G][chunk_cap]
  const int len = row_len[m];
  int chunk = (len + S - 1) / S;
  chunk = (chunk + 3) & ~3;
  const int j0 = s * chunk, j1 = min(len, j0 + chunk);
  const int64_t seq = row_seq[m];
  const float* Kb = kv_cache + ((seq * 2 + 0) * n_kv + kvh) * t_max * HD;
  const float* Vb = kv_cache + ((seq * 2 + 1) * n_kv + kvh) * t_max * HD;
  const uint8_t* mk = key_mask ? key_mask + (int64_t)m * ld_mask : nullptr;
  constexpr int PER = HD / 16;                 // floats per lane in the score pass (16 lanes per key)
  const int sub = lane & 15, kq = lane >> 4;
  float qv[G][PER];
#pragma unroll
  for (int g = 0; g < G; ++g)
#pragma unroll
    for (int i = 0; i < PER; ++i) qv[g][i] = q[((int64_t)m * n_q + kvh * G + g) * HD + sub * PER + i];
  float mx[G];
#pragma unroll
  for (int g = 0; g < G; ++g) mx[g] = -INFINITY;
#pragma unroll 2
  for (int j = j0 + kq; j < j0 + chunk; j += 4) {
    float d[G];
#pragma unroll
    for (int g = 0; g < G; ++g) d[g] = 0.f;
    const bool ok = j < j1;
    if (ok) {
      const float* kr = Kb + (int64_t)j * HD + sub * PER;
#pragma unroll
      for (int i = 0; i < PER; i += 4) {
        const f32x4 kv = *reinterpret_cast<const f32x4*>(kr + i);
#pragma unroll
        for (int g = 0; g < G; ++g) {
          d[g] = fmaf(kv.x, qv[g][i], d[g]); d[g] = fmaf(kv.y, qv[g][i + 1], d[g]);
          d[g] = fmaf(kv.z, qv[g][i + 2], d[g]); d[g] = fmaf(kv.w, qv[g][i + 3], d[g]);
        }
      }
    }
    const bool keep = ok && (!mk || mk[j] != 0);
#pragma unroll
    for (int g = 0; g < G; ++g) {
      float v = d[g];
      v = row16_sum(v);         // the 16 lanes of a key are one DPP row
      const float sv = keep ? v : -INFINITY;
      if (sub == 0 && (j - j0) < chunk_cap) sc[g * chunk_cap + (j - j0)] = sv;
      mx[g] = fmaxf(mx[g], sv);
    }
  }
#pragma unroll
  for (int g = 0; g < G; ++g) mx[g] = wave_max(mx[g]);
  __syncthreads();
  const int n = max(0, j1 - j0);
  float l[G];
#pragma unroll
  for (int g = 0; g < G; ++g) {
    float a = 0.f;
    for (int j = lane; j < n; j += 64) {
      const float pj = (mx[g] == -INFINITY) ? 0.f : __expf(sc[g * chunk_cap + j] - mx[g]);
      sc[g * chunk_cap + j] = pj;
      a += pj;
    }
    l[g] = wave_sum(a);
  }
  __syncthreads();
  constexpr int DPL = HD / 64;                 // dims per lane in the PV pass
  float acc[G][DPL];
#pragma unroll
  for (int g = 0; g < G; ++g)
#pragma unroll
    for (int i = 0; i < DPL; ++i) acc[g][i] = 0.f;
  const float* vr = Vb + (int64_t)j0 * HD + lane * DPL;
  int j = 0;
  for (; j + 4 <= n; j += 4) {
    float v[4][DPL];
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int i = 0; i < DPL; ++i) v[u][i] = vr[(int64_t)(j + u) * HD + i];
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const f32x4 pj = *reinterpret_cast<const f32x4*>(sc + g * chunk_cap + j);      // chunk_cap % 4 == 0, j % 4 == 0
      const float pv[4] = {pj.x, pj.y, pj.z, pj.w};
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int i = 0; i < DPL; ++i) acc[g][i] = fmaf(pv[u], v[u][i], acc[g][i]);
    }
  }
  for (; j < n; ++j) {
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const float pj = sc[g * chunk_cap + j];
#pragma unroll
      for (int i = 0; i < DPL; ++i) acc[g][i] = fmaf(pj, vr[(int64_t)j * HD + i], acc[g][i]);
    }
  }
  if (active) {
#pragma unroll
    for (int g = 0; g < G; ++g) {
      float* out = partial + (((int64_t)m * n_q + kvh * G + g) * S + s) * (HD + 2);
#pragma unroll
      for (int i = 0; i < DPL; ++i) out[lane * DPL + i] = acc[g][i];
      if (lane == 0) { out[HD] = mx[g]; out[HD + 1] = l[g]; }
    }
  }
}

// out (fp32 [M, n_q*HD]) and / or split (bf16 [2][M][n_q*HD]: hi rows then lo rows, the next GEMV's MFMA operand)
template <int HD>
__global__ void attn_decode_combine_kernel(const float* __restrict__ partial, int n_q, int S, float* __restrict__ out,
                                           bf16_t* __restrict__ split, int M, const float* __restrict__ kv_cache, int n_kv,
                                           int64_t t_max, const int32_t* __restrict__ row_seq, const int32_t* __restrict__ row_len) {
  const int m = blockIdx.x, h = blockIdx.y, d = threadIdx.x;
  const float* p = partial + (((int64_t)m * n_q + h) * S) * (HD + 2);
  float l = 0.f, acc = 0.f;
  if (S <= 64) {
    // lane s of every wave holds split s: the statistics are one parallel load + wave reductions, and the weighted sum over
    // the splits runs on independent loads (the serial form cost 14 us at 32 splits: 64 dependent round trips to L2)
    const int lane = d & 63;
    float ms = -INFINITY, ls = 0.f;
    if (lane < S) { ms = p[lane * (HD + 2) + HD]; ls = p[lane * (HD + 2) + HD + 1]; }
    const float mx = wave_max(ms);
    const float f = (ms == -INFINITY) ? 0.f : __expf(ms - mx);
    l = wave_sum(f * ls);
    for (int s0 = 0; s0 < S; s0 += 8) {
      float v[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = s0 + j < S ? p[(s0 + j) * (HD + 2) + d] : 0.f;
#pragma unroll
      for (int j = 0; j < 8; ++j) acc = fmaf(lane_f(f, (s0 + j) & 63), v[j], acc);      // uniform source lane: v_readlane, not ds_bpermute
    }
  } else {
    float mx = -INFINITY;
    for (int s = 0; s < S; ++s) mx = fmaxf(mx, p[s * (HD + 2) + HD]);
    for (int s = 0; s < S; ++s) {
      const float ms = p[s * (HD + 2) + HD];
      const float f = (ms == -INFINITY) ? 0.f : __expf(ms - mx);
      l = fmaf(f, p[s * (HD + 2) + HD + 1], l);
      acc = fmaf(f, p[s * (HD + 2) + d], acc);
    }
  }
  float v;
  if (l > 0.f) {
    v = acc / l;
  } else {
    // No attended key among the row's keys: the reference's additive finfo.min mask (modeling_bailing_moe.py:1466, :802-806) then
    // absorbs every score (s + finfo.min == finfo.min in fp32), the softmax is UNIFORM over the row's keys [0, len) and the output
    // is the mean of their V rows.  Degenerate (no caller builds such a row); computed here, off the fast path, for parity.
    const int len = row_len[m];
    const int kvh = h / (n_q / n_kv);
    const float* Vb = kv_cache + (((int64_t)row_seq[m] * 2 + 1) * n_kv + kvh) * t_max * HD;
    float sum = 0.f;
    for (int j = 0; j < len; ++j) sum += Vb[(int64_t)j * HD + d];
    v = len > 0 ? sum / (float)len : 0.f;
  }
  const int64_t o = ((int64_t)m * n_q + h) * HD + d;
  if (out) out[o] = v;
  if (split) {
    const bf16_t hi = f32_to_bf16(v);
    split[o] = hi;
    split[(int64_t)M * n_q * HD + o] = f32_to_bf16(v - bf16_to_f32(hi));
  }
}

// -------------------------------------------------------------------------------------------
// One-launch form for a few rows with short caches (the reference's call shapes: 1 row of text decode, the 2-3 CFG rows of an image,
// the semantic decoder's row; <= 1024 keys): one 16-wave workgroup per (row, q head).  The key range is split over the WAVES of the
// workgroup, their (acc, max, sum) partials meet in LDS — no partial round trip through memory and no combine launch (split 9.8 us +
// combine 4.7 us per layer at 2 rows before).  Scores and PV run on 16 / 8 keys' loads in flight per wave.
// (A form with ALL of a wave's K and V loads issued before the first score — <= 24 keys per wave, 123 VGPRs — measured no faster:
// 2.046 vs 2.059 ms per 28-layer step at 1 row / 296 keys, slower at 40 keys; removed.  profiles/r04_attn_fused_ab.txt)
template <int HD>
__global__ __launch_bounds__(1024) void attn_decode_one_kernel(
    const float* __restrict__ q, int n_q, int n_kv, const float* __restrict__ kv_cache, int64_t t_max,
    const int32_t* __restrict__ row_seq, const int32_t* __restrict__ row_len, const uint8_t* __restrict__ key_mask,
    int64_t ld_mask, int chunk_cap, float* __restrict__ out, bf16_t* __restrict__ split, int M) {
  extern __shared__ __attribute__((aligned(16))) float sm[];      // [16][chunk_cap] scores, [16][HD + 2] partials
  constexpr int NW = 16;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int m = blockIdx.x, h = blockIdx.y;
  float* sc = sm + wave * chunk_cap;
  float* part = sm + NW * chunk_cap;
  const int len = row_len[m];
  int chunk = (len + NW - 1) / NW;
  chunk = (chunk + 3) & ~3;
  const int j0 = wave * chunk, j1 = min(len, j0 + chunk);
  const int kvh = h / (n_q / n_kv);
  const int64_t seq = row_seq[m];
  const float* Kb = kv_cache + ((seq * 2 + 0) * n_kv + kvh) * t_max * HD;
  const float* Vb = kv_cache + ((seq * 2 + 1) * n_kv + kvh) * t_max * HD;
  const uint8_t* mk = key_mask ? key_mask + (int64_t)m * ld_mask : nullptr;
  // ---- scores: 16 lanes per key, 4 keys per step, 4 steps' loads in flight
  constexpr int PER = HD / 16;
  constexpr int DPL = HD / 64;
  const int sub = lane & 15, kq = lane >> 4;
  const int n = max(0, j1 - j0);
  float qv[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) qv[i] = q[((int64_t)m * n_q + h) * HD + sub * PER + i];
  float mx = -INFINITY;
  for (int jb = j0; jb < j0 + chunk; jb += 16) {
    f32x4 kv[4][PER / 4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int j = jb + u * 4 + kq;
#pragma unroll
      for (int i = 0; i < PER / 4; ++i) {
        kv[u][i] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (j < j1) kv[u][i] = *reinterpret_cast<const f32x4*>(Kb + (int64_t)j * HD + sub * PER + i * 4);
      }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int j = jb + u * 4 + kq;
      float d = 0.f;
#pragma unroll
      for (int i = 0; i < PER / 4; ++i) {
        d = fmaf(kv[u][i].x, qv[i * 4], d); d = fmaf(kv[u][i].y, qv[i * 4 + 1], d);
        d = fmaf(kv[u][i].z, qv[i * 4 + 2], d); d = fmaf(kv[u][i].w, qv[i * 4 + 3], d);
      }
      d = row16_sum(d);
      const bool keep = j < j1 && (!mk || mk[j] != 0);
      const float sv = keep ? d : -INFINITY;
      if (sub == 0 && j < j0 + chunk && (j - j0) < chunk_cap) sc[j - j0] = sv;
      mx = fmaxf(mx, sv);
    }
  }
  mx = wave_max(mx);
  __syncthreads();
  float l = 0.f;
  for (int j = lane; j < n; j += 64) {
    const float p = (mx == -INFINITY) ? 0.f : __expf(sc[j] - mx);
    sc[j] = p;
    l += p;
  }
  l = wave_sum(l);
  __syncthreads();
  // ---- PV: lane owns HD / 64 dims, 8 keys' loads in flight
  float acc[DPL];
#pragma unroll
  for (int i = 0; i < DPL; ++i) acc[i] = 0.f;
  for (int jb = 0; jb < n; jb += 8) {
    float v[8][DPL];
#pragma unroll
    for (int u = 0; u < 8; ++u)
#pragma unroll
      for (int i = 0; i < DPL; ++i) {
        const int j = j0 + jb + u;
        v[u][i] = 0.f;
        if (jb + u < n) v[u][i] = Vb[(int64_t)j * HD + lane * DPL + i];
      }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      const float p = jb + u < n ? sc[jb + u] : 0.f;
#pragma unroll
      for (int i = 0; i < DPL; ++i) acc[i] = fmaf(p, v[u][i], acc[i]);
    }
  }
  float* pw = part + wave * (HD + 2);
#pragma unroll
  for (int i = 0; i < DPL; ++i) pw[lane * DPL + i] = acc[i];
  if (lane == 0) { pw[HD] = mx; pw[HD + 1] = l; }
  __syncthreads();
  // ---- the 16 waves' partials -> the head's output
  const int d = threadIdx.x;
  if (d >= HD) return;
  float mall = -INFINITY;
#pragma unroll
  for (int w = 0; w < NW; ++w) mall = fmaxf(mall, part[w * (HD + 2) + HD]);
  float lt = 0.f, at = 0.f;
#pragma unroll
  for (int w = 0; w < NW; ++w) {
    const float ms = part[w * (HD + 2) + HD];
    const float fw = (ms == -INFINITY) ? 0.f : __expf(ms - mall);
    lt = fmaf(fw, part[w * (HD + 2) + HD + 1], lt);
    at = fmaf(fw, part[w * (HD + 2) + d], at);
  }
  float v;
  if (lt > 0.f) {
    v = at / lt;
  } else {      // no attended key: uniform over the row's keys (see attn_decode_combine_kernel)
    float sum = 0.f;
    for (int j = 0; j < len; ++j) sum += Vb[(int64_t)j * HD + d];
    v = len > 0 ? sum / (float)len : 0.f;
  }
  const int64_t o = ((int64_t)m * n_q + h) * HD + d;
  if (out) out[o] = v;
  if (split) {
    const bf16_t hi = f32_to_bf16(v);
    split[o] = hi;
    split[(int64_t)M * n_q * HD + o] = f32_to_bf16(v - bf16_to_f32(hi));
  }
}

// -------------------------------------------------------------------------------------------
// One launch for a few rows over caches of any length: a workgroup per (row, KV head, key split), all G query heads of the group from one read of K and V, RoPE and the K / V
// append of the new token with it (as in the one-workgroup form above), and the last split of a (row, KV head) to arrive joins them all.
// What bounds it is latency: the kernel's arguments, the row's numbers, K and V together, the partial results, the arrival, the join are one round trip each.
//   * a lane group of 16 owns a key; it keeps its own running maximum, sum and G outputs, so that nothing crosses lanes inside the key loop but the score itself;
//   * K and V of U keys a group are asked for at once, before the query is rotated;
//   * a split is at least `keys` long: a short row is one split, which needs no join;
//   * rows of one step differ in length, which only the device knows: with `fill` every workgroup reads all rows' lengths (one round trip, as its own row's alone would be), a row gets as
//     many of `fill` splits a key head as its share of all keys is, at least one, and the workgroup's index says whose split it is; those behind the last one leave;
//   * partials leave write-through (agent scope) and are drained before the arrival is counted; the last arrival (one counter a (row, KV head), zero between launches)
//     reads them past its L1 in split order: the result does not depend on who is last.
// -------------------------------------------------------------------------------------------
__device__ __forceinline__ int join_splits(int len, int keys, int most) {
  const int n = (len + keys - 1) >> __builtin_ctz(keys);
  return len <= keys + keys / 2 ? 1 : min(most, n <= JOIN_SHORT ? n : max(JOIN_SHORT, (n + JOIN_LONG - 1) / JOIN_LONG));
}
// inclusive prefix sum over the lanes
__device__ __forceinline__ int wave_prefix(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);      // row_shr 1, 2, 4, 8
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);      // row_bcast 15 into rows 1 and 3, 31 into rows 2 and 3
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);
  return v;
}

template <int HD, int G, int NW, int U, int WPE>
__global__ __launch_bounds__(NW * 64, WPE) void attn_decode_join_kernel(int n_q, int n_kv, int64_t t_max, const int32_t* __restrict__ row_seq, const int32_t* __restrict__ row_len,
                                                                   const uint8_t* __restrict__ key_mask, int64_t ld_mask, int S_max, int keys, int fill, float* __restrict__ partial,
                                                                   uint32_t* __restrict__ arrived, float* __restrict__ out, bf16_t* __restrict__ split, const AttnFuse fz) {
  constexpr int half = HD / 2, PER = HD / 16, V4 = PER / 4, GR = 4 * NW, N = G * PER, TH = NW * 64, RL = JOIN_ROWS / 64;
  __shared__ __attribute__((aligned(16))) float qs[G * HD], knew[HD], vnew[HD];
  __shared__ __attribute__((aligned(16))) float part[NW][G * HD], mw[NW][G], lw[NW][G];
  __shared__ uint32_t last;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), sub = lane & 15, row4 = lane >> 4, grp = wave * 4 + row4;
  const int kvh = blockIdx.y;
  int m, s, S, len, slot, first;                         // first: the row's first slot among the partial results
  int64_t seq;
  if (fill == 0) {
    m = blockIdx.x;
    s = blockIdx.z;
    len = row_len[m];
    slot = fz.row_slot[m];
    seq = row_seq[m];
    S = join_splits(len, keys, S_max);
    if (s >= S) return;                                  // uniform
    first = m * S_max;
  } else {
    const int c = (fz.M + 63) >> 6, idx = blockIdx.z;    // rows lane * c .. + c - 1 are this lane's
    int l[RL], at[RL], sq[RL], n[RL], own = 0, cnt = 0;
#pragma unroll
    for (int i = 0; i < RL; ++i) {
      const int r = lane * c + i;
      l[i] = at[i] = sq[i] = 0;
      if (i < c && r < fz.M) { l[i] = row_len[r]; at[i] = fz.row_slot[r]; sq[i] = row_seq[r]; }
      own += l[i];
    }
    const float share = (float)fill * 1.00001f * __builtin_amdgcn_rcpf(fmaxf(wave_sum((float)own), 1.f));      // (a whole number of splits stays one; they are `fill` together at most)
#pragma unroll
    for (int i = 0; i < RL; ++i) {
      n[i] = 0;
      if (i < c && lane * c + i < fz.M) n[i] = max(1, min(join_splits(l[i], keys, S_max), (int)((float)l[i] * share)));
      cnt += n[i];
    }
    const int upto = wave_prefix(cnt);
    if (idx >= __builtin_amdgcn_readlane(upto, 63)) return;      // uniform
    const int src = __builtin_ctzll(__ballot(upto > idx));
    first = __builtin_amdgcn_readlane(upto, src) - __builtin_amdgcn_readlane(cnt, src);
    int i0 = 0;
    S = __builtin_amdgcn_readlane(n[0], src);
    len = __builtin_amdgcn_readlane(l[0], src);
    slot = __builtin_amdgcn_readlane(at[0], src);
    seq = __builtin_amdgcn_readlane(sq[0], src);
#pragma unroll
    for (int i = 1; i < RL; ++i)
      if (i < c && idx >= first + S) {                   // uniform
        first += S;
        i0 = i;
        S = __builtin_amdgcn_readlane(n[i], src);
        len = __builtin_amdgcn_readlane(l[i], src);
        slot = __builtin_amdgcn_readlane(at[i], src);
        seq = __builtin_amdgcn_readlane(sq[i], src);
      }
    m = src * c + i0;
    s = idx - first;
  }
  const int chunk = (len + S - 1) / S, j0 = s * chunk, j1 = min(len, j0 + chunk);
  const int held = (int)min((int64_t)j1, t_max), behind = slot >= t_max && slot < j1 ? slot : -1;      // (a new key behind a full cache is attended, and kept nowhere)
  const float* Kb = fz.kv_cache_w + ((seq * 2 + 0) * n_kv + kvh) * t_max * HD + sub * PER;
  const float* Vb = fz.kv_cache_w + ((seq * 2 + 1) * n_kv + kvh) * t_max * HD + sub * PER;
  const uint8_t* mk = key_mask ? key_mask + (int64_t)m * ld_mask : nullptr;
  f32x4 k[U][V4], v[U][V4];
  bool keep[U];
  auto fetch = [&](int jb) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int j = jb + u * GR + grp, jc = min(j, held - 1);
      keep[u] = j < held || j == behind;
      if (mk && (j < held || (j == behind && j < ld_mask))) keep[u] = mk[j] != 0;      // (a mask of the cache's length alone says nothing of the key behind it)
#pragma unroll
      for (int i = 0; i < V4; ++i) {
        k[u][i] = *reinterpret_cast<const f32x4*>(Kb + (int64_t)jc * HD + i * 4);
        v[u][i] = *reinterpret_cast<const f32x4*>(Vb + (int64_t)jc * HD + i * 4);
      }
    }
  };
  if (j0 < j1) fetch(j0);
  // ---- the row's query heads of this group, and the new key and value where the split holds them: slabs summed, rotated, into LDS ----
  const bool fresh = slot >= j0 && slot < j1;
  {
    const float* row = fz.qkv + (int64_t)m * fz.ldqkv;
    for (int t = tid; t < (fresh ? G + 2 : G) * half; t += TH) {
      const int hh = t / half, i = t % half, head = hh < G ? kvh * G + hh : n_q + (hh - G) * n_kv + kvh;
      const float* p_ = row + (int64_t)head * HD + i;
      float x1 = 0.f, x2 = 0.f, c = 1.f, sn = 0.f;
      const bool rot = fz.rope && hh <= G;
      if (rot) {
        const int stream = fz.sec_t <= 0 ? 0 : (i < fz.sec_t ? 0 : (i < fz.sec_t + fz.sec_h ? 1 : 2));
        const int pos = fz.row_pos[stream * fz.M + m];
        c = fz.cos_tab[(int64_t)pos * half + i];
        sn = fz.sin_tab[(int64_t)pos * half + i];
      }
      for (int z0 = 0; z0 < fz.nz; z0 += 8) {            // eight slabs' loads in flight, added in slab order
        float a1[8], a2[8];
#pragma unroll
        for (int z = 0; z < 8; ++z) {
          a1[z] = z0 + z < fz.nz ? p_[(int64_t)(z0 + z) * fz.slab] : 0.f;
          a2[z] = z0 + z < fz.nz ? p_[(int64_t)(z0 + z) * fz.slab + half] : 0.f;
        }
#pragma unroll
        for (int z = 0; z < 8; ++z) { x1 += a1[z]; x2 += a2[z]; }
      }
      if (rot) rotate_pair(x1, x2, c, sn);
      if (hh < G) { x1 *= fz.q_scale; x2 *= fz.q_scale; }
      float* dst = hh < G ? qs + hh * HD : hh == G ? knew : vnew;
      dst[i] = x1;
      dst[i + half] = x2;
      if (hh >= G && (uint64_t)slot < (uint64_t)t_max) {   // the new token's line of the arena
        float* ad = fz.kv_cache_w + (((seq * 2 + (hh - G)) * n_kv + kvh) * t_max + slot) * HD;
        ad[i] = x1;
        ad[i + half] = x2;
      }
    }
  }
  __syncthreads();
  f32x4 q[G][V4];
  float acc[N], mx[G], l[G];
#pragma unroll
  for (int g = 0; g < G; ++g) {
    mx[g] = -INFINITY;
    l[g] = 0.f;
#pragma unroll
    for (int i = 0; i < V4; ++i) q[g][i] = *reinterpret_cast<const f32x4*>(qs + g * HD + sub * PER + i * 4);
  }
#pragma unroll
  for (int i = 0; i < N; ++i) acc[i] = 0.f;
  for (int jb = j0; jb < j1; jb += U * GR) {
    if (jb > j0) fetch(jb);
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (fresh && jb + u * GR + grp == slot) {
#pragma unroll
        for (int i = 0; i < V4; ++i) {
          k[u][i] = *reinterpret_cast<const f32x4*>(knew + sub * PER + i * 4);
          v[u][i] = *reinterpret_cast<const f32x4*>(vnew + sub * PER + i * 4);
        }
      }
#pragma unroll
    for (int g = 0; g < G; ++g) {
      float d[U], top = mx[g];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        float a = 0.f;
#pragma unroll
        for (int i = 0; i < V4; ++i) {
          a = fmaf(k[u][i].x, q[g][i].x, a); a = fmaf(k[u][i].y, q[g][i].y, a);
          a = fmaf(k[u][i].z, q[g][i].z, a); a = fmaf(k[u][i].w, q[g][i].w, a);
        }
        a = row16_sum(a);
        d[u] = keep[u] ? a : -INFINITY;
        top = fmaxf(top, d[u]);
      }
      const float f = mx[g] == -INFINITY ? 0.f : __expf(mx[g] - top);
      l[g] *= f;
#pragma unroll
      for (int i = 0; i < PER; ++i) acc[g * PER + i] *= f;
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const float p = d[u] == -INFINITY ? 0.f : __expf(d[u] - top);
        l[g] += p;
        if (keep[u]) {                                   // (a key that is not attended may hold anything)
#pragma unroll
          for (int i = 0; i < PER; ++i) acc[g * PER + i] = fmaf(p, v[u][i / 4][i % 4], acc[g * PER + i]);
        }
      }
      mx[g] = top;
    }
  }
  // ---- a wave's four groups: one maximum, then a sum that leaves each group a quarter of the outputs (values i + N / 4 (row4 >> 1) + N / 2 (row4 & 1)) ----
#pragma unroll
  for (int g = 0; g < G; ++g) {
    float top = fmaxf(mx[g], __shfl_xor(mx[g], 16));
    top = fmaxf(top, __shfl_xor(top, 32));
    const float f = mx[g] == -INFINITY ? 0.f : __expf(mx[g] - top);
    float a = l[g] * f;
    a += __shfl_xor(a, 16);
    a += __shfl_xor(a, 32);
#pragma unroll
    for (int i = 0; i < PER; ++i) acc[g * PER + i] *= f;
    if (lane == 0) { mw[wave][g] = top; lw[wave][g] = a; }
  }
#pragma unroll
  for (int i = 0; i < N / 2; ++i) {
    const auto x = __builtin_amdgcn_permlane16_swap(__float_as_uint(acc[i]), __float_as_uint(acc[i + N / 2]), false, false);
    acc[i] = __uint_as_float(x[0]) + __uint_as_float(x[1]);
  }
#pragma unroll
  for (int i = 0; i < N / 4; ++i) {
    const auto x = __builtin_amdgcn_permlane32_swap(__float_as_uint(acc[i]), __float_as_uint(acc[i + N / 4]), false, false);
    const int at = i + N / 4 * (row4 >> 1) + N / 2 * (row4 & 1);
    part[wave][at / PER * HD + sub * PER + at % PER] = __uint_as_float(x[0]) + __uint_as_float(x[1]);
  }
  __syncthreads();
  // ---- the waves' results meet in LDS; they are the row's (one split) or leave as the split's ----
  float* base = partial + ((int64_t)first * n_q + (int64_t)kvh * G * S) * (HD + 2);      // [query head][split]
  auto put = [&](int g, int d, float lt, float at) {
    float val;
    if (lt > 0.f) {
      val = at / lt;
    } else {                                             // no attended key: uniform over the row's keys (see attn_decode_combine_kernel)
      const float* Vd = fz.kv_cache_w + ((seq * 2 + 1) * n_kv + kvh) * t_max * HD + d;
      const float* vp = fz.qkv + (int64_t)m * fz.ldqkv + (int64_t)(n_q + n_kv + kvh) * HD + d;
      float sum = 0.f;
      for (int j = 0; j < len; ++j) {
        float y = 0.f;
        if (j == slot) for (int z = 0; z < fz.nz; ++z) y += vp[(int64_t)z * fz.slab];      // (the arena's line of it may be another split's to write)
        else if (j < t_max) y = Vd[(int64_t)j * HD];
        sum += y;
      }
      val = len > 0 ? sum / (float)len : 0.f;
    }
    const int64_t o = ((int64_t)m * n_q + kvh * G + g) * HD + d;
    if (out) out[o] = val;
    if (split) {
      const bf16_t hi = f32_to_bf16(val);
      split[o] = hi;
      split[(int64_t)fz.M * n_q * HD + o] = f32_to_bf16(val - bf16_to_f32(hi));
    }
  };
  for (int t = tid; t < G * HD; t += TH) {
    const int g = t / HD, d = t % HD;
    float top = -INFINITY, lt = 0.f, at = 0.f;
#pragma unroll
    for (int r = 0; r < NW; ++r) top = fmaxf(top, mw[r][g]);
#pragma unroll
    for (int r = 0; r < NW; ++r) {
      const float f = mw[r][g] == -INFINITY ? 0.f : __expf(mw[r][g] - top);
      lt = fmaf(f, lw[r][g], lt);
      at = fmaf(f, part[r][t], at);
    }
    if (S == 1) {
      put(g, d, lt, at);
      continue;
    }
    float* o = base + ((int64_t)g * S + s) * (HD + 2);
    __hip_atomic_store(o + d, at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (d == 0) {
      __hip_atomic_store(o + HD, top, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_store(o + HD + 1, lt, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
  if (S == 1) return;                                    // uniform
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  uint32_t* cnt = arrived + (int64_t)m * n_kv + kvh;
  if (tid == 0) last = __hip_atomic_fetch_add(cnt, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (uint32_t)S - 1;
  __syncthreads();
  if (!last) return;
  if (tid == 0) __hip_atomic_store(cnt, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  for (int t = tid; t < G * HD; t += TH) {               // (whole waves of one head; lane z holds split z's statistics)
    const int g = t / HD, d = t % HD;
    const float* p = base + (int64_t)g * S * (HD + 2);
    auto ld = [&](int z, int i) { return __hip_atomic_load(p + (int64_t)z * (HD + 2) + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); };
    float ms = -INFINITY, ls = 0.f, x[16], a = 0.f;
    if (lane < S) { ms = ld(lane, HD); ls = ld(lane, HD + 1); }
#pragma unroll
    for (int z = 0; z < 16; ++z) x[z] = z < S ? ld(z, d) : 0.f;
    const float top = wave_max(ms), f = ms == -INFINITY ? 0.f : __expf(ms - top), lt = wave_sum(f * ls);
#pragma unroll
    for (int z = 0; z < 16; ++z) a = fmaf(lane_f(f, z), x[z], a);
    for (int z0 = 16; z0 < S; z0 += 16) {
#pragma unroll
      for (int z = 0; z < 16; ++z) x[z] = z0 + z < S ? ld(z0 + z, d) : 0.f;
#pragma unroll
      for (int z = 0; z < 16; ++z) a = fmaf(lane_f(f, z0 + z), x[z], a);
    }
    put(g, d, lt, a);
  }
}

// Key-range splits (flash-decoding): enough workgroups to fill the chip at few rows, none needed at hundreds of rows;
// one split never holds more than 4096 keys (its scores live in LDS).
// One wave a (row, KV head, split) reads every key once for its four heads, where there are enough (row, KV head) pairs: 40, with two KV heads 48 (cold caches, us,
// this form against one wave a head: 12 rows x 4 KV heads 28 / 32, 64 x 4 65 / 90, 24 x 2 33 / 38, 16 x 3 23 / 25; but 8 x 4 25.6 / 23.9, 20 x 2 22.9 / 21.7, 12 x 3
// 26.5 / 26.1; a step of 28 layers with 11 rows 5.82 / 5.92 ms, with 8 5.28 / 5.24).  With one KV head three of a workgroup's four waves repeat the fourth's
// work (64 x 1 37 / 29).
static bool attn_use_gqa(int M, int n_q, int n_kv, int hd) {
  return (M > 64 || (n_kv >= 2 && M * n_kv >= (n_kv == 2 ? 48 : 40))) && hd == 128 && n_q == 4 * n_kv;
}
// the one-launch form: <= g_one_rows rows whose caches hold <= 1024 keys (dev-library A/B: mn_attn_tune_one)
static int g_one_rows = 16;
#ifdef MN_DEV_HOOKS
extern "C" MN_DEV_API void mn_attn_tune_one(int max_rows) { g_one_rows = max_rows; }
#endif
static bool attn_use_one(int M, int64_t t_max) { return M <= g_one_rows && t_max <= 1024; }
static int attn_splits(int M, int n_q, int64_t t_max) {
  int S = (int)mn_cdiv(t_max, 32);
  if (S > 32) S = 32;
  const int want = (int)mn_cdiv(4096, M);       // a few thousand waves on the chip whatever the row count
  if (S > want) S = want;
  const int need = (int)mn_cdiv(t_max, 1024);   // scores of a split live in LDS (4 heads x 1024 keys per wave at most)
  if (S < need) S = need;
  if (S < 1) S = 1;
  return S;
}

extern "C" size_t mn_attn_decode_workspace_bytes(int M, int n_q, int hd, int64_t t_max) {
  return (size_t)M * n_q * attn_splits(M, n_q, t_max) * (hd + 2) * sizeof(float);
}

static int attn_decode_launch(const float* q, int M, int n_q, int n_kv, int hd, const float* kv_cache, int64_t t_max,
                              const int32_t* row_seq, const int32_t* row_len, const uint8_t* key_mask, int64_t ld_mask, float* out,
                              uint16_t* split, void* workspace, size_t workspace_bytes, void* stream) {
  hipStream_t st0 = mn_stream(stream);
  if (attn_use_one(M, t_max)) {                 // a few rows, short caches: one launch, the key split lives inside the workgroup
    int cc = (int)mn_cdiv(t_max, 16);
    cc = (cc + 3) & ~3;
    const size_t lds1 = ((size_t)16 * cc + 16 * (hd + 2)) * sizeof(float);
    const dim3 g1(M, n_q), b1(1024);
#define MN_ONE(HD_) hipLaunchKernelGGL(attn_decode_one_kernel<HD_>, g1, b1, lds1, st0, q, n_q, n_kv, kv_cache, t_max, row_seq, row_len, key_mask, ld_mask, cc, out, split, M)
    if (hd == 128) MN_ONE(128); else MN_ONE(64);
#undef MN_ONE
    MN_CHECK_LAUNCH("mn_attn_decode(one launch)");
    return MN_OK;
  }
  const int S = attn_splits(M, n_q, t_max);
  const size_t need = (size_t)M * n_q * S * (hd + 2) * sizeof(float);
  if (workspace_bytes < need) { mn_set_error("mn_attn_decode: workspace %zu < %zu", workspace_bytes, need); return MN_ENOSPACE; }
  int chunk_cap = (int)mn_cdiv(t_max, S);
  chunk_cap = (chunk_cap + 3) & ~3;
  const size_t lds = (size_t)4 * chunk_cap * sizeof(float);
  float* partial = reinterpret_cast<float*>(workspace);
  dim3 grid(M, (n_q + 3) / 4, S);
  hipStream_t st = mn_stream(stream);
  if (attn_use_gqa(M, n_q, n_kv, hd)) {
    hipLaunchKernelGGL((attn_decode_gqa_kernel<128, 4>), dim3(M, (n_kv + 3) / 4, S), dim3(256), lds * 4, st, q, n_q, n_kv, kv_cache,
                       t_max, row_seq, row_len, key_mask, ld_mask, S, chunk_cap, partial);
  } else if (hd == 128) {
    hipLaunchKernelGGL(attn_decode_split_kernel<128>, grid, dim3(256), lds, st, q, n_q, n_kv, kv_cache, t_max, row_seq,
                       row_len, key_mask, ld_mask, S, chunk_cap, partial);
  } else {
    hipLaunchKernelGGL(attn_decode_split_kernel<64>, grid, dim3(256), lds, st, q, n_q, n_kv, kv_cache, t_max, row_seq,
                       row_len, key_mask, ld_mask, S, chunk_cap, partial);
  }
  if (hd == 128)
    hipLaunchKernelGGL(attn_decode_combine_kernel<128>, dim3(M, n_q), dim3(128), 0, st, partial, n_q, S, out, split, M, kv_cache, n_kv, t_max,
                       row_seq, row_len);
  else
    hipLaunchKernelGGL(attn_decode_combine_kernel<64>, dim3(M, n_q), dim3(64), 0, st, partial, n_q, S, out, split, M, kv_cache, n_kv, t_max,
                       row_seq, row_len);
  MN_CHECK_LAUNCH("mn_attn_decode");
  return MN_OK;
}

// Internal (engine.hip): mn_attn_decode whose output can also (or only) be written as bf16 hi/lo rows.
extern "C" int mn_attn_decode_split(const float* q, int M, int n_q, int n_kv, int hd, const float* kv_cache,
                                    int64_t t_max, const int32_t* row_seq, const int32_t* row_len,
                                    const uint8_t* key_mask, int64_t ld_mask, float* out, uint16_t* split, void* workspace,
                                    size_t workspace_bytes, void* stream) {
  MN_CHECK_ARG(M >= 1 && n_q >= 1 && n_kv >= 1 && n_q % n_kv == 0 && (hd == 64 || hd == 128), "mn_attn_decode: bad shape");
  MN_CHECK_ARG(q && kv_cache && row_seq && row_len && (out || split) && workspace, "mn_attn_decode: null pointer");
  return attn_decode_launch(q, M, n_q, n_kv, hd, kv_cache, t_max, row_seq, row_len, key_mask, ld_mask, out, split, workspace,
                            workspace_bytes, stream);
}

// Internal (engine.hip): RoPE + q scale + KV append + masked decode attention in ONE launch from the raw QKV projection (optionally as nz K-slice partial slabs): what
// mn_rope_kv_append_3d / mn_rope_kv_from_partials followed by mn_attn_decode_split compute.  Rows of distinct sequences with row_len == row_slot + 1; n_q / n_kv in {1, 2, 4}.
// arrived: mn_attn_arrivals' counters, zero (they are left zero), or NULL for one split a row.
// us a launch over 24 layers' caches, the launches before (one workgroup a head up to 16 rows over 1024 keys; else the append, a launch of 32 splits and one that joins them; from
// 40 (row, key head) pairs on a wave a key head) / this one.  16 heads of 128 over 4: 1 row of 80 keys 6.5 / 6.4, 330 13.1 / 7.7, 1100 13.0 / 9.7, 1900 16.9 / 9.9; 4 rows 7.1 / 7.5,
// 13.3 / 8.9, 19.7 / 14.3, 27.0 / 15.7; 10 rows 7.7 / 7.6, 18.0 / 11.0, 25.7 / 16.4, 35.7 / 21.4; 36 rows 18.9 / 10.1, 22.8 / 18.0, 43.5 / 37.4, 64 / 57; 64 rows 19.6 / 11.3, 27.2 / 22.8,
// 69.6 / 55.5 (5.2 TB/s), 110 / 89; 200 rows 26.7 / 23.1, 66 / 60, 192 / 169; 1536 rows of 80 147 / 127.  16 heads of 64: 1 row of 40 keys 4.4 / 3.3, 250 6.9 / 5.8, 600 10.7 / 7.1;
// 16 rows 5.9 / 4.7, 11.2 / 10.1, 19.3 / 18.4; 64 rows 16.8 / 9.6, 37.3 / 27.3, 71 / 58.
static int g_attn_fuse = 1;                          // dev-library A/B switch: 0 = never fused
#ifdef MN_DEV_HOOKS
extern "C" MN_DEV_API void mn_attn_tune_fuse(int on) { g_attn_fuse = on; }
#endif
extern "C" int mn_attn_fused_ok(int M, int n_q, int n_kv, int hd) {
  if (g_kv_round_bf16 || !g_attn_fuse) return 0;     // the bf16-KV measurement hook lives in the stand-alone append kernel
  const int ratio = n_kv > 0 && n_q % n_kv == 0 ? n_q / n_kv : 0;
  return M >= 1 && (hd == 64 || hd == 128) && (ratio == 1 || ratio == 2 || ratio == 4);
}
// Splits of a launch.  keys: 64 KB of K and V, what a workgroup asks for at once.  Where all rows can have all the splits their lengths allow, or a row has few of them, their number is that of
// rows of one length: as many as make one round of the CUs.  Else, up to 128 rows, the lengths say (fill splits a key head), and with more rows 1024 keys are a split.  us a layer of a step with
// small experts, a number of splits for all rows / this: 36 rows of 100 keys but one of 8000 223 / 56, 64 of 200 but one of 16000 550 / 73, 100 of 100 but one of 4000 166 / 64, 200 183 / 114; rows
// of one length 3 x 1900 43.5 / 44.3, 36 x 1100 75.2 / 74.7, 64 x 1100 94.8 / 94.4, 100 x 1100 132 / 130.  The lengths cost 0.3 .. 0.7 (2 rows of 330 keys 30.5 / 31.3: not there), of 200 rows 3.7
// (4 a lane: not there); empty workgroups of 1024 keys' splits 2 (200 rows of 100 keys, cache of 8192, 79.7 / 81.8).
struct JoinPlan { int most, keys, fill, z; int64_t slots; };
static JoinPlan attn_join_plan(int M, int n_kv, int hd, int64_t t_max) {
  constexpr int LONG_KEYS = 1024, SHORT = 8;
  JoinPlan p{1, 64 * 128 / hd, 0, 1, 0};
  const int64_t fill = mn_num_cus() / n_kv;
  if (M > JOIN_ROWS) p.keys = LONG_KEYS;
  int64_t most = mn_cdiv(t_max, p.keys);
  if (most > JOIN_MOST) most = JOIN_MOST;
  if (M <= JOIN_ROWS && most > fill) most = fill;
  p.fill = M <= JOIN_ROWS && M * most > fill && most > SHORT && t_max < 1 << 24 ? (int)fill : 0;      // (128 lengths' sum is of 32 bits)
  if (M <= JOIN_ROWS && !p.fill && most > fill / M) most = fill / M;
  if (most <= 1 || t_max <= p.keys + p.keys / 2) return JoinPlan{1, p.keys, 0, 1, 0};
  p.most = p.z = (int)most;
  p.slots = M * most;
  if (p.fill) {
    if (p.slots > M + fill) p.slots = M + fill;          // rows of one split, and the rest shares `fill`
    p.z = (int)p.slots;
  }
  return p;
}
// The arrival counters of mn_attn_decode_fused, behind the partials in the scratch that mn_attn_decode_workspace_bytes sizes: [M][n_kv],
// to be zeroed once before a step's first layer (*n words); NULL: one split a row, which needs none.
extern "C" uint32_t* mn_attn_arrivals(int M, int n_q, int n_kv, int hd, int64_t t_max, void* workspace, size_t workspace_bytes, int* n) {
  const JoinPlan p = attn_join_plan(M, n_kv, hd, t_max);
  const size_t part = (size_t)p.slots * n_q * (hd + 2) * sizeof(float), need = part + (size_t)M * n_kv * sizeof(uint32_t);
  *n = 0;
  if (p.most == 1 || !workspace || need > workspace_bytes) return nullptr;
  *n = M * n_kv;
  return reinterpret_cast<uint32_t*>(reinterpret_cast<char*>(workspace) + part);
}
extern "C" int mn_attn_decode_fused(const float* qkv, int64_t ldqkv, int nz, int64_t slab, int M, int n_q, int n_kv, int hd, int rope,
                                    const float* cos_tab, const float* sin_tab, const int32_t* row_seq, const int32_t* row_slot,
                                    const int32_t* row_pos, int sec_t, int sec_h, float q_scale, float* kv_cache, int64_t t_max,
                                    const int32_t* row_len, const uint8_t* key_mask, int64_t ld_mask, float* out, uint16_t* split,
                                    void* workspace, uint32_t* arrived, void* stream) {
  MN_CHECK_ARG(mn_attn_fused_ok(M, n_q, n_kv, hd) && nz >= 1, "mn_attn_decode_fused: unsupported shape");
  MN_CHECK_ARG(qkv && kv_cache && row_seq && row_slot && row_len && (out || split) && (workspace || !arrived), "mn_attn_decode_fused: null pointer");
  MN_CHECK_ARG(!rope || (cos_tab && sin_tab && row_pos), "mn_attn_decode_fused: rope needs tables and positions");
  MN_CHECK_ARG(sec_t >= 0 && sec_h >= 0 && sec_t + sec_h <= hd / 2, "mn_attn_decode_fused: bad rotary sections %d/%d", sec_t, sec_h);
  AttnFuse fz;
  fz.qkv = qkv; fz.ldqkv = ldqkv; fz.nz = nz; fz.slab = slab; fz.rope = rope; fz.cos_tab = cos_tab; fz.sin_tab = sin_tab;
  fz.row_slot = row_slot; fz.row_pos = row_pos; fz.sec_t = sec_t; fz.sec_h = sec_h; fz.q_scale = q_scale; fz.M = M; fz.kv_cache_w = kv_cache;
  const JoinPlan p = arrived ? attn_join_plan(M, n_kv, hd, t_max) : JoinPlan{1, 64 * 128 / hd, 0, 1, 0};
  const int64_t pairs = (int64_t)M * n_kv, cu = mn_num_cus();
  float* partial = reinterpret_cast<float*>(workspace);
  const dim3 grid(p.fill ? 1 : M, n_kv, p.z);
  hipStream_t st = mn_stream(stream);
#define MN_JOIN(HD_, G_, NW_, U_, W_) hipLaunchKernelGGL((attn_decode_join_kernel<HD_, G_, NW_, U_, W_>), grid, dim3(NW_ * 64), 0, st, n_q, n_kv, t_max, row_seq, row_len, key_mask, \
                                                         ld_mask, p.most, p.keys, p.fill, partial, arrived, out, split, fz)
  // from a workgroup a CU on: with one key a group in flight two of them fit a CU (1536 rows of 80 keys 195 -> 127 us, 64 rows 57 -> 55.5; 36 rows 37.4 -> 47); heads of 64, from four a
  // CU on: four waves each (64 rows of 40 keys 10.7 -> 9.6 us; 32 rows 9.9 -> 10.4)
#define MN_JOIN_HD128(G_) do { if (pairs >= cu) MN_JOIN(128, G_, 8, 1, 4); else MN_JOIN(128, G_, 8, 2, 2); } while (0)
#define MN_JOIN_HD64(G_) do { if (pairs >= 4 * cu) MN_JOIN(64, G_, 4, 2, 4); else MN_JOIN(64, G_, 8, 2, 2); } while (0)
  const int ratio = n_q / n_kv;
  if (hd == 128) { if (ratio == 4) MN_JOIN_HD128(4); else if (ratio == 2) MN_JOIN_HD128(2); else MN_JOIN_HD128(1); }
  else           { if (ratio == 4) MN_JOIN_HD64(4); else if (ratio == 2) MN_JOIN_HD64(2); else MN_JOIN_HD64(1); }
#undef MN_JOIN_HD128
#undef MN_JOIN_HD64
#undef MN_JOIN
  MN_CHECK_LAUNCH("mn_attn_decode_fused");
  return MN_OK;
}

extern "C" int mn_attn_decode(const float* q, int M, int n_q, int n_kv, int hd, const float* kv_cache,
                                 int64_t t_max, const int32_t* row_seq, const int32_t* row_len,
                                 const uint8_t* key_mask, int64_t ld_mask, float* out, void* workspace,
                                 size_t workspace_bytes, void* stream) {
  MN_CHECK_ARG(out, "mn_attn_decode: null pointer");
  return mn_attn_decode_split(q, M, n_q, n_kv, hd, kv_cache, t_max, row_seq, row_len, key_mask, ld_mask, out, nullptr, workspace,
                              workspace_bytes, stream);
}
