// moe_down.hip — the MoE down projection of a 1- / 2-row decode step (text decode; the 2-row CFG step of one image):
//
//   out[b][n] = res[b][n] + sum_{s < n_slot} tw[b, s] * sum_{k < I} hmid[b][s][k] * Wdown[ti[b, s]][n][k]
//
// (moe_infer's weighted un-permute over the selected experts + the shared ones, modeling_bailing_moe.py:604-639, for ONE row per batch
// entry).  The K-segment form of the fp32-FMA skinny kernel is slow here: a wave owns a few output rows and walks all
// n_slot x ceil(I / 512) weight chunks of a row IN SEQUENCE through a 4-deep ring — 24 chunks = six dependent HBM round trips, and every
// workgroup stages the 45 KB 8-segment activation image: 22.9 us for 92 MB at 2 rows, 16 us for 46 MB at one (2.9 TB/s; unchanged
// by fp8 bytes: latency, not bytes).
// Here the segments are spread over the waves instead: a workgroup owns RW = 8 output rows, wave s multiplies segment s (one expert)
// for all of them — its slice of the activation (I floats, scaled by the router weight) lives in its REGISTERS, no LDS image — with DR
// rows in flight, each multiplied while the later ones arrive (all RW at once, multiplied chunk by chunk behind the last: 10.3 us for 46 MB at one row and 18.3 for two of different sequences; here
// 9.3 and 15.9).  The n_slot partial sums of a row meet in LDS, in slot order (deterministic).
#include <type_traits>

#include "common.h"
#include "w8_codec.h"

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

namespace {

constexpr int RW = 8;                // output rows per workgroup
constexpr int DR = 3;                // of them in flight (2, 3, 4, 8: 9.43, 9.32, 9.35, 10.34 us for the 46 MB of one row)
constexpr int MAX_SLOTS = 8;         // segments = waves per workgroup

struct DownArgs {
  const float* hmid; int64_t ld_hmid;               // [batch][n_slot * I] fp32
  const void* W; int64_t w_stride;                  // [E + S][H][I] bf16 (or e4m3 bytes), elements between experts
  const float* wscale; int64_t wscale_stride;       // e4m3 / int8: one fp32 scale per output row, [E + S][H]; NF4: one absmax per 64 k, [E + S][H][I / 64]
  const int32_t* ti; const float* tw;               // [batch][n_slot]
  const float* res; int64_t ld_res;                 // [batch][H]
  float* out; int64_t ld_out;
  int H, I, n_slot;
  const float* P; int nz; int64_t slab;             // optional: res[b][n] += sum of nz partial slabs P [nz][batch][H] (the decoder chain's attention output projection)
};

template <int NCK, int WQ>                          // WQ 0: bf16 weights, 1: e4m3 bytes + row scales (on the K sums), 2: int8 (quanto), 3: NF4
__global__ __launch_bounds__(MAX_SLOTS * 64) void moe_down_kernel(const DownArgs a) {
  __shared__ float part[MAX_SLOTS][RW];
  const int tid = threadIdx.x, lane = tid & 63, s = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int b = blockIdx.y, n0 = blockIdx.x * RW, I = a.I;
  const bool live = s < a.n_slot;
  // ---- this wave's slice of the activation first (loads retire in order: it lands before the weights) ...
  float xk[NCK][8];
  float sc = 0.f;
  // a piece = this lane's 8 consecutive weights of one row and chunk: 16 bytes of bf16, 8 of e4m3 / int8, 4 of NF4 codes
  typedef typename std::conditional<WQ == 0, u32x4, typename std::conditional<WQ == 3, uint32_t, u32x2>::type>::type wv;
  constexpr int BPP = WQ == 0 ? 16 : (WQ == 3 ? 4 : 8);
  const uint8_t* wbase = static_cast<const uint8_t*>(a.W);
  const float* sbase = a.wscale;
  if (live) {
    sc = a.tw[(int64_t)b * a.n_slot + s];
    const int e = a.ti[(int64_t)b * a.n_slot + s];
    wbase += ((int64_t)e * a.w_stride >> 3) * BPP;
    if constexpr (WQ != 0) sbase += (int64_t)e * a.wscale_stride;
    const float* xp = a.hmid + (int64_t)b * a.ld_hmid + (int64_t)s * I;
#pragma unroll
    for (int c = 0; c < NCK; ++c) {
      const int k = c * 512 + lane * 8;
      typedef float f4 __attribute__((ext_vector_type(4)));
      f4 lo = {0.f, 0.f, 0.f, 0.f}, hi = {0.f, 0.f, 0.f, 0.f};
      if (k < I) { lo = *reinterpret_cast<const f4*>(xp + k); hi = *reinterpret_cast<const f4*>(xp + k + 4); }      // I % 8 == 0
      xk[c][0] = lo.x; xk[c][1] = lo.y; xk[c][2] = lo.z; xk[c][3] = lo.w; xk[c][4] = hi.x; xk[c][5] = hi.y; xk[c][6] = hi.z; xk[c][7] = hi.w;
    }
  }
  // ---- ... then the rows' weights, DR of the RW rows in flight: a row is multiplied while later ones arrive
  wv wq[DR][NCK];
  float rs[DR][WQ == 3 ? NCK : 1];                    // e4m3 / int8: the row's scale; NF4: the absmax of the piece's 64-block
  auto request = [&](int r) {
    const int64_t row = min(n0 + r, a.H - 1);
    const uint8_t* wr = wbase + ((row * I) >> 3) * BPP;
#pragma unroll
    for (int c = 0; c < NCK; ++c) {
      const int k = min(c * 512 + lane * 8, I - 8);          // beyond I the activation registers are zero: any finite weights will do
      wq[r % DR][c] = __builtin_nontemporal_load(reinterpret_cast<const wv*>(wr + (k >> 3) * BPP));
      if constexpr (WQ == 3) rs[r % DR][c] = sbase[row * (I >> 6) + (k >> 6)];
    }
    if constexpr (WQ == 1 || WQ == 2) rs[r % DR][0] = sbase[row];
  };
  if (live) {
#pragma unroll
    for (int r = 0; r < DR; ++r) request(r);
  }
  // (the epilogue's residual is requested now, behind the weights, and used after the reduction)
  float r_old = 0.f;
  if (tid < RW && n0 + tid < a.H && a.res) {
    r_old = a.res[(int64_t)b * a.ld_res + n0 + tid];
    for (int z = 0; z < a.nz; ++z) r_old += a.P[(int64_t)z * a.slab + (int64_t)b * a.H + n0 + tid];      // (slab order, like llm_glue_kernel)
  }
  if (live) {
#pragma unroll
    for (int c = 0; c < NCK; ++c)
#pragma unroll
      for (int e = 0; e < 8; ++e) xk[c][e] *= sc;             // the router weight rides the activation (as in the K-segment form)
#pragma unroll
    for (int r = 0; r < RW; ++r) {
      float t = 0.f;
      const float row_scale = WQ == 1 ? rs[r % DR][0] : 1.f;
#pragma unroll
      for (int c = 0; c < NCK; ++c) {
        const float* x = xk[c];
        if constexpr (WQ >= 2) {                          // int8: bf16(q * scale), NF4: bf16(NF4[code] * absmax) — rounded per element (w8_codec.h)
          u32x4 q;
          if constexpr (WQ == 2) q = w8x8_to_bf16<true>(wq[r % DR][c].x, wq[r % DR][c].y, rs[r % DR][0]);
          else q = nf4x8_to_bf16(nf4_table(rs[r % DR][c]), wq[r % DR][c]);
          t = fmaf(bf16lo_to_f32(q.x), x[0], t); t = fmaf(bf16hi_to_f32(q.x), x[1], t);
          t = fmaf(bf16lo_to_f32(q.y), x[2], t); t = fmaf(bf16hi_to_f32(q.y), x[3], t);
          t = fmaf(bf16lo_to_f32(q.z), x[4], t); t = fmaf(bf16hi_to_f32(q.z), x[5], t);
          t = fmaf(bf16lo_to_f32(q.w), x[6], t); t = fmaf(bf16hi_to_f32(q.w), x[7], t);
        } else if constexpr (WQ == 1) {
          float w0[4], w1[4];
          fp8x4_to_f32(wq[r % DR][c].x, w0);
          fp8x4_to_f32(wq[r % DR][c].y, w1);
#pragma unroll
          for (int e = 0; e < 4; ++e) t = fmaf(w0[e], x[e], t);
#pragma unroll
          for (int e = 0; e < 4; ++e) t = fmaf(w1[e], x[4 + e], t);
        } else {
          const u32x4 q = wq[r % DR][c];
          t = fmaf(bf16lo_to_f32(q.x), x[0], t); t = fmaf(bf16hi_to_f32(q.x), x[1], t);
          t = fmaf(bf16lo_to_f32(q.y), x[2], t); t = fmaf(bf16hi_to_f32(q.y), x[3], t);
          t = fmaf(bf16lo_to_f32(q.z), x[4], t); t = fmaf(bf16hi_to_f32(q.z), x[5], t);
          t = fmaf(bf16lo_to_f32(q.w), x[6], t); t = fmaf(bf16hi_to_f32(q.w), x[7], t);
        }
      }
      if (r + DR < RW) {
        __builtin_amdgcn_sched_barrier(0);
        request(r + DR);
        __builtin_amdgcn_sched_barrier(0);
      }
      t = wave_sum(t);
      if (lane == 0) part[s][r] = WQ == 1 ? t * row_scale : t;       // (e4m3: the row scale on the sum)
    }
  } else if (lane < RW) {
    part[s][lane] = 0.f;
  }
  __syncthreads();
  if (tid < RW && n0 + tid < a.H) {
    float y = r_old;
    for (int q = 0; q < a.n_slot; ++q) y += part[q][tid];     // slot order: the same bits every run
    a.out[(int64_t)b * a.ld_out + n0 + tid] = y;
  }
}

}  // namespace

// Can the down projection of this shape run here?  (bf16, e4m3, int8 or NF4 weights; one wave per slot; I in whole 8-element pieces, <= 4 chunks of 512)
bool moe_down_ok(int wfmt, int n_slot, int H, int I) {
  return (wfmt == MN_W_BF16 || wfmt == MN_W_FP8_E4M3 || wfmt == MN_W_INT8 || (wfmt == MN_W_NF4 && (I % 64) == 0)) && n_slot >= 1 &&
         n_slot <= MAX_SLOTS && H >= 1 && I >= 8 && (I % 8) == 0 && I <= 2048;
}

int moe_down_rows(int wfmt, const float* hmid, int64_t ld_hmid, const void* W, int64_t w_stride, const float* wscale, int64_t wscale_stride,
                  const int32_t* ti, const float* tw, const float* res, int64_t ld_res, float* out, int64_t ld_out, int batch, int H, int I,
                  int n_slot, void* stream, const float* P, int nz, int64_t slab) {
  MN_CHECK_ARG(hmid && W && ti && tw && out && batch >= 1 && moe_down_ok(wfmt, n_slot, H, I) && (ld_hmid % 4) == 0 &&
                   (((uintptr_t)W) & 15) == 0 && (w_stride % 8) == 0 && (wfmt == MN_W_BF16 || wscale), "moe_down_rows: bad args");
  const DownArgs a{hmid, ld_hmid, W, w_stride, wscale, wscale_stride, ti, tw, res, ld_res, out, ld_out, H, I, n_slot, P, P ? nz : 0, slab};
  const dim3 grid((unsigned)mn_cdiv(H, RW), (unsigned)batch), block(MAX_SLOTS * 64);
  const int nck = (I + 511) / 512;
  hipStream_t st = mn_stream(stream);
#define MN_DOWN(WQ_)                                                                            \
  do {                                                                                          \
    if (nck == 1) hipLaunchKernelGGL((moe_down_kernel<1, WQ_>), grid, block, 0, st, a);         \
    else if (nck == 2) hipLaunchKernelGGL((moe_down_kernel<2, WQ_>), grid, block, 0, st, a);    \
    else if (nck == 3) hipLaunchKernelGGL((moe_down_kernel<3, WQ_>), grid, block, 0, st, a);    \
    else hipLaunchKernelGGL((moe_down_kernel<4, WQ_>), grid, block, 0, st, a);                  \
  } while (0)
  if (wfmt == MN_W_FP8_E4M3) MN_DOWN(1); else if (wfmt == MN_W_INT8) MN_DOWN(2); else if (wfmt == MN_W_NF4) MN_DOWN(3); else MN_DOWN(0);
#undef MN_DOWN
  MN_CHECK_LAUNCH("moe_down_rows");
  return MN_OK;
}
