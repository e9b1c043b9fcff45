// delta_device.h — device pieces shared by the delta-rule operators (pnorm_ops.hip) and the operators with a decay per key channel
// (chan_ops.hip): gate functions, the 8-lane sum, the preparation of a row (filters, silu, unit norms, write strengths).
#pragma once
#include "common.h"

namespace {

__device__ __forceinline__ float sigmoid_f(float z) { return 1.0f / (1.0f + expf(-z)); }
__device__ __forceinline__ float silu_x(float z) { return z / (1.0f + expf(-z)); }
__device__ __forceinline__ float softplus_f(float z) { return z > 20.0f ? z : log1pf(expf(z)); }

__device__ __forceinline__ float sum8(float v) {                    // over the 8 lanes of an aligned group; every lane gets the sum
  return dpp_add<0x141>(dpp_add<0x4E>(dpp_add<0xB1>(v)));
}

// First row of the step's sequence j (its rows' row_back counts 0, 1, ..), -1 if the step has fewer: 256 threads, the same result in all of them.
// A launch of sequences x channels whose workgroups look theirs up beats one workgroup a row of which most find nothing to do: 1409 rows x 64
// workgroups with 35 KB of LDS each took 33 us to come and go.  (Rows beyond sequence_starts's table.)
__device__ __forceinline__ int sequence_start(const int32_t* __restrict__ row_back, int M, int j, uint64_t (&mask)[32]) {
  const int tid = threadIdx.x;
  for (int base = 0; base < M; base += 2048) {
    __syncthreads();                            // the masks of the rows (or the call) before are read
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int m = base + 256 * k + tid;
      const uint64_t b = __ballot(m < M && row_back[m < M ? m : 0] == 0);
      if ((tid & 63) == 0) mask[4 * k + (tid >> 6)] = b;
    }
    __syncthreads();
    for (int i = 0; i < 32; ++i) {
      uint64_t b = mask[i];
      const int c = __popcll(b);
      if (j < c) {
        for (; j > 0; --j) b &= b - 1;
        return base + 64 * i + __ffsll((unsigned long long)b) - 1;
      }
      j -= c;
    }
  }
  return -1;
}

// The step's sequences at once, where its rows are at most 2048: first[j] = sequence j's first row, first[count] = M; the count comes back (256 threads).  far (or null): does a wave see a
// sequence of `rows` rows?
__device__ __forceinline__ int sequence_starts(const int32_t* __restrict__ row_back, int M, uint64_t (&mask)[32], uint16_t (&first)[2049], int rows = 0, int* far = nullptr) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  bool there = false;
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const int m = 256 * k + tid, back = m < M ? row_back[m] : -1;
    const uint64_t b = __ballot(back == 0);
    there |= back + 1 >= rows;
    if (lane == 0) mask[4 * k + wave] = b;
  }
  if (far) {
    const bool any = __ballot(there) != 0;
    if (lane == 0) far[wave] = any;
  }
  __syncthreads();
  const int own = lane < 32 ? __popcll(mask[lane & 31]) : 0;
  int upto = own;
#pragma unroll
  for (int o = 1; o < 32; o <<= 1) {
    const int t = __shfl_up(upto, o, 64);
    upto += lane >= o ? t : 0;
  }
  const int count = __shfl(upto, 31, 64);
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const uint64_t b = mask[4 * k + wave];
    const int before = __shfl(upto - own, 4 * k + wave, 64);
    if ((b >> lane) & 1) first[before + __popcll(b & (((uint64_t)1 << lane) - 1))] = (uint16_t)(256 * k + tid);
  }
  if (tid == 0) first[count] = (uint16_t)M;
  __syncthreads();
  return __builtin_amdgcn_readfirstlane(count);
}

// Gated delta rule, preparation of a row: channels [q: G dim ; k: G dim ; v: H vdim] of the raw projections go through their causal
// filter (earlier inputs from the rows before it in this call, then from the sequence's state) and silu; q and k heads become unit
// vectors (q also times q_scale); beta = sigmoid(b), decay = exp(-exp(a_log) softplus(a + dt_bias)) (a_log NULL: no decay per head).
struct DeltaPrepArgs {
  const float* proj; int64_t ld;             // raw [q ; k ; v] at column 0, b at off_b, a at off_a
  int H, G, dim, vdim, taps, off_b, off_a;
  const bf16_t* w_conv;                      // [2 G dim + H vdim, taps], the last tap multiplies the current row
  float* state;                              // [n_seq, taps - 1, channels]
  int advance;                               // 1: every row is alone in its sequence and moves the state on by itself
  const float *a_log, *dt_bias;              // device fp32 [H]
  float unit_eps, q_scale;
  const int32_t *row_seq, *row_slot, *row_back;
  float* qkv; int64_t ldo;                   // [M, channels]
  float* bd; int64_t ldbd;                   // [M, 2 H]: beta, decay ([M, H]: beta)
};

__device__ __forceinline__ float conv_silu(const DeltaPrepArgs& a, int m, int c, int n, int seq, int slot, int back) {
  float acc = 0.f;
  for (int k = 0; k < a.taps; ++k) {
    float v = 0.f;
    if (k <= back) v = a.proj[(int64_t)(m - k) * a.ld + c];
    else if (slot - k >= 0) v = a.state[((int64_t)seq * (a.taps - 1) + (k - back - 1)) * n + c];
    acc = fmaf(bf16_to_f32(a.w_conv[(int64_t)c * a.taps + (a.taps - 1 - k)]), v, acc);
  }
  if (a.advance && a.taps > 1) {                // a one-row sequence: entry i becomes entry i - 1, entry 0 this row's input
    float* st = a.state + (int64_t)seq * (a.taps - 1) * n + c;
    for (int i = a.taps - 2; i >= 1; --i) st[(int64_t)i * n] = st[(int64_t)(i - 1) * n];
    st[0] = a.proj[(int64_t)m * a.ld + c];
  }
  return silu_x(acc);
}

// The same for filters of four taps, C channels c, c + 64, .. at once: all loads are on their way before the first is used (tap by tap, behind a branch each, a wave waited 4 C round trips: 1409
// rows of 8 heads of 128 + 128 18.7 -> 12.0 us, 45 MB; 1900 of 16 heads 44.9 -> 26.7).  Channels from `end` on count as the last one before it.
template <int C>
__device__ __forceinline__ void conv4_silu(const DeltaPrepArgs& a, int m, int c, int end, int n, int seq, int slot, int back, float (&out)[C]) {
  float v[C][4];
  ushort4 w[C];
#pragma unroll
  for (int j = 0; j < C; ++j) {
    const int cj = min(c + 64 * j, end - 1);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const bool here = k <= back, there = !here && slot - k >= 0;
      const float* p = there ? a.state + ((int64_t)seq * 3 + (k - back - 1)) * n + cj : a.proj + (int64_t)(m - (here ? k : 0)) * a.ld + cj;
      const float x = *p;
      v[j][k] = here || there ? x : 0.f;
    }
    w[j] = *reinterpret_cast<const ushort4*>(a.w_conv + (int64_t)cj * 4);
  }
#pragma unroll
  for (int j = 0; j < C; ++j) {
    float acc = bf16_to_f32(w[j].w) * v[j][0];
    acc = fmaf(bf16_to_f32(w[j].z), v[j][1], acc);
    acc = fmaf(bf16_to_f32(w[j].y), v[j][2], acc);
    out[j] = silu_x(fmaf(bf16_to_f32(w[j].x), v[j][3], acc));
  }
}

// one wave (back: rows of the same sequence directly before row m in this call): unit < 2 G = a q or k head of row m (its unit norm is a wave's reduction), then 256 value channels per unit
__device__ __forceinline__ void delta_prep_unit(const DeltaPrepArgs& a, int m, int unit, int lane, int back) {
  const int nqk = 2 * a.G * a.dim, nv = a.H * a.vdim, n = nqk + nv;
  const int seq = a.row_seq[m], slot = a.row_slot[m];
  float* out = a.qkv + (int64_t)m * a.ldo;
  if (!a.advance && a.taps == 4 && a.dim <= 128 && ((uintptr_t)a.w_conv & 7) == 0) {
    if (unit < 2 * a.G) {
      const int c0 = unit * a.dim;
      float v[2];
      conv4_silu<2>(a, m, c0 + lane, c0 + a.dim, n, seq, slot, back, v);
      const float ss = wave_sum((lane < a.dim ? v[0] * v[0] : 0.f) + (lane + 64 < a.dim ? v[1] * v[1] : 0.f)), r = (unit < a.G ? a.q_scale : 1.0f) / sqrtf(ss + a.unit_eps);
      if (lane < a.dim) out[c0 + lane] = v[0] * r;
      if (lane + 64 < a.dim) out[c0 + lane + 64] = v[1] * r;
    } else {
      const int e0 = (unit - 2 * a.G) * 256, end = min(nv, e0 + 256);
      if (e0 >= end) return;
      float v[4];
      conv4_silu<4>(a, m, nqk + e0 + lane, nqk + end, n, seq, slot, back, v);
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (e0 + lane + 64 * j < end) out[nqk + e0 + lane + 64 * j] = v[j];
    }
    return;
  }
  if (unit < 2 * a.G) {
    const int c0 = unit * a.dim;
    float ss = 0.f;
    for (int d = lane; d < a.dim; d += 64) {
      const float v = conv_silu(a, m, c0 + d, n, seq, slot, back);
      out[c0 + d] = v;
      ss = fmaf(v, v, ss);
    }
    ss = wave_sum(ss);
    const float r = (unit < a.G ? a.q_scale : 1.0f) / sqrtf(ss + a.unit_eps);
    for (int d = lane; d < a.dim; d += 64) out[c0 + d] *= r;      // the lane rereads what it wrote itself
  } else {
    const int e0 = (unit - 2 * a.G) * 256;
    for (int e = e0 + lane; e < min(nv, e0 + 256); e += 64) out[nqk + e] = conv_silu(a, m, nqk + e, n, seq, slot, back);
  }
}

// 256 threads: the write strengths (and decays) of row m
__device__ __forceinline__ void delta_prep_strengths(const DeltaPrepArgs& a, int m, int tid) {
  const float* row = a.proj + (int64_t)m * a.ld;
  for (int h = tid; h < a.H; h += 256) {
    a.bd[(int64_t)m * a.ldbd + h] = sigmoid_f(row[a.off_b + h]);
    if (a.a_log) a.bd[(int64_t)m * a.ldbd + a.H + h] = expf(-expf(a.a_log[h]) * softplus_f(row[a.off_a + h] + a.dt_bias[h]));
  }
}

inline int64_t delta_prep_units(int H, int G, int vdim) { return 2 * (int64_t)G + mn_cdiv((int64_t)H * vdim, 256); }

}  // namespace
