// mfma_f32_tiles.h — pieces shared by the attention kernels that run on the fp32 matrix cores (v_mfma_f32_16x16x4_f32: fp32
// operands, fp32 accumulate): staging 16-row tiles through registers into LDS, the LDS-only barrier, the hardware exponential, the walk of decode rows over latents.
// Operand layouts (lane l, c = l % 16, g = l / 16): A[row c][k g], B[k g][col c], D[row 4 g + i][col c] in VGPR i.
#pragma once
#include "common.h"

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

// Workgroup barrier that orders LDS traffic only: the compiler's __syncthreads also drains the global loads in flight, which would
// put the prefetched tile's memory latency back on every barrier of the key walk.
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
}

// exp on the hardware's base-2 exponential (one multiply + v_exp_f32, about 1e-6 relative over the softmax's range): the library
// expf is some forty instructions, and eight of them per 16-key tile in every wave were the larger part of the key walk's time
__device__ __forceinline__ float fast_exp(float x) { return __expf(x); }

typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));      // rows start at any float: a 16-byte load needs 4-byte alignment here

// four consecutive values src[d .. d + 3], zero from n on (VEC: n is a multiple of 4)
template <bool VEC>
__device__ __forceinline__ f32x4 load4(const float* src, int d, int n, bool on) {
  f32x4 t;
  if (VEC) {
    t = *reinterpret_cast<const f32x4u*>(src + (d < n ? d : 0));
    return on && d < n ? t : f32x4{0.f, 0.f, 0.f, 0.f};
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float x = src[d + e < n ? d + e : 0];
    t[e] = on && d + e < n ? x : 0.f;
  }
  return t;
}

// 16 rows x 64 NBW floats HBM -> registers (raw: a select on a loaded value would wait for it here) and registers -> LDS (zero from n on and in
// rows that do not count): 16 threads per row, 16 bytes per thread and pass
template <int NBW, bool VEC>
__device__ __forceinline__ void rows_fetch(f32x4 (&v)[NBW], const float* src, int n, int cg) {
#pragma unroll
  for (int ps = 0; ps < NBW; ++ps) {
    const int d = 4 * (cg + 16 * ps);
    if (VEC) {
      v[ps] = *reinterpret_cast<const f32x4u*>(src + (d < n ? d : 0));
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) v[ps][e] = src[d + e < n ? d + e : 0];
    }
  }
}
template <int NBW, int LDC, bool VEC>
__device__ __forceinline__ void rows_put(float* __restrict__ dst, const f32x4 (&v)[NBW], int n, int j, int cg, bool ok) {
#pragma unroll
  for (int ps = 0; ps < NBW; ++ps) {
    const int d = 4 * (cg + 16 * ps);
    f32x4 t = v[ps];
    if (VEC) {
      if (!(ok && d < n)) t = f32x4{0.f, 0.f, 0.f, 0.f};
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (!(ok && d + e < n)) t[e] = 0.f;
    }
    *reinterpret_cast<f32x4*>(dst + j * LDC + d) = t;
  }
}

// Decode rows over latents (values = the first columns of the keys): the key walk of one workgroup, 4 waves and up to 16 query vectors of one
// cache sequence.  Keys of n values come HBM -> registers -> one LDS tile of 16 KF keys while the tile before it is multiplied; everything is
// transposed, S^T[key, q] = K Q^T and O^T[d, q] += V^T P^T: every wave takes a quarter of a key's values for the scores (its slice of the
// queries stays in registers), the four partial score tiles meet in LDS and every wave sums them and takes the same softmax, whose weights are
// then the B operands of the value products as they lie; wave w owns the 16-column blocks w, w + 4, .. of the sums.  Three LDS-only
// barriers a tile.  What bounds it is memory (4 n bytes a key); the products need half of that time.
// kb: first key, ldk: its row stride, nk: keys of the sequence, mine: how many of them this lane's query (lane % 16) sees, [t0, t1): tiles.
// lrun comes back summed.
template <int NB, int KF, bool VEC, typename Score>
struct LatentWalk {
  static constexpr int KT = 16 * KF, LDK = 64 * NB + 4, LDS_S = KT + 4, LDS_FLOATS = KT * LDK + 4 * 16 * LDS_S;
  static __device__ __forceinline__ void run(float* __restrict__ lds, const float* kb, int64_t ldk, int n, int nk, int mine, int t0, int t1, const f32x4 (&q)[NB],
                                             Score score, float& mrun, float& lrun, f32x4 (&acc)[NB]) {
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, c = lane & 15, g4 = lane >> 4, fj = tid >> 4, fc = tid & 15;
    const int dw = wave * 16 * NB;
    float* K = lds;                      // [16 KF keys][LDK]
    float* Sp = lds + KT * LDK;          // [4 waves][16 q][LDS_S] partial scores
    int all = mine;
#pragma unroll
    for (int o = 1; o < 16; o <<= 1) all = min(all, __shfl_xor(all, o));
    all = __builtin_amdgcn_readfirstlane(all);
    mrun = -INFINITY;
    lrun = 0.f;
#pragma unroll
    for (int x = 0; x < NB; ++x) acc[x] = f32x4{0.f, 0.f, 0.f, 0.f};
    f32x4 vk[KF][NB];
    auto fetch = [&](int tile) {
#pragma unroll
      for (int f = 0; f < KF; ++f) rows_fetch<NB, VEC>(vk[f], kb + (int64_t)min(tile * KT + 16 * f + fj, nk - 1) * ldk, n, fc);
    };
    if (t0 < t1) fetch(t0);
    for (int tile = t0; tile < t1; ++tile) {
      const int key0 = tile * KT;
      lds_barrier();                     // the previous tile's values and partial scores are read
#pragma unroll
      for (int f = 0; f < KF; ++f) rows_put<NB, LDK, VEC>(K + 16 * f * LDK, vk[f], n, fj, fc, key0 + 16 * f + fj < nk);
      if (tile + 1 < t1) fetch(tile + 1);                      // in flight while this tile is multiplied
      lds_barrier();
      {
        f32x4 s[KF][2];
#pragma unroll
        for (int f = 0; f < KF; ++f) s[f][0] = s[f][1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int it = 0; it < NB; ++it) {
          f32x4 kf[KF];
#pragma unroll
          for (int f = 0; f < KF; ++f) kf[f] = *reinterpret_cast<const f32x4*>(K + (16 * f + c) * LDK + dw + 16 * it + 4 * g4);
#pragma unroll
          for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int f = 0; f < KF; ++f) s[f][e & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[f][e], q[it][e], s[f][e & 1], 0, 0, 0);
        }
#pragma unroll
        for (int f = 0; f < KF; ++f) *reinterpret_cast<f32x4*>(Sp + (wave * 16 + c) * LDS_S + 16 * f + 4 * g4) = s[f][0] + s[f][1];
      }
      lds_barrier();
      f32x4 p[KF];
      const bool whole = key0 + KT <= all;
      float mx = -INFINITY;
#pragma unroll
      for (int f = 0; f < KF; ++f) {
        const float* o = Sp + c * LDS_S + 16 * f + 4 * g4;
        p[f] = (*reinterpret_cast<const f32x4*>(o) + *reinterpret_cast<const f32x4*>(o + 16 * LDS_S)) +
               (*reinterpret_cast<const f32x4*>(o + 32 * LDS_S) + *reinterpret_cast<const f32x4*>(o + 48 * LDS_S));
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          p[f][i] = score(p[f][i]);
          if (!whole && key0 + 16 * f + 4 * g4 + i >= mine) p[f][i] = -INFINITY;
        }
        mx = fmaxf(mx, fmaxf(fmaxf(p[f][0], p[f][1]), fmaxf(p[f][2], p[f][3])));
      }
      mx = fmaxf(mx, __shfl_xor(mx, 16));
      mx = fmaxf(mx, __shfl_xor(mx, 32));
      const float mnew = fmaxf(mrun, mx);
      const float corr = mrun == -INFINITY ? 0.f : fast_exp(mrun - mnew);
      float sum = 0.f;
#pragma unroll
      for (int f = 0; f < KF; ++f)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          p[f][i] = p[f][i] == -INFINITY ? 0.f : fast_exp(p[f][i] - mnew);
          sum += p[f][i];
        }
      lrun = lrun * corr + sum;
      if (__ballot(mnew != mrun)) {      // some query's maximum moved
#pragma unroll
        for (int x = 0; x < NB; ++x) acc[x] *= corr;
      }
      mrun = mnew;
#pragma unroll
      for (int f = 0; f < KF; ++f)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          float v[NB];
#pragma unroll
          for (int x = 0; x < NB; ++x) v[x] = K[(16 * f + 4 * g4 + i) * LDK + 16 * (wave + 4 * x) + c];
#pragma unroll
          for (int x = 0; x < NB; ++x) acc[x] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[x], p[f][i], acc[x], 0, 0, 0);
        }
    }
    lrun += __shfl_xor(lrun, 16);
    lrun += __shfl_xor(lrun, 32);
  }
};

}  // namespace
