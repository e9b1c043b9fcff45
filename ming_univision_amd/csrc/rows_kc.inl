// rows_kc.inl — a Linear of 2 .. 32 rows in one launch (included inside skinny_gemm.hip's anonymous namespace).
//
// The three-launch form (split the rows into hi / lo, stream the weights in K-slices, sum the slices) pays 4 .. 6 us for each of its small launches; at
// the sizes of a decoder's projections that is more than the product.  Here a workgroup owns NT tiles of 16 columns with ALL of K: its 8 waves take
// 64-value chunks of K in turn, read weights and fp32 rows straight into MFMA operands (lane l: row / column l & 15, values 8 (l >> 4) .. + 7
// of every 32), split the rows there into three bf16 parts (24 bits: products of all of an fp32 value of 2^-110 and more; the last bits of
// smaller ones fall off bf16's subnormals: 1e-7 of the summed magnitudes at rows around 2^-114, 2e-6 at 2^-118) and meet once, in LDS, for the sum of the eight
// waves' tiles and the epilogue.  A chunk's sum joins the running one with its rounding kept (two-sum): 1.5e-8 of the summed magnitudes off 64 bits at
// the most, 2.0e-8 on the fp32 FMA kernel, 4e-7 as hi + lo.  Every workgroup reads all rows (M K 4 bytes, from L2), every weight byte is read once; the
// next chunk's loads are in flight during a chunk's products.  What bounds it is the load and conversion of the rows (0.85 us + 0.042 a row for each 512
// values of K; weights two or four chunks ahead, or 8-byte pieces that coalesce better, changed nothing or cost 25 %).  2048 x 2048: 6.2 us at 2 rows, 8.2 at
// 16, 12.1 at 32 (10.0, 11.3, 13.7 as three launches); 4096 x 1024 4.6, 5.7, 8.0 (9.6, 10.9, 13.1).
// RMSNorm: the gain multiplies the values, 1 / rms the sums (each wave adds up the squares of its chunks).
// Paired epilogues (gate, up): tile t < NT / 2 holds gate columns, tile t + NT / 2 the up columns of the same units.
typedef short bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));      // rows start at any float: a 16-byte load needs 4-byte alignment here

// a pair of values as three pairs of bf16, 24 bits.  ODD: of values that bf16 rounds to infinity; a finite one starts from the largest finite
// bf16, what is left of an infinite one is nothing (not inf - inf).
constexpr float BF16_TO_INF = 0x1.ffp127f, BF16_MAX = 0x1.fep127f;
template <bool ODD>
__device__ __forceinline__ void split3_pk_bf16(float a, float b, u32x4 (&part)[3], int at) {
  uint32_t h = ODD ? cvt_pk_bf16(fabsf(a) < INFINITY ? fminf(fmaxf(a, -BF16_MAX), BF16_MAX) : a, fabsf(b) < INFINITY ? fminf(fmaxf(b, -BF16_MAX), BF16_MAX) : b)
                   : cvt_pk_bf16(a, b);
  part[0][at] = h;
  a -= bf16lo_to_f32(h); b -= bf16hi_to_f32(h);
  if (ODD) { a = a == a ? a : 0.f; b = b == b ? b : 0.f; }
  h = cvt_pk_bf16(a, b);
  part[1][at] = h;
  part[2][at] = cvt_pk_bf16(a - bf16lo_to_f32(h), b - bf16hi_to_f32(h));
}

template <int MT, int NT, int PRO>
__global__ __launch_bounds__(512) void rows_kc_kernel(const mn_skinny_args a, int paired) {
  constexpr int NW = 8, CK = 64, R = MT * NT * 4;
  __shared__ float red[NW][R][64];
  __shared__ float sq[PRO == MN_PRO_RMSNORM ? NW : 1][16 * MT];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, r = lane & 15, q = lane >> 4;
  const int K = a.K, M = a.M, N = a.N, G = paired ? NT / 2 : NT;             // G: tiles of units per workgroup
  const int n0 = blockIdx.x * 16 * G;
  const bf16_t* wp[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) wp[t] = a.w + (int64_t)(min(n0 + 16 * (t % G) + r, N - 1) + (t >= G ? N : 0)) * K + 8 * q;
  const float *xp[MT], *pp[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const int m = min(16 * i + r, M - 1);
    xp[i] = a.x + (int64_t)m * a.ldx + 8 * q;
    pp[i] = PRO == MN_PRO_ADD_SILU ? a.pro_a + (int64_t)m * a.ld_pro_a + 8 * q : nullptr;
  }
  f32x4 acc[MT][NT], low[MT][NT], xf[MT][2][2];
  u32x4 wf[NT][2];
  float ss[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    ss[i] = 0.f;
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[i][t] = low[i][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  // K is a multiple of 8: a lane's 8 values are all inside K or all beyond it, where it reads its row's start and both operands become zeros
  auto fetch = [&](int k0) {
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int k = k0 + 32 * s, kk = k + 8 * q < K ? k : -8 * q;
#pragma unroll
      for (int t = 0; t < NT; ++t) wf[t][s] = *reinterpret_cast<const u32x4*>(wp[t] + kk);
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        xf[i][s][0] = *reinterpret_cast<const f32x4u*>(xp[i] + kk);
        xf[i][s][1] = *reinterpret_cast<const f32x4u*>(xp[i] + kk + 4);
      }
    }
  };
  if (wave * CK < K) fetch(wave * CK);
  for (int k0 = wave * CK; k0 < K; k0 += NW * CK) {
    f32x4 cx[MT][2][2];
    u32x4 cw[NT][2];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
#pragma unroll
      for (int t = 0; t < NT; ++t) cw[t][s] = wf[t][s];
#pragma unroll
      for (int i = 0; i < MT; ++i) { cx[i][s][0] = xf[i][s][0]; cx[i][s][1] = xf[i][s][1]; }
    }
    if (k0 + NW * CK < K) fetch(k0 + NW * CK);
    f32x4 sum[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int t = 0; t < NT; ++t) sum[i][t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int k = k0 + 32 * s + 8 * q;
      const bool in = k < K;
      f32x4 g0, g1;
      if (PRO == MN_PRO_RMSNORM) {
        const u32x4 gw = *reinterpret_cast<const u32x4*>(a.ln_g + (in ? k : 0));
        g0 = f32x4{bf16lo_to_f32(gw.x), bf16hi_to_f32(gw.x), bf16lo_to_f32(gw.y), bf16hi_to_f32(gw.y)};
        g1 = f32x4{bf16lo_to_f32(gw.z), bf16hi_to_f32(gw.z), bf16lo_to_f32(gw.w), bf16hi_to_f32(gw.w)};
      }
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        f32x4 v0 = cx[i][s][0], v1 = cx[i][s][1];
        if (PRO == MN_PRO_ADD_SILU) {
          const int kk = in ? k - 8 * q : -8 * q;
          v0 += *reinterpret_cast<const f32x4u*>(pp[i] + kk);
          v1 += *reinterpret_cast<const f32x4u*>(pp[i] + kk + 4);
        }
        if (PRO == MN_PRO_SILU || PRO == MN_PRO_ADD_SILU) {
#pragma unroll
          for (int e = 0; e < 4; ++e) { v0[e] = silu_f(v0[e]); v1[e] = silu_f(v1[e]); }
        }
        if (!in) v0 = v1 = f32x4{0.f, 0.f, 0.f, 0.f};
        if (PRO == MN_PRO_RMSNORM) {
#pragma unroll
          for (int e = 0; e < 4; ++e) ss[i] = fmaf(v0[e], v0[e], fmaf(v1[e], v1[e], ss[i]));
          v0 *= g0; v1 *= g1;
        }
        u32x4 part[3];
        float most = 0.f;
#pragma unroll
        for (int e = 0; e < 4; ++e) most = fmaxf(most, fmaxf(fabsf(v0[e]), fabsf(v1[e])));
        if (__ballot(most >= BF16_TO_INF) == 0) {
#pragma unroll
          for (int e = 0; e < 2; ++e) { split3_pk_bf16<false>(v0[2 * e], v0[2 * e + 1], part, e); split3_pk_bf16<false>(v1[2 * e], v1[2 * e + 1], part, 2 + e); }
        } else {
#pragma unroll
          for (int e = 0; e < 2; ++e) { split3_pk_bf16<true>(v0[2 * e], v0[2 * e + 1], part, e); split3_pk_bf16<true>(v1[2 * e], v1[2 * e + 1], part, 2 + e); }
        }
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          const bf16x8 w = __builtin_bit_cast(bf16x8, in ? cw[t][s] : u32x4{0, 0, 0, 0});
#pragma unroll
          for (int p = 2; p >= 0; --p) sum[i][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, part[p]), w, sum[i][t], 0, 0, 0);
        }
      }
    }
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          float a0 = acc[i][t][e], l0 = low[i][t][e];
          two_sum(a0, l0, sum[i][t][e]);
          acc[i][t][e] = a0; low[i][t][e] = l0;
        }
  }
#pragma unroll
  for (int i = 0; i < MT; ++i) {
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float v = acc[i][t][e] + low[i][t][e];
        red[wave][(i * 4 + e) * NT + t][lane] = v == v ? v : acc[i][t][e];   // a sum at infinity has no error term
      }
    if (PRO == MN_PRO_RMSNORM) {
      ss[i] += __shfl_xor(ss[i], 16);
      ss[i] += __shfl_xor(ss[i], 32);
      if (q == 0) sq[wave][16 * i + r] = ss[i];
    }
  }
  __syncthreads();
  for (int j = wave; j < 4 * MT; j += NW) {                                  // row 16 (j / 4) + 4 q + j % 4 of every tile
    const int ml = 16 * (j >> 2) + 4 * q + (j & 3);
    float rstd = 1.f;
    if (PRO == MN_PRO_RMSNORM) {
      float t = 0.f;
#pragma unroll
      for (int w = 0; w < NW; ++w) t += sq[w][ml];
      rstd = rsqrtf(t / (float)K + a.eps);
    }
    float y[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      float p[NW];
#pragma unroll
      for (int w = 0; w < NW; ++w) p[w] = red[w][j * NT + t][lane];
      const float v = ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
      y[t] = PRO == MN_PRO_RMSNORM ? v * rstd : v;
    }
    if (ml >= M) continue;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int n = n0 + 16 * t + r;
      if (t >= G || n >= N) continue;
      medium_finish(a, ml, n, y[t], NT > 1 ? y[NT > 1 && paired ? t + NT / 2 : 0] : 0.f);
    }
  }
}

// The same with rows and weights on their way through LDS: a wave instruction fetches whole 64- or 128-byte pieces of a row (64 bytes a cycle and CU), where
// operands read straight from memory, 16 rows apart lane by lane, come at a quarter of that (38 GB/s a CU: 7 of 12 us for 32 rows of 2048).  Each wave has a ring of
// its own, so nothing but the sum at the end is a barrier.  What is left is the split (130 vector instructions for 32 values of 32 rows, 4 us of the
// 2048).  Rows of 16-byte aligned values; 2048 x 2048 at 32 rows 14.5 -> 11.1 us.  NX eights of rows are fetched, as many as there are: with sixteen of them always, 5 rows of
// 32000 x 1024 took 23.4 us beside other work, with eight 16.5.  Grid (tiles, rows / 8 NX): 17 .. 32 rows go 16 and the rest where a CU is free for either: half of the rows a CU takes in, and half of
// the split; the weights come a second time from L2 (us, 32 rows at once / in halves: 2048 x 2048 11.1 / 7.8, 2048 x 768 5.6 / 4.2, 1024 x 1024 6.5 / 4.6; 17
// rows of 2048 x 2048 10.5 / 7.4; against three launches 2048 x 4096 17.2 / 12.1).
template <int NX, int NT, int PRO>
__global__ __launch_bounds__(512) void rows_kc_lds_kernel(const mn_skinny_args a, int paired) {
  constexpr int MT = (NX + 1) / 2;                     // NX: eights of rows that are fetched
  constexpr int NW = 8, CK = 64, R = MT * NT * 4, S = 3, XB = NX * 1024, SUB = XB + NT * 1024;      // a ring holds S pieces of 32 values of K: rows of 128 bytes, then weights of 64
  constexpr int BYTES = NW * S * SUB > NW * R * 256 ? NW * S * SUB : NW * R * 256;
  __shared__ __attribute__((aligned(1024))) char lds[BYTES];
  float (*red)[R][64] = reinterpret_cast<float (*)[R][64]>(lds);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, r = lane & 15, q = lane >> 4;
  const int mb = blockIdx.y * (8 * NX), K = a.K, M = a.M - mb, N = a.N, G = paired ? NT / 2 : NT;      // mb: this workgroup's first row; G: tiles of units per workgroup
  const int n0 = blockIdx.x * 16 * G;
  // what this lane fetches: row 8 i + lane / 8 of the rows (16 bytes: slot lane % 8, in the order that leaves no bank twice), row lane / 4 of every weight tile
  typedef const __attribute__((address_space(1))) void gptr;
  typedef __attribute__((address_space(3))) void lptr;
  const int xr = lane >> 3, wr = lane >> 2;
  const float* xp[NX];
  int xk[NX];
#pragma unroll
  for (int i = 0; i < NX; ++i) {
    const int row = 8 * i + xr;
    xk[i] = 4 * ((lane & 7) ^ ((row >> 1) & 7));
    xp[i] = a.x + (int64_t)(mb + min(row, M - 1)) * a.ldx;
  }
  const int wk = 8 * ((lane & 3) ^ ((wr >> 2) & 3));
  const bf16_t* wp[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) wp[t] = a.w + (int64_t)(min(n0 + 16 * (t % G) + wr, N - 1) + (t >= G ? N : 0)) * K;
  char* ring = lds + wave * (S * SUB);
  f32x4 acc[MT][NT], low[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i) {
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[i][t] = low[i][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  // K is a multiple of 8: 8 values are all inside K or all beyond it, where the row's start is fetched and both operands become zeros
  const int pieces = wave * CK < K ? 2 * ((K - wave * CK + NW * CK - 1) / (NW * CK)) : 0;
  auto fetch = [&](int c, int buf) {
    const int k0 = (wave + NW * (c >> 1)) * CK + 32 * (c & 1);
    char* dst = ring + buf * SUB;
#pragma unroll
    for (int t = 0; t < NT; ++t) __builtin_amdgcn_global_load_lds((gptr*)(wp[t] + (k0 + wk < K ? k0 + wk : 0)), (lptr*)(dst + XB + t * 1024), 16, 0, 0);
#pragma unroll
    for (int i = 0; i < NX; ++i) __builtin_amdgcn_global_load_lds((gptr*)(xp[i] + (k0 + xk[i] < K ? k0 + xk[i] : 0)), (lptr*)(dst + i * 1024), 16, 0, 0);
  };
#pragma unroll
  for (int c = 0; c < S; ++c)
    if (c < pieces) fetch(c, c);
  int buf = 0;
  for (int c0 = 0; c0 < pieces; c0 += 2) {
    const int k0 = (wave + NW * (c0 >> 1)) * CK;
    f32x4 sum[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int t = 0; t < NT; ++t) sum[i][t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int k = k0 + 32 * s + 8 * q, left = pieces - 1 - c0 - s;
      const bool in = k < K;
      if (left >= 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * (NX + NT)) : "memory");
      else if (left == 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NX + NT) : "memory");
      else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      f32x4 cx[MT][2];
      u32x4 cw[NT];
      const char* src = ring + buf * SUB;
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int h = 0; h < 2; ++h) cx[i][h] = *reinterpret_cast<const f32x4*>(src + (2 * i + 1 < NX ? 16 * i + r : 16 * i + (r & 7)) * 128 + (((2 * q + h) ^ ((r >> 1) & (2 * i + 1 < NX ? 7 : 3))) << 4));
#pragma unroll
      for (int t = 0; t < NT; ++t) cw[t] = *reinterpret_cast<const u32x4*>(src + XB + t * 1024 + r * 64 + ((q ^ ((r >> 2) & 3)) << 4));
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      if (c0 + s + S < pieces) fetch(c0 + s + S, buf);           // the piece is in registers
      buf = buf + 1 == S ? 0 : buf + 1;
#pragma unroll
      for (int i = 0; i < MT; ++i) {
        f32x4 v0 = cx[i][0], v1 = cx[i][1];
        if (PRO == MN_PRO_SILU) {
#pragma unroll
          for (int e = 0; e < 4; ++e) { v0[e] = silu_f(v0[e]); v1[e] = silu_f(v1[e]); }
        }
        if (!in) v0 = v1 = f32x4{0.f, 0.f, 0.f, 0.f};
        u32x4 part[3];
        float most = 0.f;
#pragma unroll
        for (int e = 0; e < 4; ++e) most = fmaxf(most, fmaxf(fabsf(v0[e]), fabsf(v1[e])));
        if (__ballot(most >= BF16_TO_INF) == 0) {
#pragma unroll
          for (int e = 0; e < 2; ++e) { split3_pk_bf16<false>(v0[2 * e], v0[2 * e + 1], part, e); split3_pk_bf16<false>(v1[2 * e], v1[2 * e + 1], part, 2 + e); }
        } else {
#pragma unroll
          for (int e = 0; e < 2; ++e) { split3_pk_bf16<true>(v0[2 * e], v0[2 * e + 1], part, e); split3_pk_bf16<true>(v1[2 * e], v1[2 * e + 1], part, 2 + e); }
        }
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          const bf16x8 w = __builtin_bit_cast(bf16x8, in ? cw[t] : u32x4{0, 0, 0, 0});
#pragma unroll
          for (int p = 2; p >= 0; --p) sum[i][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, part[p]), w, sum[i][t], 0, 0, 0);
        }
      }
    }
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          float a0 = acc[i][t][e], l0 = low[i][t][e];
          two_sum(a0, l0, sum[i][t][e]);
          acc[i][t][e] = a0; low[i][t][e] = l0;
        }
  }
  __syncthreads();                                     // the rings are read: the tiles' sums take their place
#pragma unroll
  for (int i = 0; i < MT; ++i) {
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float v = acc[i][t][e] + low[i][t][e];
        red[wave][(i * 4 + e) * NT + t][lane] = v == v ? v : acc[i][t][e];   // a sum at infinity has no error term
      }
  }
  __syncthreads();
  for (int j = wave; j < 4 * MT; j += NW) {                                  // row 16 (j / 4) + 4 q + j % 4 of every tile
    const int ml = 16 * (j >> 2) + 4 * q + (j & 3);
    float y[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      float p[NW];
#pragma unroll
      for (int w = 0; w < NW; ++w) p[w] = red[w][j * NT + t][lane];
      y[t] = ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
    }
    if (ml >= M) continue;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int n = n0 + 16 * t + r;
      if (t >= G || n >= N) continue;
      medium_finish(a, mb + ml, n, y[t], NT > 1 ? y[NT > 1 && paired ? t + NT / 2 : 0] : 0.f);
    }
  }
}
