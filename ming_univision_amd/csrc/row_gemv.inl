// row_gemv.inl — a product of ONE row whose weights are one round trip: bf16 W [N or 2 N, K], N rows over all the CUs' waves at once (included inside skinny_gemm.hip's
// anonymous namespace; same prologues and epilogues).
//
// Such a launch is latency: 12 MB of weights are 2 us of memory, and the kernel that stages its row in LDS has its round trips one behind the other: the row, its square sum through
// two barriers, the norm's gain, a ring of chunks.  Here a wave asks for everything at once, its R weight rows first, then the row, gain, bias and residual, norms the row by itself in
// registers (NCK chunks of 512, 8 values a lane) and stores: nothing crosses waves, no LDS, no barrier.  A workgroup is 4 waves where 3 rows each are enough, else 8: a wave more is the row
// once more from L2.  us a launch with weights from memory, staged -> here (the sums' order is the same): behind an RMSNorm 3072 x 2048 6.6 -> 5.0, behind a LayerNorm 3072 x 1024 5.5 -> 3.8, 2736
// units of 1024 6.6 -> 4.9; 2048 x 2048 5.0 -> 3.9, 1024 x 2736 6.1 -> 3.6, 1024 x 1024 3.7 -> 2.5, 8192 x 2048 8.9 -> 8.0, 4096 units of 1024 6.6 -> 5.2, 64 x 2048 4.3 -> 2.6.
// GATE (4 waves of 2 rows, N % 8 == 0): the outputs are the row that a 64-expert router reads behind an RMSNorm, and the launch leaves its share of that for the next one: the workgroup's 8 outputs
// times their gains and gate columns, part [N / 8][64], and their square sum, part [N / 8][64] + [N / 8]; the norm's scale, known once all are there, goes on the sums.  The gate is then
// read once by the whole launch, 8 columns a workgroup under the weights' round trip, where every workgroup of the next one read all of it (moe_gate_up.hip): 4.2 - 4.6 us with and without here, 22.4 -> 17.7 there.
struct RowGemv { mn_skinny_args a; const bf16_t* gate_w; const bf16_t* gain; float* part; int experts; };

template <int NCK, int R, int SW, bool NORM, bool GATE = false>
__global__ __launch_bounds__(512, 2) void row_gemv_kernel(const RowGemv p) {
  typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));
  const mn_skinny_args& a = p.a;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), N = a.N, K = a.K;
  const int n0 = (blockIdx.x * (blockDim.x >> 6) + wave) * R;
  if (n0 >= N) return;
  __shared__ float hs[GATE ? 8 : 1];
  u32x4 gq = {0u, 0u, 0u, 0u}, gg = {0u, 0u, 0u, 0u};
  u32x4 w[SW][R][NCK];
#pragma unroll
  for (int s = 0; s < SW; ++s)
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const bf16_t* wr = a.w + (int64_t)(min(n0 + r, N - 1) + s * N) * a.ldw;
#pragma unroll
      for (int c = 0; c < NCK; ++c) w[s][r][c] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(wr + min(c * 512 + lane * 8, K - 8)));      // (past K: any finite values, the row is zero there)
    }
  float x[NCK][8];
#pragma unroll
  for (int c = 0; c < NCK; ++c) {
    const int k = c * 512 + lane * 8, kc = min(k, K - 8);
    const f4u lo = *reinterpret_cast<const f4u*>(a.x + kc), hi = *reinterpret_cast<const f4u*>(a.x + kc + 4);
#pragma unroll
    for (int e = 0; e < 4; ++e) { x[c][e] = k < K ? lo[e] : 0.f; x[c][4 + e] = k < K ? hi[e] : 0.f; }
  }
  const int pro = a.prologue;
  u32x4 g[NORM ? NCK : 1], b[NORM ? NCK : 1];
  if constexpr (NORM) {
#pragma unroll
    for (int c = 0; c < NCK; ++c) {
      const int kc = min(c * 512 + lane * 8, K - 8);
      g[c] = u32x4{0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u};
      b[c] = u32x4{0u, 0u, 0u, 0u};
      if (a.ln_g) g[c] = *reinterpret_cast<const u32x4*>(a.ln_g + kc);
      if (a.ln_b && pro == MN_PRO_LN) b[c] = *reinterpret_cast<const u32x4*>(a.ln_b + kc);
    }
  }
  if constexpr (GATE) {
    if (wave == 0) {                                                    // lane e: expert e's 8 weights for these outputs
      gq = *reinterpret_cast<const u32x4*>(p.gate_w + (int64_t)min(lane, p.experts - 1) * N + n0);
      gg = *reinterpret_cast<const u32x4*>(p.gain + n0);
    }
  }
  // lane r: what output n0 + r needs beside its sums
  const int n = min(n0 + min(lane, R - 1), N - 1);
  float b0 = 0.f, b1 = 0.f, res = 0.f, gate = 1.f;
  if (a.bias) { b0 = bf16_to_f32(a.bias[n]); if (SW == 2) b1 = bf16_to_f32(a.bias[n + N]); }
  if (a.epilogue == MN_EPI_RESID || a.epilogue == MN_EPI_RESID_GATE) res = a.res[n];
  if (a.epilogue == MN_EPI_RESID_GATE) gate = a.gate[n];
  if constexpr (NORM) {
    float mean = 0.f, ss = 0.f;
    if (pro == MN_PRO_LN) {
#pragma unroll
      for (int c = 0; c < NCK; ++c) ss += ((x[c][0] + x[c][1]) + (x[c][2] + x[c][3])) + ((x[c][4] + x[c][5]) + (x[c][6] + x[c][7]));
      mean = wave_sum(ss) / (float)K;
      ss = 0.f;
    }
#pragma unroll
    for (int c = 0; c < NCK; ++c) {
      float q = 0.f;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        x[c][e] = c * 512 + lane * 8 < K ? x[c][e] - mean : 0.f;
        q = fmaf(x[c][e], x[c][e], q);
      }
      ss += q;
    }
    const float rstd = rsqrtf(wave_sum(ss) / (float)K + a.eps);
#pragma unroll
    for (int c = 0; c < NCK; ++c)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        x[c][2 * e] = x[c][2 * e] * rstd * bf16lo_to_f32(g[c][e]) + bf16lo_to_f32(b[c][e]);
        x[c][2 * e + 1] = x[c][2 * e + 1] * rstd * bf16hi_to_f32(g[c][e]) + bf16hi_to_f32(b[c][e]);
        if (c * 512 + lane * 8 >= K) x[c][2 * e] = x[c][2 * e + 1] = 0.f;
      }
  } else if (pro == MN_PRO_SILU) {
#pragma unroll
    for (int c = 0; c < NCK; ++c)
#pragma unroll
      for (int e = 0; e < 8; ++e) x[c][e] = silu_f(x[c][e]);
  }
  float y = 0.f, y2 = 0.f;
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int s = 0; s < SW; ++s) {
      float t = 0.f;
#pragma unroll
      for (int c = 0; c < NCK; ++c)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          t = fmaf(bf16lo_to_f32(w[s][r][c][e]), x[c][2 * e], t);
          t = fmaf(bf16hi_to_f32(w[s][r][c][e]), x[c][2 * e + 1], t);
        }
      t = wave_sum(t);
      if (lane == r) { if (s == 0) y = t; else y2 = t; }
      __builtin_amdgcn_sched_barrier(0);                                // (a row's weights are widened where they are used)
    }
  if (!GATE && (lane >= R || n0 + lane >= N)) return;
  y += b0;
  y2 += b1;
  switch (a.epilogue) {
    case MN_EPI_SILU: y = silu_f(y); break;
    case MN_EPI_GELU: y = gelu_erf_f(y); break;
    case MN_EPI_SWIGLU: y = silu_f(y) * y2; break;
    case MN_EPI_GEGLU_TANH: y = gelu_tanh_f(y) * y2; break;
    case MN_EPI_RESID: y += res; break;
    case MN_EPI_RESID_GATE: y = res + gate * y; break;
    default: break;
  }
  if constexpr (GATE) {
    if (lane < R) { a.out[n] = y; hs[wave * R + lane] = y; }
    __syncthreads();
    if (wave != 0) return;
    float t = 0.f, q = 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float h0 = hs[2 * e], h1 = hs[2 * e + 1];
      t = fmaf(bf16lo_to_f32(gq[e]) * bf16lo_to_f32(gg[e]), h0, t);      // (a product of two bf16 values is exact)
      t = fmaf(bf16hi_to_f32(gq[e]) * bf16hi_to_f32(gg[e]), h1, t);
      q = fmaf(h0, h0, q);
      q = fmaf(h1, h1, q);
    }
    if (lane < p.experts) p.part[(int64_t)blockIdx.x * 64 + lane] = t;
    if (lane == 0) p.part[(int64_t)gridDim.x * 64 + blockIdx.x] = q;
  } else {
    a.out[n] = y;
  }
}

// One row of one matrix, where a wave's weights (R rows, gate and up; at most 32 pieces of 16 bytes a lane, 4 K values behind no norm and 2 K behind one) are in flight at once with a wave
// for every row: up to 24 MB, 33 MB of 2 K.  Beyond (12288 x 2048 11.2 and 11.1 us, 16384 x 1024 8.9 and 8.9) the ring streams as fast.  Not where the output lies over the row: a wave stores while
// another still reads.  false: another kernel's.
bool row_gemv(const mn_skinny_args& a, hipStream_t st, const bf16_t* gate_w = nullptr, const bf16_t* gain = nullptr, int experts = 0, float* part = nullptr) {
  auto al = [](const void* q) { return ((uintptr_t)q & 15) == 0; };
  if (a.M != 1 || a.wfmt != MN_W_BF16 || a.K > 4096 || a.w_index || a.seg_index || a.seg_scale || !(a.x + a.K <= a.out || a.out + a.N <= a.x) ||
      !(a.prologue == MN_PRO_NONE || a.prologue == MN_PRO_SILU || a.prologue == MN_PRO_RMSNORM || a.prologue == MN_PRO_LN) || !al(a.ln_g) || !al(a.ln_b)) return false;
  const int sw = mn_epi_pairs(a.epilogue) ? 2 : 1, nck = (a.K + 511) / 512, cus = mn_num_cus();
  int waves = 4, R = (int)mn_cdiv(a.N, (int64_t)cus * 4);
  auto fits = [&](int r) { return r <= 6 && r * sw * (nck <= 2 ? nck : (nck + 1) / 2 * 2) <= 32; };
  if (R == 5) R = 6;
  if (!fits(R) || R > 3) { waves = 8; R = (int)mn_cdiv(a.N, (int64_t)cus * 8); if (R == 5) R = 6; }
  if (!fits(R)) return false;
  const RowGemv p{a, gate_w, gain, part, experts};
  const dim3 grid((unsigned)mn_cdiv(mn_cdiv(a.N, R), waves)), block((unsigned)waves * 64);
  const bool norm = a.prologue >= MN_PRO_RMSNORM;
  if (part) {
    if (norm || sw != 1 || waves != 4 || R != 2 || (a.N % 8) || experts < 1 || experts > 64 || !al(gate_w) || !al(gain)) return false;
    switch (nck) {
      case 1: hipLaunchKernelGGL((row_gemv_kernel<1, 2, 1, false, true>), grid, block, 0, st, p); return true;
      case 2: hipLaunchKernelGGL((row_gemv_kernel<2, 2, 1, false, true>), grid, block, 0, st, p); return true;
      case 3: case 4: hipLaunchKernelGGL((row_gemv_kernel<4, 2, 1, false, true>), grid, block, 0, st, p); return true;
      case 5: case 6: hipLaunchKernelGGL((row_gemv_kernel<6, 2, 1, false, true>), grid, block, 0, st, p); return true;
      default: hipLaunchKernelGGL((row_gemv_kernel<8, 2, 1, false, true>), grid, block, 0, st, p); return true;
    }
  }
#define MN_RG(C_, R_, S_, N_) hipLaunchKernelGGL((row_gemv_kernel<C_, R_, S_, N_>), grid, block, 0, st, p)
#define MN_RG_N(C_, R_, S_)                                                                    \
  do {                                                                                         \
    if constexpr (C_ <= 4) { if (norm) { MN_RG(C_, R_, S_, true); return true; } }             \
    if (!norm) { MN_RG(C_, R_, S_, false); return true; }                                      \
    return false;                                                                              \
  } while (0)
#define MN_RG_S(C_, R_)                                                                        \
  do {                                                                                         \
    if constexpr (R_ * C_ * 2 <= 32) { if (sw == 2) MN_RG_N(C_, R_, 2); }                      \
    if constexpr (R_ * C_ <= 32) { if (sw == 1) MN_RG_N(C_, R_, 1); }                          \
    return false;                                                                              \
  } while (0)
#define MN_RG_R(C_) do { switch (R) { case 1: MN_RG_S(C_, 1); case 2: MN_RG_S(C_, 2); case 3: MN_RG_S(C_, 3); case 4: MN_RG_S(C_, 4); default: MN_RG_S(C_, 6); } } while (0)
  switch (nck) {
    case 1: MN_RG_R(1);
    case 2: MN_RG_R(2);
    case 3: case 4: MN_RG_R(4);
    case 5: case 6: MN_RG_R(6);
    default: MN_RG_R(8);
  }
#undef MN_RG_R
#undef MN_RG_S
#undef MN_RG_N
#undef MN_RG
}
