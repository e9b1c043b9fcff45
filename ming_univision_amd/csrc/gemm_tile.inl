// gemm_tile.inl — the small-tile form of gemm256.hip's GEMM, for problems whose 256 x 256 tiles leave most of the chip idle
// (included inside gemm256.hip's anonymous namespace; same operands, pairing modes, split-K and epilogues).
//
// What bounds such a problem is not the matrix cores but latency: a 256-tile kernel on 36 workgroups (1025 hi/lo rows x 1024 columns) or a
// two-buffer 128-tile kernel on 24 .. 96 spends its time waiting for one K-tile after another (0.6 .. 1 us each from HBM / L2).  So:
//   * BM x BN tiles from 64 x 64 to 128 x 128, so that a few hundred workgroups exist;
//   * S stages of LDS (S - 1 K-tiles in flight per workgroup, filled by global_load_lds, retired by counted vmcnt): the first products wait for
//     one round trip, the rest stream;
//   * one barrier per K-tile: it says both that every wave's part of K-tile t has landed and that every wave has read K-tile t - 1, whose
//     buffer the loads of K-tile t + S - 1 may then overwrite.
// HILO: the LDS image of a K-tile holds BM hi rows, then the same rows' lo parts; both are multiplied into accumulators of their own (the
// sum is taken once, in the epilogue, as in the 256-tile kernel).
// TWO: the hi products of a K-tile's halves go to two accumulators, so that a chain of fp32 additions is half as long, as it is in the K-slices that the flow head's few
// rows had before these tiles: latents against 64 bits at 16 rows, 2 x 96 draws, 7.59e-6 and 7.73e-6 with one chain, 7.49e-6 and 7.56e-6 with two (slices: 7.50e-6
// and 7.63e-6); the time is the same (a sampler call of 16 rows 8.13 ms; a total every 8 K-tiles instead of a second accumulator 8.25).
template <int N>
__device__ __forceinline__ void wait_vm_n() { asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N) : "memory"); }

// all but `rem` K-tiles of L loads each have landed, and this wave's fragment reads are done (rem <= MAX, wave-uniform)
template <int L, int MAX>
__device__ __forceinline__ void wait_tiles(int rem) {
  if constexpr (MAX == 0) {
    wait_vm_n<0>();
  } else {
    if (rem >= MAX) wait_vm_n<L * MAX>();
    else wait_tiles<L, MAX - 1>(rem);
  }
}

// GROUP 1, 2: the products of groups of rows with weights of their own (MoE experts), row tiles of BM from a device-built list.  2 and 3 (one dense product): the weights are read past
// the caches, where all rows, or most groups, are one row tile: nobody reads them again, and lines that are let go at once stream faster (66 experts' 2816 x 2048 / 2048 x 1408 of 100
// rows in tiles of 32 x 128, 6 picks a row and two for all: 146 -> 140 us / 74 -> 70, 70 rows 146 -> 135 / 73 -> 67, 5.6 TB/s; 240 rows, where a third of the groups are two tiles, 162 -> 165 /
// 87 -> 89).  4: one dense product, tiles in bands (order_band; a kernel of its own, as the divisions behind a branch cost every small product 0.2 us of 4 .. 8).
template <int EPI, bool HILO, int BM, int BN, int WM, int WN, int S, bool TWO = false, int GROUP = 0>
__global__ __launch_bounds__(WM * WN * 64) void gemm_tile_kernel(const G256 p) {
  constexpr int NW = WM * WN, AR = HILO ? 2 * BM : BM, QA = AR / 8 / NW, QW = BN / 8 / NW, STAGE = (AR + BN) * 128;
  constexpr int MI = BM / WM / 16, NJ = BN / WN / 16, AI = HILO ? 2 * MI : MI;
  constexpr bool paired = epi_paired(EPI), GROUPED = GROUP == 1 || GROUP == 2;
  constexpr bool quads = paired && NJ == 1;            // gate and up of a unit within one fragment: a lane's 4 columns are 2 gates, then their 2 ups
  static_assert(QA * 8 * NW == AR && QW * 8 * NW == BN && MI >= 1 && NJ >= 1 && (!quads || EPI == E_SWIGLU_SPLIT), "whole instructions and fragments per wave");
  static_assert((QA + QW) * (S - 2) < 64 && S * STAGE <= 160 * 1024, "vmcnt range, LDS");
  __shared__ __attribute__((aligned(1024))) char lds[S * STAGE];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WN, wn = wave % WN, fr = lane & 15, fq = lane >> 4;
  constexpr int cols = paired ? BN / 2 : BN;
  const int tiles_m = (p.M + BM - 1) / BM;
  // XCD-aware order: an XCD's tiles are consecutive, row tiles fastest, so each XCD reads its own part of the weights and all of the rows
  int bid = blockIdx.x, nt = gridDim.x, nl = 0;
  const int tiles_n = (p.N + cols - 1) / cols;
  if constexpr (GROUPED) {
    nl = *p.n_tiles;
    nt = min(nt, nl * tiles_n);                        // the live tiles
    if (bid >= nt) return;                             // uniform
  }
  {
    const int q = nt / 8, r = nt % 8, xcd = bid % 8, idx = bid / 8;
    bid = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + idx;
  }
  int m0, n0, row0 = 0, Mg = p.M, grp = 0;
  if constexpr (GROUPED) {                             // column tiles fastest (bands of four row tiles: the same to 4 % slower)
    const int t = bid / tiles_n;
    grp = p.tile_g[t];
    m0 = p.tile_m0[t];
    n0 = (bid - t * tiles_n) * cols;
    row0 = p.g_off[grp];
    Mg = p.g_cnt[grp];
  } else {
    int tm = bid % tiles_m, tn = bid / tiles_m;
    if constexpr (GROUP == 4) {                        // bands of column tiles, row by row
      const int per = tiles_m * p.group_m, b = bid / per, in = bid - b * per, w = min(p.group_m, tiles_n - b * p.group_m);
      tm = in / w;
      tn = b * p.group_m + in - tm * w;
    }
    m0 = tm * BM;
    n0 = tn * cols;
  }
  const int kbeg = blockIdx.y * p.Kc, kend = min(p.K, kbeg + p.Kc);
  const int nk = (kend - kbeg) / BK;

  // per-lane byte offsets (from A / W) of the row behind each 8-row instruction of this wave, k-slot swizzle folded in
  uint32_t srcA[QA], srcW[QW];
  const int rin = lane >> 3;
#pragma unroll
  for (int q = 0; q < QA; ++q) {
    const int L = (wave * QA + q) * 8 + rin;
    int gm = row0 + min(m0 + (HILO && L >= BM ? L - BM : L), Mg - 1);
    if (GROUPED && p.a_rows) gm = p.a_rows[gm];
    srcA[q] = (uint32_t)(((int64_t)gm * p.lda + (HILO && L >= BM ? p.a_lo_off : 0) + kbeg) * 2 + (((lane & 7) ^ ((L >> 1) & 7)) << 4));
  }
#pragma unroll
  for (int q = 0; q < QW; ++q) {
    const int L = (wave * QW + q) * 8 + rin;
    int gn;
    if (quads) {
      gn = min(n0 + (L >> 4) * 8 + ((L >> 2) & 3) * 2 + (L & 1), p.N - 1) + (L & 2 ? (int)p.w_pair_rows : 0);
    } else if (paired) {                               // a wave's columns: its gate rows, then the up rows of the same units
      constexpr int WC = BN / WN, half = WC / 2;
      const int w = L / WC, r = L % WC;
      gn = min(n0 + w * half + (r % half), p.N - 1) + (r >= half ? (int)p.w_pair_rows : 0);
    } else {
      gn = min(n0 + L, p.N - 1);
    }
    srcW[q] = (uint32_t)(((int64_t)gn * p.ldw + kbeg) * 2 + (((lane & 7) ^ ((L >> 1) & 7)) << 4));
  }
  const char* Ab = reinterpret_cast<const char*>(p.A);
  const char* Wb = reinterpret_cast<const char*>(p.W) + (GROUPED ? (int64_t)grp * p.w_gstride * 2 : 0);
  auto stage = [&](int kt, int buf) {
    const uint32_t koff = (uint32_t)kt * (BK * 2);
    char* dst = &lds[buf * STAGE];
#pragma unroll
    for (int q = 0; q < QW; ++q)
      __builtin_amdgcn_global_load_lds((glb_void*)(Wb + (srcW[q] + koff)), (lds_void*)(dst + AR * 128 + (wave * QW + q) * 1024), 16, 0, GROUP == 2 || GROUP == 3 ? 2 : 0);
#pragma unroll
    for (int q = 0; q < QA; ++q)
      __builtin_amdgcn_global_load_lds((glb_void*)(Ab + (srcA[q] + koff)), (lds_void*)(dst + (wave * QA + q) * 1024), 16, 0, 0);
  };
  int lane_off[2];
#pragma unroll
  for (int kk = 0; kk < 2; ++kk) lane_off[kk] = fr * 128 + (((4 * kk + fq) ^ ((fr >> 1) & 7)) << 4);
  f32x4 acc[AI][NJ];
#pragma unroll
  for (int i = 0; i < AI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  f32x4 odd[TWO ? MI : 1][NJ];
  if constexpr (TWO) {
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j) odd[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  }

#pragma unroll
  for (int t = 0; t < S - 1; ++t)
    if (t < nk) stage(t, t);
  int buf = 0, nbuf = S - 1;
  for (int t = 0; t < nk; ++t) {
    wait_tiles<QA + QW, S - 2>(nk - 1 - t);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    if (t + S - 1 < nk) stage(t + S - 1, nbuf);
    const char* a = &lds[buf * STAGE + wm * (BM / WM) * 128];
    if (GROUPED && m0 + wm * (BM / WM) >= Mg) {          // uniform: no row of this wave is live
      buf = buf + 1 == S ? 0 : buf + 1;
      nbuf = nbuf + 1 == S ? 0 : nbuf + 1;
      continue;
    }
    const char* w = &lds[buf * STAGE + AR * 128 + wn * (BN / WN) * 128];
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      bf16x8 af[AI], wf[NJ];
#pragma unroll
      for (int j = 0; j < NJ; ++j) wf[j] = *reinterpret_cast<const bf16x8*>(w + j * 2048 + lane_off[kk]);
#pragma unroll
      for (int i = 0; i < AI; ++i) af[i] = *reinterpret_cast<const bf16x8*>(a + (i < MI ? i * 2048 : BM * 128 + (i - MI) * 2048) + lane_off[kk]);
#pragma unroll
      for (int i = 0; i < AI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
          f32x4& c = TWO && kk == 1 && i < MI ? odd[TWO ? i % MI : 0][j] : acc[i][j];
          c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[j], af[i], c, 0, 0, 0);
        }
    }
    buf = buf + 1 == S ? 0 : buf + 1;
    nbuf = nbuf + 1 == S ? 0 : nbuf + 1;
  }

  if constexpr (TWO) {
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j) acc[i][j] += odd[i][j];
  }

  char* Cz = reinterpret_cast<char*>(p.C);
  if (EPI == E_F32) Cz += (int64_t)blockIdx.y * p.c_zstride * 4;
  if constexpr (quads) {
    const int n = n0 + wn * 8 + fq * 2;                // two units (N % 4 == 0: both in or both out)
    float bg[2] = {0.f, 0.f}, bu[2] = {0.f, 0.f};
    if (p.bias && n < p.N) {
#pragma unroll
      for (int e = 0; e < 2; ++e) { bg[e] = bf16_to_f32(p.bias[n + e]); bu[e] = bf16_to_f32(p.bias[p.w_pair_rows + n + e]); }
    }
#pragma unroll
    for (int i = 0; i < MI; ++i) {
      const int m = m0 + i * 16 + fr;
      if (m >= p.M || n >= p.N) continue;
      f32x4 v = acc[i][0];
      if (HILO) v += acc[(i + MI) % AI][0];
      uint32_t hi, lo;
      split_pk_bf16(silu_f(v.x + bg[0]) * (v.z + bu[0]), silu_f(v.y + bg[1]) * (v.w + bu[1]), hi, lo);
      bf16_t* c = reinterpret_cast<bf16_t*>(p.C) + (int64_t)m * p.ldc + n;
      *reinterpret_cast<uint32_t*>(c) = hi;
      *reinterpret_cast<uint32_t*>(c + p.c_lo_off) = lo;
    }
    return;
  }
  g256_out<EPI, false, MI, paired ? (NJ + 1) / 2 : NJ>(
      p, Cz, blockIdx.y, row0, Mg, grp, [&](int i) { return m0 + wm * (BM / WM) + i * 16 + fr; }, [&](int j) { return n0 + wn * (cols / WN) + j * 16 + fq * 4; },
      [&](int i, int j, f32x4& v, f32x4& u) {
        v = acc[i][j];
        if (HILO) v += acc[(i + MI) % AI][j];
        if (paired) { u = acc[i][(j + NJ / 2) % NJ]; if (HILO) u += acc[(i + MI) % AI][(j + NJ / 2) % NJ]; }
      });
}
