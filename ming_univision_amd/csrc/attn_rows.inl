// attn_rows.inl — attention of runs of rows on the fp32 matrix cores (included inside pmix_ops.hip's anonymous namespace).
//
// v_mfma_f32_16x16x4_f32: scores, weights and sums stay 32-bit.  What bounds it is the fp32 MFMA rate (157 TFLOP/s); everything else is laid out so
// that the products can follow each other.  A workgroup of 4 waves owns up to 64 query vectors of one key/value head — `hv` heads of 64 / hv
// rows, gathered from consecutive runs of the table — so a staged key tile serves 64 vectors.  (One run of 4 rows x 4 heads per
// workgroup, the form before, re-read every key for 16 vectors and put four barriers around every 16 keys: 27 TFLOP/s.)
// Both kernels multiply transposed, S^T[key, q] = K Q^T and O^T[d, q] += V^T P^T: a lane's four scores of a 16-key fragment are exactly the B
// operand of the value products of those keys (k slot g of step i = key 4 g + i), so the softmax of a query is four registers x two lane
// swaps and the weights never leave the registers.  Keys and values go HBM -> registers -> one of two LDS tiles while the other is multiplied.
// Runs of several sequences do not share a workgroup: each takes one of its own (attn_run).  A tile that none of the queries sees is skipped, one that
// all of them see whole takes no mask arithmetic.  Key splits write the partial layout of the merge kernel, run by run.

// A launch's workgroups: first the groups of every (head chunk, key split), then `alone` that take one run after the other.
// Workgroup x of the launch.  Where all are on the chip at once (two a CU), group by group of a (head chunk, split), every other CU-full the other way round, so that a CU holds a long walk and a
// short one.  Where they follow each other: the table's last groups (a sequence's long walks) first, the head chunks and splits of a group side by side, so that what is taken last is short; of the
// workgroups that start together the second half the other way round.
// Sequences whose workgroups are a multiple of 16 would meet on the CUs with their long walks (the launch's count is then one, which spares the others the look at the table, 1 us): where all are as
// long as the last one and a whole number of groups, as 64 runs of the table say, groups go by length, a group of every sequence after the other.
// us, every CU-full the other way round / the table's order backwards / as here: heads of 128, 16 over four, 8000 tokens 2984 / 2360 / 2340 (112 TFLOP/s), 4096 950 / 683 / 630, 2600 453 / 316 / 294,
// 1030 in two splits 115 / 81 / 70, window 1024 of 3000 280 / 246 / 249, 16 sequences of 512 326 / 246 / 195, 8 of 512 118 / 148 / 104, 16 of 256 72 / 92 / 69; over 16 of 64, 8 of 512 71 / 84 / 66; keys of
// 320 with the values inside, 5 prompts of 93 .. 470 in two splits 91 / 68 / 70, 10 of 384 146 / 153 / 103, 16 heads, 16 of 128 58 / 74 / 54.  Over 230 batches of equal prompts of 24 .. 1000 tokens 1 / 0.98 /
// 0.91 of the time on average, unequal ones 0.94.  What is left slower than the first form: many sequences of some 64 rows whose workgroups are no multiple of 16 (93 of 64, 8 heads of 128, 33 / 38 / 37).
constexpr int ROWS_CUS = 256;          // (the card's; as another argument it costs every kernel here scalar registers, which they spill: 16 heads of 64, 85 sequences of 48, 190 -> 205 us)
struct RowsItem { int group, gy, sp; };
__device__ __forceinline__ RowsItem rows_item(const AttnTArgs& a, int x, int groups, int nbw, int n_blk, int gys, int items) {
  if (items <= 2 * ROWS_CUS) {
    const int g = x % groups, first = x - g;                             // of this (head chunk, split): one direction for all of its groups
    return {((first / ROWS_CUS) & 1) ? g : groups - 1 - g, x / groups % gys, x / groups / gys};
  }
  if (x >= ROWS_CUS && x < 2 * ROWS_CUS) x = 3 * ROWS_CUS - 1 - x;
  const int yzs = items / groups, yz = x % yzs, r = x / yzs;
  int g = groups - 1 - r;
  if ((items & 15) == 0) {
    const int q = (groups + 63) >> 6, b = min(min((((int)threadIdx.x & 63) + 1) * q, groups) * nbw, n_blk) - 1;
    const int first = a.row_slot[a.blk_tab[0]], at = a.row_slot[a.blk_tab[2 * b]] - first, len = __builtin_amdgcn_readlane(at, 63) / a.rows_per_blk + 1;      // len: runs of the last sequence
    if (len * a.rows_per_blk >= 64 && len < n_blk && len % nbw == 0 && __ballot(at != a.rows_per_blk * (b % len)) == 0) {
      const int seqs = n_blk / len, per = len / nbw;                     // (the last run is where it lies in all of them: n_blk = seqs len)
      g = r % seqs * per + per - 1 - r / seqs;
    }
  }
  return {g, yz % gys, yz / gys};
}

// the workgroup's runs: first row, rows, cache sequence, first position
__device__ __forceinline__ void rows_table(const AttnTArgs& a, int b0, int nb, int nbw, int tid, int (*tab)[4]) {
  if (tid < nbw) {
    const bool in = tid < nb;
    const int r = in ? a.blk_tab[2 * (b0 + tid)] : 0;
    tab[tid][0] = r;
    tab[tid][1] = in ? min(a.blk_tab[2 * (b0 + tid) + 1], a.rows_per_blk) : 0;
    tab[tid][2] = in ? a.row_seq[r] : -1;
    tab[tid][3] = in ? a.row_slot[r] : 0;
  }
  __syncthreads();
}

// Is the group of one cache sequence?  (rows_table has run)
__device__ __forceinline__ bool rows_one_sequence(const int (*tab)[4], int nb) {
  bool one = true;
  for (int i = 1; i < nb; ++i) one &= tab[i][2] == tab[0][2];
  return one;
}

// The tasks (run, head chunk, split) of workgroup t of n: the runs of groups (nbw runs each) of several sequences
template <typename F>
__device__ __forceinline__ void rows_alone(const AttnTArgs& a, int n_blk, int gys, int nbw, int t, int n, F f) {
  const int tasks = n_blk * gys * a.nsplit, lane = threadIdx.x & 63;
  for (int base = t; base < tasks; base += 64 * n) {                      // 64 tasks are looked at together
    const int mine = min(base + n * lane, tasks - 1), b = mine % n_blk, first = b / nbw * nbw, last = min(first + nbw, n_blk) - 1;
    int seq[4], differ = 0;
    for (int i0 = 0; i0 < nbw; i0 += 4) {
#pragma unroll
      for (int i = 0; i < 4; ++i) seq[i] = a.blk_tab[2 * min(first + i0 + i, last)];
#pragma unroll
      for (int i = 0; i < 4; ++i) seq[i] = a.row_seq[seq[i]];
      differ |= (seq[0] ^ seq[1]) | (seq[0] ^ seq[2]) | (seq[0] ^ seq[3]);
      if (i0 > 0) differ |= seq[0] ^ a.row_seq[a.blk_tab[2 * first]];
    }
    for (uint64_t left = __ballot(differ && base + n * lane < tasks); left; left &= left - 1) {      // (the same in every wave)
      const int task = base + n * (__ffsll((unsigned long long)left) - 1), yz = task / n_blk;
      f(task - yz * n_blk, yz % gys, yz / gys);
    }
  }
}

// An infinite or NaN value at a key that a query does not see would meet its weight 0 there and turn into NaN (the rows of a workgroup share the walk).  So
// such values stay out of the tiles, one product by zero a value says whether there are any, and a workgroup that met some looks its keys
// over again behind the walk: every query then takes them as they are from the keys it sees.  (It costs 0 .. 2.5 % of either kernel: 16 heads of 256 375 -> 384 us,
// of 128 as before; keys of 576 744 -> 761.)
template <int NF, int NB>
__device__ __forceinline__ void finite_only(f32x4 (&v)[NF][NB], int& met) {
  float z[2] = {0.f, 0.f};
#pragma unroll
  for (int f = 0; f < NF; ++f)
#pragma unroll
    for (int x = 0; x < NB; ++x)
#pragma unroll
      for (int e = 0; e < 4; ++e) z[e & 1] = fmaf(v[f][x][e], 0.f, z[e & 1]);
  if (__ballot(z[0] + z[1] != 0.f) == 0) return;
  met = 1;
#pragma unroll
  for (int f = 0; f < NF; ++f)
#pragma unroll
    for (int x = 0; x < NB; ++x)
#pragma unroll
      for (int e = 0; e < 4; ++e) v[f][x][e] = fabsf(v[f][x][e]) < INFINITY ? v[f][x][e] : 0.f;
}

// values d .. d + 3 of one query vector's result
__device__ __forceinline__ void emit4(const AttnTArgs& a, f32x4 v, int row, int64_t col0, int d, bool vec) {
#pragma unroll
  for (int e = 0; e < 4; ++e)
    if (d + e < a.vdim) v[e] = gated(a, v[e], row, col0 + d + e);
  if (vec) {
    if (a.out) *reinterpret_cast<f32x4*>(a.out + (int64_t)row * a.ldo + col0 + d) = v;
    if (a.out16) *reinterpret_cast<uint2*>(a.out16 + (int64_t)row * a.ldo16 + col0 + d) = uint2{cvt_pk_bf16(v[0], v[1]), cvt_pk_bf16(v[2], v[3])};
    return;
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    if (d + e >= a.vdim) continue;
    if (a.out) a.out[(int64_t)row * a.ldo + col0 + d + e] = v[e];
    if (a.out16) a.out16[(int64_t)row * a.ldo16 + col0 + d + e] = f32_to_bf16(v[e]);
  }
}
// values d .. d + 3 of vector qv's sums in a split's partial slab, 16 bytes at a time (value by value a launch of 5 prompts in three splits spent 18 of its 67 us on them and their merge)
__device__ __forceinline__ void part4(const AttnTArgs& a, float* part, int qv, int d, f32x4 v) {
  float* p = part + 2 * a.sq + (int64_t)qv * a.vdim + d;
  if (d + 4 <= a.vdim) {
    *reinterpret_cast<f32x4u*>(p) = v;
    return;
  }
#pragma unroll
  for (int e = 0; e < 4; ++e)
    if (d + e < a.vdim) p[e] = v[e];
}
__device__ __forceinline__ bool emit_vec(const AttnTArgs& a) {
  return (a.vdim & 3) == 0 && (!a.out || ((a.ldo & 3) == 0 && ((uintptr_t)a.out & 15) == 0)) &&
         (!a.out16 || ((a.ldo16 & 3) == 0 && ((uintptr_t)a.out16 & 7) == 0));
}

// The sum of what is not finite among column d of the values that a query sees (keys j0 .. j1 - 1; 0: all are finite), and its way out
__device__ __forceinline__ float seen_odd_sum(const AttnTArgs& a, const float* vb, const float* pvb, int d, int nbL, int j0, int j1, int my_nb, int lo, int hi) {
  float odd = 0.f;
#pragma unroll 1
  for (int j = j0; j < j1; ++j) {
    const float v = (j < nbL ? pvb + (int64_t)j * a.G * a.vdim : vb + (int64_t)(j - nbL) * a.ldv)[d];
    const bool see = ((j < nbL) & (j < my_nb)) | ((j >= lo) & (j <= hi));
    odd += see && !(fabsf(v) < INFINITY) ? v : 0.f;
  }
  return odd;
}
__device__ __forceinline__ void emit_odd(const AttnTArgs& a, float odd, float* part, int qv, int row, int64_t col0, int d) {
  if (part) { part[2 * a.sq + (int64_t)qv * a.vdim + d] = odd; return; }
  odd = gated(a, odd, row, col0 + d);
  if (a.out) a.out[(int64_t)row * a.ldo + col0 + d] = odd;
  if (a.out16) a.out16[(int64_t)row * a.ldo16 + col0 + d] = f32_to_bf16(odd);
}
// Values inside keys: a key that is not finite has no finite score either, so nothing of a row that sees one (keys lo .. hi of j0 .. j1 - 1) is known.  All lanes.
__device__ __forceinline__ bool seen_not_finite(const AttnTArgs& a, const float* kb, int j0, int j1, int lo, int hi) {
  bool met = false;
#pragma unroll 1
  for (int j = j0; j < j1; ++j) {
    bool odd = false;
#pragma unroll 1
    for (int d = threadIdx.x & 63; d < a.dim; d += 64) odd |= !(fabsf(kb[(int64_t)j * a.ldk + d]) < INFINITY);
    if (__ballot(odd)) met |= j >= lo && j <= hi;
  }
  return met;
}

// One run by itself (at most 16 query vectors): every wave takes a quarter of a key's dims for the scores and a quarter of the value columns, the partial score
// tiles meet in LDS as in the walk of decode rows (mfma_f32_tiles.h).  Runs of several sequences gain nothing from a workgroup of 64 vectors, whose walks
// would follow each other, nor do launches of so few runs that the chip is idle (8 heads of 128 over two key heads, us, in groups / by runs: 8 sequences of 2 rows behind
// 500 keys 62 / 12, 32 of 4 behind 1000 68 / 26, one of 16 behind 500 28 / 14, one of 256 28 / 16).
// VK: the values are the first columns of the keys.  lds: KT (LDK + LDV, VK: LDK) + 64 (KT + 4) floats, KT = 16 KF.
template <int NBD, int NBV, int KF, bool VEC, bool VK>
__device__ __forceinline__ void attn_run(const AttnTArgs& a, int b, int gy, int sp, float* __restrict__ lds, int& met) {
  constexpr int KT = 16 * KF, LDK = 64 * NBD + 4, LDV = VK ? LDK : 64 * NBV + 4, LDS_S = KT + 4;
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, c = lane & 15, g4 = lane >> 4, fj = tid >> 4, fc = tid & 15;
  const int rep = a.H / a.G, chunks = (rep + a.hpc - 1) / a.hpc;
  const int g = gy / chunks, h0 = g * rep + (gy % chunks) * a.hpc;
  const int Rc = min(a.hpc, g * rep + rep - h0);
  const int r0 = a.blk_tab[2 * b], nr = min(a.blk_tab[2 * b + 1], a.rows_per_blk);
  if (nr < 1) return;
  const int seq = a.row_seq[r0], pos0 = a.row_slot[r0], posL = pos0 + nr - 1;
  const bool valid = c < nr * Rc;
  const int rin = valid ? c / Rc : 0, hc = valid ? c % Rc : 0, row = r0 + rin, pos = pos0 + rin;
  f32x4 q[NBD];
  {
    const float* src = a.q + (int64_t)row * a.ldq + (int64_t)(h0 + hc) * a.dim;
#pragma unroll
    for (int it = 0; it < NBD; ++it) q[it] = load4<VEC>(src, wave * 16 * NBD + 16 * it + 4 * g4, a.dim, valid);
  }
  const int tF = first_key(a, pos0), nbL = win_nb(posL, a.window, a.pool), nk = nbL + (posL - tF + 1);
  const int ntile = (nk + KT - 1) / KT, tps = (ntile + a.nsplit - 1) / a.nsplit;
  const int t0 = sp * tps, t1 = min(ntile, t0 + tps);
  const int my_nb = valid ? win_nb(pos, a.window, a.pool) : 0, lo = valid ? nbL + first_key(a, pos) - tF : 0x7fffffff, hi = valid ? nbL + pos - tF : -1;
  int lo_all = valid ? lo : -1, hi_all = valid ? hi : 0x7fffffff;
#pragma unroll
  for (int o = 1; o < 16; o <<= 1) { lo_all = max(lo_all, __shfl_xor(lo_all, o)); hi_all = min(hi_all, __shfl_xor(hi_all, o)); }
  lo_all = __builtin_amdgcn_readfirstlane(lo_all); hi_all = __builtin_amdgcn_readfirstlane(hi_all);
  const int Gd = a.G * a.dim, Gv = a.G * a.vdim;
  const float* kb = a.k + ((int64_t)seq * a.t_max + tF) * a.ldk + (int64_t)g * a.dim;
  const float* vb = a.v + ((int64_t)seq * a.t_max + tF) * a.ldv + (int64_t)g * a.vdim;
  const float* pkb = a.pk ? a.pk + (int64_t)seq * a.n_pool_max * Gd + (int64_t)g * a.dim : nullptr;
  const float* pvb = a.pv ? a.pv + (int64_t)seq * a.n_pool_max * Gv + (int64_t)g * a.vdim : nullptr;
  float* K = lds;
  float* V = VK ? lds : lds + KT * LDK;
  float* Sp = lds + KT * LDK + (VK ? 0 : KT * LDV);      // [4 waves][16 q][LDS_S] partial scores
  f32x4 vk[KF][NBD], vv[VK ? 1 : KF][VK ? 1 : NBV];
  auto fetch = [&](int tile) {
#pragma unroll
    for (int f = 0; f < KF; ++f) {
      const int jj = min(tile * KT + 16 * f + fj, nk - 1);
      rows_fetch<NBD, VEC>(vk[f], !VK && jj < nbL ? pkb + (int64_t)jj * Gd : kb + (int64_t)(jj - nbL) * a.ldk, a.dim, fc);
      if constexpr (!VK) rows_fetch<NBV, VEC>(vv[f], jj < nbL ? pvb + (int64_t)jj * Gv : vb + (int64_t)(jj - nbL) * a.ldv, a.vdim, fc);
    }
  };
  float mrun = -INFINITY, lrun = 0.f;
  f32x4 acc[NBV];
#pragma unroll
  for (int x = 0; x < NBV; ++x) acc[x] = f32x4{0.f, 0.f, 0.f, 0.f};
  if (t0 < t1) fetch(t0);
  for (int tile = t0; tile < t1; ++tile) {
    const int key0 = tile * KT;
    if constexpr (VK) finite_only(vk, met);
    else finite_only(vv, met);
    lds_barrier();                                       // the previous tile's values and partial scores are read
#pragma unroll
    for (int f = 0; f < KF; ++f) {
      const bool ok = key0 + 16 * f + fj < nk;
      rows_put<NBD, LDK, VEC>(K + 16 * f * LDK, vk[f], a.dim, fj, fc, ok);
      if constexpr (!VK) rows_put<NBV, LDV, VEC>(V + 16 * f * LDV, vv[f], a.vdim, fj, fc, ok);
    }
    if (tile + 1 < t1) fetch(tile + 1);                  // in flight while this tile is multiplied
    lds_barrier();
    {
      f32x4 s[KF][2];
#pragma unroll
      for (int f = 0; f < KF; ++f) s[f][0] = s[f][1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int it = 0; it < NBD; ++it) {
        f32x4 kf[KF];
#pragma unroll
        for (int f = 0; f < KF; ++f) kf[f] = *reinterpret_cast<const f32x4*>(K + (16 * f + c) * LDK + wave * 16 * NBD + 16 * it + 4 * g4);
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
    const bool whole = key0 >= nbL && key0 >= lo_all && key0 + KT - 1 <= hi_all;
    float mx = -INFINITY;
#pragma unroll
    for (int f = 0; f < KF; ++f) {
      const float* o = Sp + c * LDS_S + 16 * f + 4 * g4;
      p[f] = (*reinterpret_cast<const f32x4*>(o) + *reinterpret_cast<const f32x4*>(o + 16 * LDS_S)) +
             (*reinterpret_cast<const f32x4*>(o + 32 * LDS_S) + *reinterpret_cast<const f32x4*>(o + 48 * LDS_S));
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        p[f][i] = soft_cap(p[f][i], a.cap);
        if (!whole) {
          const int j = key0 + 16 * f + 4 * g4 + i;
          const bool see = ((j < nbL) & (j < my_nb)) | ((j >= lo) & (j <= hi));
          p[f][i] = see ? p[f][i] : -INFINITY;
        }
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
    if (__ballot(mnew != mrun)) {
#pragma unroll
      for (int x = 0; x < NBV; ++x) acc[x] *= corr;
    }
    mrun = mnew;
#pragma unroll
    for (int f = 0; f < KF; ++f)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float v[NBV];
#pragma unroll
        for (int x = 0; x < NBV; ++x) v[x] = V[(16 * f + 4 * g4 + i) * LDV + 16 * (wave + 4 * x) + c];
#pragma unroll
        for (int x = 0; x < NBV; ++x) acc[x] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[x], p[f][i], acc[x], 0, 0, 0);
      }
  }
  lrun += __shfl_xor(lrun, 16);
  lrun += __shfl_xor(lrun, 32);
  if (VK && met) lrun = seen_not_finite(a, kb, t0 * KT, min(nk, t1 * KT), lo, hi) ? NAN : lrun;
  if (!valid) return;
  float* part = a.nsplit > 1 ? a.part + (((int64_t)b * (a.G * chunks) + gy) * a.nsplit + sp) * ((int64_t)a.sq * (2 + a.vdim)) : nullptr;
  const int64_t col0 = (int64_t)(h0 + hc) * a.vdim;
  const float inv = part ? 1.f : a.out_scale * softmax_inv(mrun, lrun, a.sink, h0 + hc);
  const bool vec = emit_vec(a);
#pragma unroll
  for (int x = 0; x < NBV; ++x) {
    const int d = 16 * (wave + 4 * x) + 4 * g4;
    if (d >= a.vdim) continue;
    const f32x4 r = acc[x] * inv;
    if (!part) { emit4(a, r, row, col0, d, vec); continue; }
    part4(a, part, c, d, r);
  }
  if (part && wave == 0 && g4 == 0) { part[c] = mrun; part[a.sq + c] = lrun; }
  if (!VK && met) {
#pragma unroll 1
    for (int x = 0; x < 4 * NBV; ++x) {                  // this lane's columns again
      const int d = 16 * (wave + 4 * (x >> 2)) + 4 * g4 + (x & 3);
      if (d < a.vdim) {
        const float odd = seen_odd_sum(a, vb, pvb, d, nbL, t0 * KT, min(nk, t1 * KT), my_nb, lo, hi);
        if (odd != 0.f) emit_odd(a, odd * inv, part, c, row, col0, d);
      }
    }
  }
}

// A workgroup a run, head chunk and split
template <int NBD, int NBV, int KF, bool VEC, bool VK>
__global__ __launch_bounds__(256) void attn_runs_kernel(AttnTArgs a) {
  constexpr int KT = 16 * KF;
  __shared__ __attribute__((aligned(16))) float lds[KT * (64 * NBD + 4) + (VK ? 0 : KT * (64 * NBV + 4)) + 64 * (KT + 4)];
  __shared__ int met;
  if (threadIdx.x == 0) met = 0;
  __syncthreads();
  attn_run<NBD, NBV, KF, VEC, VK>(a, blockIdx.x, blockIdx.y, blockIdx.z, lds, met);
}

// Keys and values in arenas of their own, heads of up to 256 values: each wave owns 16 of the 64 vectors with all their dims, queries in registers.
// K is read 16 bytes at a time (a lane's k slot = dims 16 it + 4 g .. + 3 over four steps, one accumulator per step: four short chains sum more
// exactly than one long one), V likewise (row c of value fragment 4 vb + e = column 64 vb + 4 c + e); with row strides of 4 mod 64 floats
// both reads touch every bank once.  One LDS-only barrier per tile.
// 2048 tokens, 16 heads of 128 over 4 key/value heads (17.2 GF): 632 us in the form before, 198 us here (87 TFLOP/s).
// VEC: dim and vdim are multiples of 4.
template <int NBD, int NBV, bool VEC>
__global__ __launch_bounds__(256, 2) void attn_rows_kernel(AttnTArgs a, int n_blk, int hv, int groups) {
  constexpr int KT = NBD + NBV > 4 ? 16 : 32, KF = KT / 16, LDK = 64 * NBD + 4, LDV = 64 * NBV + 4, TILE = KT * (LDK + LDV);
  __shared__ __attribute__((aligned(16))) float lds[2 * TILE];        // [2][K tile | V tile]
  __shared__ int tab[16][4], met;                      // met: an infinite or NaN value
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, c = lane & 15, g4 = lane >> 4;
  if (tid == 0) met = 0;
  const int rep = a.H / a.G, chunks = (rep + a.hpc - 1) / a.hpc, gys = a.G * chunks;
  const int rw = 16 / hv, nbw = rw * 4 / a.rows_per_blk;                // rows per wave; runs per workgroup
  const int in_groups = groups * gys * a.nsplit;
  if ((int)blockIdx.x >= in_groups) {
    __syncthreads();                                                    // met
    rows_alone(a, n_blk, gys, nbw, blockIdx.x - in_groups, gridDim.x - in_groups,
               [&](int b, int gy, int sp) { attn_run<NBD, NBV, KF, VEC, false>(a, b, gy, sp, lds, met); });
    return;
  }
  const RowsItem it = rows_item(a, blockIdx.x, groups, nbw, n_blk, gys, in_groups);
  const int gy = it.gy, sp = it.sp;
  const int g = gy / chunks, h0 = g * rep + (gy % chunks) * a.hpc;
  const int Rc = min(a.hpc, g * rep + rep - h0);
  const int b0 = it.group * nbw, nb = min(nbw, n_blk - b0);
  rows_table(a, b0, nb, nbw, tid, tab);
  if (!rows_one_sequence(tab, nb)) return;
  // this lane's query: column c of the wave's 16
  const int slot = wave * rw + c / hv, hc = c % hv, run = slot / a.rows_per_blk, rin = slot % a.rows_per_blk;
  const bool valid = rin < tab[run][1] && hc < Rc;
  const int row = valid ? tab[run][0] + rin : 0, pos = tab[run][3] + rin;
  f32x4 q[4 * NBD];
  {
    const float* src = a.q + (int64_t)row * a.ldq + (int64_t)(h0 + (valid ? hc : 0)) * a.dim;
#pragma unroll
    for (int it = 0; it < 4 * NBD; ++it) q[it] = load4<VEC>(src, 16 * it + 4 * g4, a.dim, valid);
  }
  const int Gd = a.G * a.dim, Gv = a.G * a.vdim;
  // ---- the keys that the group's runs see between them ----
  const int seq = tab[0][2];
  int tF = 0x7fffffff, posL = -1;
  for (int i = 0; i < nb; ++i) {
    tF = min(tF, first_key(a, tab[i][3]));
    posL = max(posL, tab[i][3] + tab[i][1] - 1);
  }
  const int nbL = win_nb(posL, a.window, a.pool), nk = nbL + (posL - tF + 1);
  const int ntile = (nk + KT - 1) / KT, tps = (ntile + a.nsplit - 1) / a.nsplit;
  const int t0 = sp * tps, t1 = min(ntile, t0 + tps);
  // what this lane's query sees: token keys [lo, hi] (as key indices of the walk) and the first my_nb block means
  const int my_nb = valid ? win_nb(pos, a.window, a.pool) : 0;
  const int lo = valid ? nbL + first_key(a, pos) - tF : 0x7fffffff, hi = valid ? nbL + pos - tF : -1;
  int w_lo = lo, w_hi = hi, w_nb = my_nb, w_lo_all = valid ? lo : -1, w_hi_all = valid ? hi : 0x7fffffff;      // over the wave's queries
#pragma unroll
  for (int o = 1; o < 16; o <<= 1) {
    w_lo = min(w_lo, __shfl_xor(w_lo, o)); w_hi = max(w_hi, __shfl_xor(w_hi, o)); w_nb = max(w_nb, __shfl_xor(w_nb, o));
    w_lo_all = max(w_lo_all, __shfl_xor(w_lo_all, o)); w_hi_all = min(w_hi_all, __shfl_xor(w_hi_all, o));
  }
  w_lo = __builtin_amdgcn_readfirstlane(w_lo); w_hi = __builtin_amdgcn_readfirstlane(w_hi); w_nb = __builtin_amdgcn_readfirstlane(w_nb);
  w_lo_all = __builtin_amdgcn_readfirstlane(w_lo_all); w_hi_all = __builtin_amdgcn_readfirstlane(w_hi_all);
  const float* kb = a.k + ((int64_t)seq * a.t_max + tF) * a.ldk + (int64_t)g * a.dim;
  const float* vb_ = a.v + ((int64_t)seq * a.t_max + tF) * a.ldv + (int64_t)g * a.vdim;
  const float* pkb = a.pk ? a.pk + (int64_t)seq * a.n_pool_max * Gd + (int64_t)g * a.dim : nullptr;
  const float* pvb = a.pv ? a.pv + (int64_t)seq * a.n_pool_max * Gv + (int64_t)g * a.vdim : nullptr;
  f32x4 vk[KF][NBD], vv[KF][NBV];
  const int fj = tid >> 4, fc = tid & 15;
  auto fetch = [&](int tile) {
#pragma unroll
    for (int f = 0; f < KF; ++f) {
      const int jj = min(tile * KT + 16 * f + fj, nk - 1);
      rows_fetch<NBD, VEC>(vk[f], jj < nbL ? pkb + (int64_t)jj * Gd : kb + (int64_t)(jj - nbL) * a.ldk, a.dim, fc);
      rows_fetch<NBV, VEC>(vv[f], jj < nbL ? pvb + (int64_t)jj * Gv : vb_ + (int64_t)(jj - nbL) * a.ldv, a.vdim, fc);
    }
  };
  auto put = [&](int tile, int buf) {
    float* K = lds + buf * TILE;
    finite_only(vv, met);
#pragma unroll
    for (int f = 0; f < KF; ++f) {
      const bool ok = tile * KT + 16 * f + fj < nk;
      rows_put<NBD, LDK, VEC>(K + 16 * f * LDK, vk[f], a.dim, fj, fc, ok);
      rows_put<NBV, LDV, VEC>(K + KT * LDK + 16 * f * LDV, vv[f], a.vdim, fj, fc, ok);
    }
  };
  float mrun = -INFINITY, lrun = 0.f;                // lrun: this lane's keys only
  f32x4 acc[4 * NBV];
#pragma unroll
  for (int x = 0; x < 4 * NBV; ++x) acc[x] = f32x4{0.f, 0.f, 0.f, 0.f};
  if (t0 < t1) { fetch(t0); put(t0, 0); }
  if (t0 + 1 < t1) fetch(t0 + 1);
  lds_barrier();
  for (int tile = t0; tile < t1; ++tile) {
    const int key0 = tile * KT, cur = (tile - t0) & 1;
    const float* K = lds + cur * TILE;
    const float* V = K + KT * LDK;
    if ((key0 <= w_hi && key0 + KT - 1 >= w_lo) || key0 < w_nb) {      // wave-uniform
      f32x4 s[KF], se[KF][4];
#pragma unroll
      for (int f = 0; f < KF; ++f)
#pragma unroll
        for (int e = 0; e < 4; ++e) se[f][e] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int it = 0; it < 4 * NBD; ++it) {
        f32x4 kf[KF];
#pragma unroll
        for (int f = 0; f < KF; ++f) kf[f] = *reinterpret_cast<const f32x4*>(K + (16 * f + c) * LDK + 16 * it + 4 * g4);
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int f = 0; f < KF; ++f) se[f][e] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[f][e], q[it][e], se[f][e], 0, 0, 0);
      }
#pragma unroll
      for (int f = 0; f < KF; ++f) s[f] = (se[f][0] + se[f][1]) + (se[f][2] + se[f][3]);
      if (a.cap > 0.f) {
#pragma unroll
        for (int f = 0; f < KF; ++f)
#pragma unroll
          for (int i = 0; i < 4; ++i) s[f][i] = soft_cap(s[f][i], a.cap);
      }
      if (!(key0 >= nbL && key0 >= w_lo_all && key0 + KT - 1 <= w_hi_all)) {
#pragma unroll
        for (int f = 0; f < KF; ++f)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int j = key0 + 16 * f + 4 * g4 + i;
            const bool see = ((j < nbL) & (j < my_nb)) | ((j >= lo) & (j <= hi));      // (lo >= nbL)
            s[f][i] = see ? s[f][i] : -INFINITY;
          }
      }
      float mx = fmaxf(fmaxf(s[0][0], s[0][1]), fmaxf(s[0][2], s[0][3]));
#pragma unroll
      for (int f = 1; f < KF; ++f) mx = fmaxf(mx, fmaxf(fmaxf(s[f][0], s[f][1]), fmaxf(s[f][2], s[f][3])));
      mx = fmaxf(mx, __shfl_xor(mx, 16));
      mx = fmaxf(mx, __shfl_xor(mx, 32));
      const float mnew = fmaxf(mrun, mx);
      const float corr = mrun == -INFINITY ? 0.f : fast_exp(mrun - mnew);
      float sum = 0.f;
#pragma unroll
      for (int f = 0; f < KF; ++f)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          s[f][i] = s[f][i] == -INFINITY ? 0.f : fast_exp(s[f][i] - mnew);
          sum += s[f][i];
        }
      lrun = lrun * corr + sum;
      if (__ballot(mnew != mrun)) {                  // some query's maximum moved
#pragma unroll
        for (int x = 0; x < 4 * NBV; ++x) acc[x] *= corr;
      }
      mrun = mnew;
#pragma unroll
      for (int f = 0; f < KF; ++f)
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int vb = 0; vb < NBV; ++vb) {
            const f32x4 v4 = *reinterpret_cast<const f32x4*>(V + (16 * f + 4 * g4 + i) * LDV + 64 * vb + 4 * c);
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[4 * vb + e] = __builtin_amdgcn_mfma_f32_16x16x4f32(v4[e], s[f][i], acc[4 * vb + e], 0, 0, 0);
          }
    }
    if (tile + 1 < t1) put(tile + 1, cur ^ 1);       // the other tile was last read before the previous barrier
    if (tile + 2 < t1) fetch(tile + 2);
    lds_barrier();
  }
  lrun += __shfl_xor(lrun, 16);
  lrun += __shfl_xor(lrun, 32);
  if (valid) {
    const int qv = rin * Rc + hc;                    // the vector's place in its run's partial slab
    float* part = a.nsplit > 1 ? a.part + (((int64_t)(b0 + run) * gys + gy) * a.nsplit + sp) * ((int64_t)a.sq * (2 + a.vdim)) : nullptr;
    const int64_t col0 = (int64_t)(h0 + hc) * a.vdim;
    const float inv = part ? 1.f : a.out_scale * softmax_inv(mrun, lrun, a.sink, h0 + hc);
    const bool vec = emit_vec(a);
#pragma unroll
    for (int vb = 0; vb < NBV; ++vb)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int d = 64 * vb + 4 * (4 * g4 + i);
        if (d >= a.vdim) continue;
        const f32x4 r = f32x4{acc[4 * vb][i], acc[4 * vb + 1][i], acc[4 * vb + 2][i], acc[4 * vb + 3][i]} * inv;
        if (!part) { emit4(a, r, row, col0, d, vec); continue; }
        part4(a, part, qv, d, r);
      }
    if (part && g4 == 0) { part[qv] = mrun; part[a.sq + qv] = lrun; }
    if (met) {
#pragma unroll 1
      for (int x = 0; x < 16 * NBV; ++x) {           // this lane's columns again: what is not finite among the seen keys' values
        const int d = 64 * (x >> 4) + 16 * g4 + (x & 15);
        if (d >= a.vdim) continue;
        const float odd = seen_odd_sum(a, vb_, pvb, d, nbL, t0 * KT, min(nk, t1 * KT), my_nb, lo, hi);
        if (odd != 0.f) emit_odd(a, odd * inv, part, qv, row, col0, d);
      }
    }
  }
}

// Latent attention (one key/value head whose values are the first columns of the keys, up to 640 of them): vectors with all their dims do not
// fit a wave's registers, so every wave takes all of a workgroup's 32 vectors with a quarter of the dims (queries in registers) and, for the
// values, a quarter of the columns.  The four partial score tiles meet in LDS, each wave sums them and takes the same softmax: 144 MFMAs of
// 32 cycles per wave and 16-key tile at 576 + 512 values stand against three barriers, and two or three workgroups share a CU.  (64 vectors
// at 512 registers and one wave per SIMD: 1450 us on the case below, nothing covers the barriers and 129 registers spill.)
// 2048 tokens, 16 heads, keys of 576 and values of 512, window 1024 (54.8 GF): 1674 us in the form before, 761 us here.
template <int NB, bool VEC>
__global__ __launch_bounds__(256, 2) void attn_latent_rows_kernel(AttnTArgs a, int n_blk, int hv, int groups) {
  constexpr int KT = 16, QF = 2, LDK = 64 * NB + 4, LDS_S = 20;
  __shared__ __attribute__((aligned(16))) float K[KT * LDK + 4 * 16 * QF * LDS_S];
  float (*Sp)[16 * QF * LDS_S] = reinterpret_cast<float (*)[16 * QF * LDS_S]>(K + KT * LDK);     // [wave][query][16 keys]: partial scores
  __shared__ int tab[16][4], met;
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, c = lane & 15, g4 = lane >> 4;
  if (tid == 0) met = 0;
  const int rep = a.H / a.G, gys = (rep + a.hpc - 1) / a.hpc;           // (one key/value head)
  const int rf = 16 / hv, nbw = rf * QF / a.rows_per_blk;               // rows per 16-vector fragment; runs per workgroup
  const int in_groups = groups * gys * a.nsplit;
  if ((int)blockIdx.x >= in_groups) {
    __syncthreads();                                                    // met
    rows_alone(a, n_blk, gys, nbw, blockIdx.x - in_groups, gridDim.x - in_groups,
               [&](int b, int gy, int sp) { attn_run<NB, NB, 1, VEC, true>(a, b, gy, sp, K, met); });
    return;
  }
  const RowsItem it = rows_item(a, blockIdx.x, groups, nbw, n_blk, gys, in_groups);
  const int gy = it.gy, sp = it.sp, h0 = gy * a.hpc;
  const int Rc = min(a.hpc, rep - h0);
  const int b0 = it.group * nbw, nb = min(nbw, n_blk - b0);
  rows_table(a, b0, nb, nbw, tid, tab);
  if (!rows_one_sequence(tab, nb)) return;
  const int hc = c % hv, dw = wave * 16 * NB;                           // this wave's dims: dw .. dw + 16 NB - 1
  int row[QF], pos[QF], run[QF];
  f32x4 q[QF][NB];
#pragma unroll
  for (int f = 0; f < QF; ++f) {
    const int slot = f * rf + c / hv, rin = slot % a.rows_per_blk;
    run[f] = slot / a.rows_per_blk;
    const bool valid = rin < tab[run[f]][1] && hc < Rc;
    row[f] = valid ? tab[run[f]][0] + rin : -1;
    pos[f] = tab[run[f]][3] + rin;
    const float* src = a.q + (int64_t)max(row[f], 0) * a.ldq + (int64_t)(h0 + (valid ? hc : 0)) * a.dim;
#pragma unroll
    for (int it = 0; it < NB; ++it) q[f][it] = load4<VEC>(src, dw + 16 * it + 4 * g4, a.dim, valid);
  }
  const int seq = tab[0][2];
  int tF = 0x7fffffff, posL = -1;
  for (int i = 0; i < nb; ++i) {
    tF = min(tF, first_key(a, tab[i][3]));
    posL = max(posL, tab[i][3] + tab[i][1] - 1);
  }
  const int nk = posL - tF + 1;
  const int ntile = (nk + KT - 1) / KT, tps = (ntile + a.nsplit - 1) / a.nsplit;
  const int t0 = sp * tps, t1 = min(ntile, t0 + tps);
  int lo[QF], hi[QF], lo_all = -1, hi_all = 0x7fffffff;
#pragma unroll
  for (int f = 0; f < QF; ++f) {
    const bool mine = row[f] >= 0;
    lo[f] = mine ? first_key(a, pos[f]) - tF : 0x7fffffff;
    hi[f] = mine ? pos[f] - tF : -1;
    if (mine) { lo_all = max(lo_all, lo[f]); hi_all = min(hi_all, hi[f]); }
  }
#pragma unroll
  for (int o = 1; o < 16; o <<= 1) { lo_all = max(lo_all, __shfl_xor(lo_all, o)); hi_all = min(hi_all, __shfl_xor(hi_all, o)); }
  lo_all = __builtin_amdgcn_readfirstlane(lo_all); hi_all = __builtin_amdgcn_readfirstlane(hi_all);
  const float* kb = a.k + ((int64_t)seq * a.t_max + tF) * a.ldk;
  f32x4 vk[1][NB];
  const int fj = tid >> 4, fc = tid & 15;
  auto fetch = [&](int tile) { rows_fetch<NB, VEC>(vk[0], kb + (int64_t)min(tile * KT + fj, nk - 1) * a.ldk, a.dim, fc); };
  auto put = [&](int tile) { rows_put<NB, LDK, VEC>(K, vk[0], a.dim, fj, fc, tile * KT + fj < nk); };
  float mrun[QF], lrun[QF];
  f32x4 acc[QF][NB];
#pragma unroll
  for (int f = 0; f < QF; ++f) {
    mrun[f] = -INFINITY;
    lrun[f] = 0.f;
#pragma unroll
    for (int x = 0; x < NB; ++x) acc[f][x] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  if (t0 < t1) fetch(t0);
  for (int tile = t0; tile < t1; ++tile) {
    const int key0 = tile * KT;
    finite_only(vk, met);
    lds_barrier();                                   // the previous tile's values and partial scores are read
    put(tile);
    if (tile + 1 < t1) fetch(tile + 1);              // in flight while this tile is multiplied
    lds_barrier();
    {                                                // partial scores over this wave's dims, two chains each
      f32x4 s[QF][2];
#pragma unroll
      for (int f = 0; f < QF; ++f) s[f][0] = s[f][1] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int it = 0; it < NB; ++it) {
        const f32x4 kf = *reinterpret_cast<const f32x4*>(K + c * LDK + dw + 16 * it + 4 * g4);
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int f = 0; f < QF; ++f) s[f][e & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[e], q[f][it][e], s[f][e & 1], 0, 0, 0);
      }
#pragma unroll
      for (int f = 0; f < QF; ++f) *reinterpret_cast<f32x4*>(&Sp[wave][(16 * f + c) * LDS_S + 4 * g4]) = s[f][0] + s[f][1];
    }
    lds_barrier();
    const bool whole = key0 >= lo_all && key0 + KT - 1 <= hi_all;
    f32x4 p[QF];
#pragma unroll
    for (int f = 0; f < QF; ++f) {
      const int o = (16 * f + c) * LDS_S + 4 * g4;
      f32x4 s = (*reinterpret_cast<const f32x4*>(&Sp[0][o]) + *reinterpret_cast<const f32x4*>(&Sp[1][o])) +
                (*reinterpret_cast<const f32x4*>(&Sp[2][o]) + *reinterpret_cast<const f32x4*>(&Sp[3][o]));
      if (a.cap > 0.f) {
#pragma unroll
        for (int i = 0; i < 4; ++i) s[i] = soft_cap(s[i], a.cap);
      }
      if (!whole) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int j = key0 + 4 * g4 + i;
          s[i] = ((j < lo[f]) | (j > hi[f])) ? -INFINITY : s[i];
        }
      }
      float mx = fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3]));
      mx = fmaxf(mx, __shfl_xor(mx, 16));
      mx = fmaxf(mx, __shfl_xor(mx, 32));
      const float mnew = fmaxf(mrun[f], mx);
      const float corr = mrun[f] == -INFINITY ? 0.f : fast_exp(mrun[f] - mnew);
      float sum = 0.f;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        p[f][i] = s[i] == -INFINITY ? 0.f : fast_exp(s[i] - mnew);
        sum += p[f][i];
      }
      lrun[f] = lrun[f] * corr + sum;
      if (__ballot(mnew != mrun[f])) {
#pragma unroll
        for (int x = 0; x < NB; ++x) acc[f][x] *= corr;
      }
      mrun[f] = mnew;
    }
    // value fragment x of this wave: columns 16 (wave + 4 x) + c
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float v[NB];
#pragma unroll
      for (int x = 0; x < NB; ++x) v[x] = K[(4 * g4 + i) * LDK + 16 * (wave + 4 * x) + c];
#pragma unroll
      for (int x = 0; x < NB; ++x)
#pragma unroll
        for (int f = 0; f < QF; ++f) acc[f][x] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[x], p[f][i], acc[f][x], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);             // (all four steps' reads at once would not fit the registers)
    }
  }
  if (met) {
#pragma unroll
    for (int f = 0; f < QF; ++f) lrun[f] = seen_not_finite(a, kb, t0 * KT, min(nk, t1 * KT), lo[f], hi[f]) ? NAN : lrun[f];
  }
  const bool vec = emit_vec(a);
#pragma unroll
  for (int f = 0; f < QF; ++f) {
    lrun[f] += __shfl_xor(lrun[f], 16);
    lrun[f] += __shfl_xor(lrun[f], 32);
    if (row[f] < 0) continue;
    const int qv = (row[f] - tab[run[f]][0]) * Rc + hc;
    float* part = a.nsplit > 1 ? a.part + (((int64_t)(b0 + run[f]) * gys + gy) * a.nsplit + sp) * ((int64_t)a.sq * (2 + a.vdim)) : nullptr;
    const int64_t col0 = (int64_t)(h0 + hc) * a.vdim;
    const float inv = part ? 1.f : a.out_scale * softmax_inv(mrun[f], lrun[f], a.sink, h0 + hc);
#pragma unroll
    for (int x = 0; x < NB; ++x) {
      const int d = 16 * (wave + 4 * x) + 4 * g4;
      if (d >= a.vdim) continue;
      const f32x4 r = acc[f][x] * inv;
      if (!part) { emit4(a, r, row[f], col0, d, vec); continue; }
      part4(a, part, qv, d, r);
    }
    if (part && wave == 0 && g4 == 0) { part[qv] = mrun[f]; part[a.sq + qv] = lrun[f]; }
  }
}

// Decode rows whose values lie inside the keys: workgroup b takes row b and up to 16 of its query heads (the walk: mfma_f32_tiles.h).
struct SoftCap { float cap; __device__ __forceinline__ float operator()(float s) const { return soft_cap(s, cap); } };
template <int NB, int KF, bool VEC>
__global__ __launch_bounds__(256) void attn_latent_decode_kernel(AttnTArgs a) {
  using Walk = LatentWalk<NB, KF, VEC, SoftCap>;
  constexpr int KT = Walk::KT;
  __shared__ __attribute__((aligned(16))) float lds[Walk::LDS_FLOATS];
  const int tid = threadIdx.x, b = blockIdx.x, gy = blockIdx.y, sp = blockIdx.z;
  const int rep = a.H / a.G, chunks = (rep + a.hpc - 1) / a.hpc;
  const int g = gy / chunks, h0 = g * rep + (gy % chunks) * a.hpc;
  const int Rc = min(a.hpc, g * rep + rep - h0);
  const int seq = a.row_seq[b], pos = a.row_slot[b], tF = first_key(a, pos);
  const int nk = pos - tF + 1;
  const int ntile = (nk + KT - 1) / KT, tps = (ntile + a.nsplit - 1) / a.nsplit;
  const int t0 = sp * tps, t1 = min(ntile, t0 + tps);
  const int wave = tid >> 6, lane = tid & 63, c = lane & 15, g4 = lane >> 4;
  const float* src = a.q + (int64_t)b * a.ldq + (int64_t)(h0 + min(c, Rc - 1)) * a.dim;
  f32x4 q[NB], acc[NB];
#pragma unroll
  for (int it = 0; it < NB; ++it) q[it] = load4<VEC>(src, wave * 16 * NB + 16 * it + 4 * g4, a.dim, c < Rc);
  float mrun, lrun;
  Walk::run(lds, a.k + ((int64_t)seq * a.t_max + tF) * a.ldk + (int64_t)g * a.dim, a.ldk, a.dim, nk, nk, t0, t1, q, SoftCap{a.cap}, mrun, lrun, acc);
  if (c >= Rc) return;
  float* part = a.nsplit > 1 ? a.part + (((int64_t)b * gridDim.y + gy) * a.nsplit + sp) * ((int64_t)a.sq * (2 + a.vdim)) : nullptr;
  const bool vec = emit_vec(a);
  const int64_t col0 = (int64_t)(h0 + c) * a.vdim;
  const float inv = part ? 1.f : a.out_scale * softmax_inv(mrun, lrun, a.sink, h0 + c);
#pragma unroll
  for (int x = 0; x < NB; ++x) {
    const int d = 16 * (wave + 4 * x) + 4 * g4;
    if (d >= a.vdim) continue;
    const f32x4 r = acc[x] * inv;
    if (!part) { emit4(a, r, b, col0, d, vec); continue; }
    part4(a, part, c, d, r);
  }
  if (part && wave == 0 && g4 == 0) { part[c] = mrun; part[a.sq + c] = lrun; }
}
