// vit_blocks.cpp — the blocks of a vision transformer as one host call: the launches of Block.forward / CausalBlock.forward (mingtok/vision_tower/
// layers/block.py:80-105, 301-327) for a whole stack, on an fp32 residual stream.  A 256 x 256 image is seven launches of 5 .. 10 us a block, and
// one call per launch from Python costs more than the launch runs: 60 blocks took 5.1 ms of host time over 3.1 ms of kernels.
#include "common.h"

namespace {

size_t up256(size_t n) { return (n + 255) & ~(size_t)255; }

// Slices of a residual product (mn_vit_resid_slices), for any number of rows
int resid_slices(int64_t M, int N, int K) {
  const int64_t tiles = mn_cdiv(M, 256) * mn_cdiv(N, 256);
  if (tiles >= 128 || K < 512 || (K % 64) || (N % 4)) return 0;
  int64_t ks = 256 / tiles;
  ks = ks < 2 ? 2 : (ks > 8 ? 8 : ks);
  while (ks > 2 && K / ks < 256) --ks;
  return (int)ks;
}

struct Plan { size_t a, b, c, p, total; };     // A: qkv, then the hidden units; B: normed rows; C: attention; P: split-K slabs
Plan plan(int64_t M, int dim, int hidden, int gelu, int precise) {
  Plan p;
  const size_t row = precise ? 4 : 2;          // bytes a value: fp32 or a hi / lo pair, bf16
  const size_t qkv = (size_t)M * 3 * dim * row;
  size_t h = (size_t)M * hidden * row;
  if (precise && gelu) h *= 2;                                              // with the product before its activation
  p.a = 0;
  p.b = up256(qkv > h ? qkv : h);
  p.c = p.b + up256((size_t)M * dim * row);
  p.p = p.c + up256((size_t)M * dim * row);
  int ks = 0;
  if (!precise) {
    const int k1 = resid_slices(M, dim, dim), k2 = resid_slices(M, dim, hidden);
    ks = k1 > k2 ? k1 : k2;
  }
  p.total = p.p + up256((size_t)ks * M * dim * 4);
  return p;
}

// the products that take their LayerNorm or residual with them (rows_gemm.hip): few rows, 16-byte weights, 8-byte biases and norm parameters
bool rows_ok(const float* x, const uint16_t* const* w, int depth, int64_t M, int dim, int hidden, int gelu) {
  if (!mn_vit_rows_ok((int)M, dim, hidden, gelu) || ((uintptr_t)x & 15)) return false;
  for (int i = 0; i < 12 * depth; ++i) {
    const int k = i % 12;
    const uintptr_t mask = k == 2 || k == 4 || k == 8 || k == 10 ? 15 : 7;
    if ((uintptr_t)w[i] & mask) return false;
  }
  return true;
}

#define TRY(e) do { const int rc_ = (e); if (rc_ < 0) return rc_; } while (0)

}  // namespace

extern "C" int mn_vit_resid_slices(int M, int N, int K) { return M < 1 || N < 1 || K < 1 ? 0 : resid_slices(M, N, K); }

extern "C" size_t mn_vit_blocks_workspace_bytes(int B, int T, int dim, int hidden, int gelu, int precise) {
  return B < 1 || T < 1 || dim < 1 || hidden < 1 ? 0 : plan((int64_t)B * T, dim, hidden, gelu, precise).total;
}

extern "C" int mn_vit_blocks(float* x, int B, int T, int dim, int depth, const uint16_t* const* w, int hidden, int gelu, int causal, int precise, float eps,
                             const uint16_t* fin_g, const uint16_t* fin_b, int fin_gelu, uint16_t* out, void* ws, size_t ws_bytes, void* stream) {
  MN_CHECK_ARG(x && w && ws && B >= 1 && T >= 1 && dim >= 64 && (dim % 64) == 0 && depth >= 1 && hidden >= 1 && (int64_t)B * T < ((int64_t)1 << 31) &&
                   (precise ? !out : (out && fin_g && fin_b)),
               "mn_vit_blocks: bad args (dim=%d: a multiple of 64)", dim);
  for (int i = 0; i < 12 * depth; ++i) MN_CHECK_ARG(w[i], "mn_vit_blocks: block %d: tensor %d is missing", i / 12, i % 12);
  const int M = B * T, nh = dim / 64;
  const Plan p = plan(M, dim, hidden, gelu, precise);
  MN_CHECK_ARG(ws_bytes >= p.total && ((uintptr_t)ws & 255) == 0, "mn_vit_blocks: workspace of %zu bytes, %zu needed (256-byte aligned)", ws_bytes, p.total);
  char* base = reinterpret_cast<char*>(ws);
  if (precise) {                               // fp32-class: hi / lo pairs (lo rows one block of rows further), products added to the stream in place
    float* wide = reinterpret_cast<float*>(base);
    uint16_t* h = reinterpret_cast<uint16_t*>(base) + (gelu ? (size_t)M * hidden * 2 : 0);
    uint16_t *xs = reinterpret_cast<uint16_t*>(base + p.b), *att = reinterpret_cast<uint16_t*>(base + p.c);
    const int64_t dlo = (int64_t)M * dim, hlo = (int64_t)M * hidden;
    MN_CHECK_ARG((hidden % 64) == 0, "mn_vit_blocks: hidden=%d must be a multiple of 64 (pad with zeros)", hidden);
    for (int i = 0; i < depth; ++i, w += 12) {
      TRY(mn_norm_act_split(x, dim, 2, w[0], w[1], eps, 0, xs, dim, dlo, nullptr, 0, M, dim, stream));
      if (mn_gemm256_supported(dim, dlo, dim, 3 * (int64_t)dim, M, 3 * dim, dim) && ((uintptr_t)w[2] & 15) == 0 && ((uintptr_t)w[3] & 7) == 0) {
        // q, k, v as a bf16 hi and a bf16 lo plane, where attention would split them for every 64 queries
        mn_g256 qkv{};
        qkv.A = xs; qkv.lda = dim; qkv.a_lo_off = dlo; qkv.W = w[2]; qkv.ldw = dim; qkv.bias = w[3]; qkv.C = wide; qkv.ldc = 3 * (int64_t)dim;
        qkv.c_lo_off = 3 * dlo; qkv.M = M; qkv.N = 3 * dim; qkv.K = dim;
        TRY(mn_gemm256_ex(&qkv, MN_G256_BF16_SPLIT, 1, stream));
        TRY(mn_attn_prefill_hd64_planes(reinterpret_cast<const uint16_t*>(wide), 3 * dlo, att, B, T, nh, causal, stream));
      } else {                                 // (refused with the product's reasons)
        TRY(mn_gemm256(xs, dim, dlo, w[2], dim, w[3], wide, 3 * (int64_t)dim, M, 3 * dim, dim, MN_GEMM_F32, stream));
        TRY(mn_attn_prefill_hd64_f32(wide, nullptr, att, B, T, nh, causal, stream));
      }
      TRY(mn_gemm256(att, dim, dlo, w[4], dim, w[5], x, dim, M, dim, dim, MN_GEMM_F32_RESID, stream));
      TRY(mn_norm_act_split(x, dim, 2, w[6], w[7], eps, 0, xs, dim, dlo, nullptr, 0, M, dim, stream));
      if (gelu) {
        TRY(mn_gemm256(xs, dim, dlo, w[8], dim, w[9], wide, hidden, M, hidden, dim, MN_GEMM_F32, stream));
        TRY(mn_norm_act_split(wide, hidden, 0, nullptr, nullptr, eps, 1, h, hidden, hlo, nullptr, 0, M, hidden, stream));
      } else {
        TRY(mn_gemm256_swiglu_split(xs, dim, dlo, w[8], dim, w[9], h, hidden, hlo, M, hidden, dim, stream));
      }
      TRY(mn_gemm256(h, hidden, hlo, w[10], hidden, w[11], x, dim, M, dim, hidden, MN_GEMM_F32_RESID, stream));
    }
    return MN_OK;
  }
  uint16_t *qkv = reinterpret_cast<uint16_t*>(base), *h = qkv, *xn = reinterpret_cast<uint16_t*>(base + p.b), *att = reinterpret_cast<uint16_t*>(base + p.c);
  float* slabs = reinterpret_cast<float*>(base + p.p);
  if (rows_ok(x, w, depth, M, dim, hidden, gelu)) {
    for (int i = 0; i < depth; ++i, w += 12) {
      TRY(mn_ln_gemm_rows(x, dim, w[0], w[1], eps, w[2], dim, w[3], 0, 0, qkv, 3 * (int64_t)dim, M, 3 * dim, dim, stream));
      TRY(mn_attn_prefill_hd64(qkv, att, B, T, nh, causal, stream));
      TRY(mn_resid_gemm_rows(att, dim, w[4], dim, w[5], x, dim, M, dim, dim, stream));
      TRY(mn_ln_gemm_rows(x, dim, w[6], w[7], eps, w[8], dim, w[9], gelu, !gelu, h, hidden, M, hidden, dim, stream));
      TRY(mn_resid_gemm_rows(h, hidden, w[10], hidden, w[11], x, dim, M, dim, hidden, stream));
    }
    return mn_layernorm_bf16(x, dim, fin_g, fin_b, eps, out, dim, M, dim, fin_gelu, stream);
  }
  bool normed = false;                         // xn holds the next product's input: the tail of the product before wrote it
  // x += A W^T + b, and the LayerNorm behind it where the product runs split-K (one launch sums the slabs, updates the stream and norms its rows)
  auto resid = [&](const uint16_t* A, int K, const uint16_t* W, const uint16_t* b, const uint16_t* g, const uint16_t* be, int act, uint16_t* y) -> int {
    const int ks = resid_slices(M, dim, K);
    normed = ks > 0 && mn_gemm256_supported(K, 0, K, dim, M, dim, K);
    if (!normed) return mn_gemm_bf16_parts(A, K, W, K, b, x, dim, M, dim, K, MN_GEMM_F32_RESID, stream);
    const int nz = mn_gemm256_splitk(A, K, 0, W, K, b, slabs, M, dim, K, ks, stream);
    return nz < 0 ? nz : mn_slab_resid_norm(slabs, nz, (int64_t)M * dim, x, dim, g, be, eps, act, y, dim, M, dim, stream);
  };
  for (int i = 0; i < depth; ++i, w += 12) {
    const bool last = i + 1 == depth;
    if (!normed) TRY(mn_layernorm_bf16(x, dim, w[0], w[1], eps, xn, dim, M, dim, 0, stream));
    TRY(mn_gemm_bf16_parts(xn, dim, w[2], dim, w[3], qkv, 3 * (int64_t)dim, M, 3 * dim, dim, MN_GEMM_BF16, stream));
    TRY(mn_attn_prefill_hd64(qkv, att, B, T, nh, causal, stream));
    TRY(resid(att, dim, w[4], w[5], w[6], w[7], 0, xn));
    if (!normed) TRY(mn_layernorm_bf16(x, dim, w[6], w[7], eps, xn, dim, M, dim, 0, stream));
    if (gelu) {
      TRY(mn_gemm_bf16(xn, dim, w[8], dim, w[9], h, hidden, M, hidden, dim, MN_GEMM_BF16_GELU, stream));
    } else {                                   // SwiGLU in the product's epilogue
      TRY(mn_gemm256_swiglu(xn, dim, 0, w[8], dim, w[9], h, hidden, M, hidden, dim, stream));
    }
    TRY(resid(h, hidden, w[10], w[11], last ? fin_g : w[12], last ? fin_b : w[13], last ? fin_gelu : 0, last ? out : xn));
  }
  if (!normed) TRY(mn_layernorm_bf16(x, dim, fin_g, fin_b, eps, out, dim, M, dim, fin_gelu, stream));
  return MN_OK;
}
