// An encoder layer of more than 64 rows: its seven launches from one call.
//
// From Python each launch costs the host 10 - 12 us (checks, views, allocations, the call): 84 of a layer stack of 12, where the
// layers of a few hundred rows take the device 30 - 60 us each, so that texts too long for a captured graph waited for the host
// (one text of 345 tokens, 12 layers of 768: 1092 us, 567 from here; 12 texts of 143 - 250, 384 wide, fp8: 1139, 719). The caller checks shapes and addresses, chooses
// each product's kernel by its own rules and lends the buffers; what is launched here, in which order and with which
// arguments is what the operations launch one by one.
#include "common.h"

namespace {

// The launchers, which live in libraries of their own.
typedef int (*GemmBf16)(const void*, int, const void*, void*, int, const void*, const void*, int, int, int, int, int, int, int,
                        void*, const void*, float, void*, void*, void*);
typedef int (*GemmF16)(const void*, int, const void*, void*, int, const void*, const void*, int, int, int, int, int, int, int,
                       void*, void*, void*, void*);
typedef int (*GemmRows)(const void*, int, const void*, void*, int, const void*, const void*, int, int, int, int, int, int, int,
                        void*);
typedef int (*GemmFp8)(const void*, int, const void*, const void*, const void*, void*, int, const void*, const void*, int, int,
                       int, int, int, void*);
typedef int (*Norm)(const void*, const void*, const void*, const void*, void*, int, int, float, void*);
typedef int (*NormFp8)(const void*, const void*, const void*, const void*, void*, void*, void*, int, int, float, void*);
typedef int (*AttnBf16)(const void*, const void*, const void*, int, int, int, const void*, int, int, int, int, int, int, float,
                        void*, int, const void*, const void*, long long, int, const void*, const void*, const void*, const void*,
                        void*);
typedef int (*AttnF16)(const void*, const void*, const void*, int, int, int, const void*, int, int, int, int, int, int, float,
                       void*, int, void*);

enum { KIND_BF16, KIND_F16, KIND_FP8 };
enum { W_QKV, B_QKV, W_O, B_O, LN1_G, LN1_B, W_UP, B_UP, W_DOWN, B_DOWN, LN2_G, LN2_B, W_QKV_SCALE, W_UP_SCALE, N_WEIGHTS };

struct Product {
  void *ws, *tail_ws, *tail_cnt;
  int tile, splits, rows, pad;  // rows: a tile of da_gemm_dk_rows
};

}  // namespace

struct EncoderLayer {
  void *gemm, *gemm_rows, *gemm_fp8, *attn, *norm;
  const void* w[N_WEIGHTS];
  void *x[3], *xq[3], *xscale[3];  // the layer's input, its middle and its result (xq, xscale: the same in e4m3)
  void *qkv, *a, *y[2], *f;
  const void* cu;
  Product p[4];
  int kind, T, B, max_len, heads, head_dim, hidden, ffn;
  float eps, scale;
};
static_assert(sizeof(EncoderLayer) == 472, "the caller's structure, field by field");

static int product(const EncoderLayer& L, int which, const void* A, int K, const void* W, const void* bias, int N, int epi,
                   const void* resid, void* C, void* s) {
  const Product& p = L.p[which];
  const int ldr = resid ? N : 0;
  if (p.rows)
    return ((GemmRows)L.gemm_rows)(A, K, W, C, N, bias, resid, ldr, L.T, N, K, epi, p.tile, L.kind == KIND_F16, s);
  if (L.kind == KIND_F16)
    return ((GemmF16)L.gemm)(A, K, W, C, N, bias, resid, ldr, L.T, N, K, epi, p.tile, p.splits, p.ws, p.tail_ws, p.tail_cnt, s);
  return ((GemmBf16)L.gemm)(A, K, W, C, N, bias, resid, ldr, L.T, N, K, epi, p.tile, p.splits, p.ws, nullptr, 0.f, p.tail_ws,
                            p.tail_cnt, s);
}

static int norm(const EncoderLayer& L, int i, int g, void* s) {
  if (L.kind == KIND_FP8)
    return ((NormFp8)L.norm)(L.y[i], nullptr, L.w[g], L.w[g + 1], L.x[i + 1], L.xq[i + 1], L.xscale[i + 1], L.T, L.hidden, L.eps, s);
  return ((Norm)L.norm)(L.y[i], nullptr, L.w[g], L.w[g + 1], L.x[i + 1], L.T, L.hidden, L.eps, s);
}

DA_EXPORT int da_encoder_layer(const EncoderLayer* layer, int epi_bias, int epi_gelu, int epi_resid, void* s) {
  const EncoderLayer& L = *layer;
  const int h = L.hidden, n = 3 * h, fp8 = L.kind == KIND_FP8;
  int e = fp8 ? ((GemmFp8)L.gemm_fp8)(L.xq[0], h, L.w[W_QKV], L.xscale[0], L.w[W_QKV_SCALE], L.qkv, n, L.w[B_QKV], nullptr, 0, L.T, n, h,
                                      epi_bias, s)
              : product(L, 0, L.x[0], h, L.w[W_QKV], L.w[B_QKV], n, epi_bias, nullptr, L.qkv, s);
  if (e) return e;
  const short *q = (const short*)L.qkv, *k = q + h, *v = k + h;
  e = L.kind == KIND_F16
          ? ((AttnF16)L.attn)(q, k, v, n, n, n, L.cu, L.B, L.max_len, L.heads, L.heads, L.head_dim, 0, L.scale, L.a, h, s)
          : ((AttnBf16)L.attn)(q, k, v, n, n, n, L.cu, L.B, L.max_len, L.heads, L.heads, L.head_dim, 0, L.scale, L.a, h, nullptr,
                               nullptr, 0, 0, nullptr, nullptr, nullptr, nullptr, s);
  if (e) return e;
  if ((e = product(L, 1, L.a, h, L.w[W_O], L.w[B_O], h, epi_resid, L.x[0], L.y[0], s))) return e;
  if ((e = norm(L, 0, LN1_G, s))) return e;
  e = fp8 ? ((GemmFp8)L.gemm_fp8)(L.xq[1], h, L.w[W_UP], L.xscale[1], L.w[W_UP_SCALE], L.f, L.ffn, L.w[B_UP], nullptr, 0, L.T, L.ffn, h,
                                  epi_gelu, s)
          : product(L, 2, L.x[1], h, L.w[W_UP], L.w[B_UP], L.ffn, epi_gelu, nullptr, L.f, s);
  if (e) return e;
  if ((e = product(L, 3, L.f, L.ffn, L.w[W_DOWN], L.w[B_DOWN], h, epi_resid, L.x[1], L.y[1], s))) return e;
  return norm(L, 1, LN2_G, s);
}
