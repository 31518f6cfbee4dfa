// A short text's encoder layers (one text, up to 64 rows) in one launch.
//
// A layer is four products that wait for one another (csrc/encoder_rows.hip: QKV; attention and its output product; the
// feed-forward's two), each of which takes 1 - 2 us of a launch of 5.5 - 7: the rest is its begin and end, and weights that are asked
// for when it begins. Here a workgroup of 16 waves takes tasks (16 rows of a strip of 16 columns, of two
// or four of the wide products), one after another, from a counter, asks for a task's weights at once, and then for its activations until they are there.
//
// Waiting. Nobody counts what is done: the activations are their own flags. All bits of the workspace are set before the launch, a layer has a
// place of its own in it, and every 8 B there are written once, by one store past the die's L2, never with all bits set (a NaN that would is
// another one); whoever reads them, past the L2s too, reads again until that is gone. That is a store and a load between two products;
// with a counter per product (store, its acknowledgement, an addition, its reading, the load) they were 7 us apart.
// Tasks are taken in order and wait for earlier ones only, and whoever took a task runs: the first that is not done always ends, with any number
// of workgroups on the chip. A wait has an end of its own all the same, after some seconds; then the result is NaNs, and a word of the host says so.
// A ticket is taken when the task before is done: taken ahead, a task of the next product began behind later ones (768 columns, 32 rows: 400 us for 229).
//
// Sums, statistics and roundings are in the order of the launches one by one (attention inside the output product): in bf16 the same bits.
//
// Activations are in strips of 16 columns, [strip][row][16], so that a store of a task fills its lines, and MFMA operands come straight from
// there in whole lines; V alone goes through LDS. What is left of a product is a chain: 1 us from the last store to the operand, norm 0.4,
// MFMAs and the waves' sums 0.6 - 0.9, epilogue 0.7. (A row block a task, also in the wide products: the norm of 32 rows in one took 0.4 longer.
// Waiting for one word first, or for one of the product before, so that waits read less: 165 - 184 us for 172, 16 rows of 768 columns.)
//
// Each phase has code of its own: as one loop body with the phase a value, its choices and the scalars that went to lanes and back were on the chain
// (12 layers of 768, 21 rows 187.5 -> 175.0, 24 of 1024, 32 rows 460 -> 446). That a wait which runs out is told costs 0.6 %.
// us, launches one by one / this, bf16: 12 layers of 384 x 1536, 16, 32, 48 and 64 rows 215 / 132, 217 / 140, 242 / 158 and 255 / 164, of 768 x 3072
// 253 / 161, 274 / 178, 346 / 217 and 348 / 253, 24 of 1024 x 4096, 16, 32, 36 and 64 rows 673 / 370, 731 / 446, 868 / 592 and 899 / 705; 4 of 768,
// 32 rows 94 / 69, 2 48 / 42.
#include <cstring>
#include <type_traits>

#include "gemm.h"

constexpr int TX_LAYERS = 32, TX_WAVES = 16;

enum { TX_QKV, TX_OUT, TX_UP, TX_DOWN };

struct TextLayer {
  const bf16_t *wqkv, *bqkv, *wo, *bo, *g1, *b1, *w1, *c1, *w2, *c2, *g2, *b2;
};

struct TextArgs {
  TextLayer L[TX_LAYERS];
  const bf16_t* x;  // [M, h]
  bf16_t* out;      // [M, h]: the last layer's sum, its norm not yet taken
  char* ws;         // per layer: qkv, the first sum, the feed-forward's middle, the second sum, and both sums' statistics; all bits set
  int* ticket;      // the last one taken; -1
  const int* cu;
  int* gave_up;  // of the host's memory, or null: 1 where a wait ran out
  int M, h, f, layers;
  int polls;  // minus the readings of a wait
  float eps, c;  // c: log2(e) times the scale of the scores
};

// A matrix of activations: strip j of 16 columns, row r and 16-B half x at j * strip + r * row + 16 x bytes.
struct TextMat {
  char* p;
  unsigned strip, row;
};

constexpr unsigned long long TX_EMPTY = ~0ull;  // four NaNs that no producer stores

__device__ __forceinline__ void tx_barrier() {  // (transfers stay on their way)
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

__device__ __forceinline__ void tx_put(void* p, unsigned long long v) {  // past the L2s, which are a die's own
  if (v == TX_EMPTY) v = 0x7fff7fff7fff7fffull;
  __hip_atomic_store((unsigned long long*)p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ bool tx_empty(const u32x4_t& v) { return (v[0] & v[1]) == ~0u || (v[2] & v[3]) == ~0u; }

template <int CTRL>
__device__ __forceinline__ float tx_dpp(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}
// Sums over 4 lanes beside one another, in each of them: lanes ^ 1, ^ 2; over 16: ^ 8, ^ 4, ^ 2, ^ 1 (as rotations, which come to that).
__device__ __forceinline__ float tx_sum4(float v) {
  v += tx_dpp<0xb1>(v);
  return v + tx_dpp<0x4e>(v);
}
__device__ __forceinline__ float tx_sum16(float v) {
  v += tx_dpp<0x128>(v);
  v += tx_dpp<0x124>(v);
  v += tx_dpp<0x122>(v);
  return v + tx_dpp<0x121>(v);
}
// op over lanes l, l ^ 16, l ^ 32 and l ^ 48
template <typename Op>
__device__ __forceinline__ float tx_rows(float v, Op op) {
  const unsigned u = __float_as_uint(v);
  const auto a = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  const unsigned x = __float_as_uint(op(__uint_as_float(a[0]), __uint_as_float(a[1])));
  const auto b = __builtin_amdgcn_permlane32_swap(x, x, false, false);
  return op(__uint_as_float(b[0]), __uint_as_float(b[1]));
}

// MB blocks of 16 rows, heads of D, NS strips a task of the wide products.
template <typename T, int MB, int D, int NS>
__global__ void __launch_bounds__(64 * TX_WAVES)
enc_text_kernel(const TextArgs p) {
  constexpr int R = 16 * MB, RED = NS * 256 > R * 32 ? NS * 256 : R * 32;
  constexpr int SC = 16;  // loads past the L2s
  __shared__ __attribute__((aligned(16))) float red[TX_WAVES][RED];  // each wave's sums; attention: its V before
  __shared__ float smean[16], srstd[16];
  __shared__ int snext;
  __shared__ int sgave;  // (in LDS: the pointer would take registers in every task)
  if (threadIdx.x == 0) sgave = 0;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int h = p.h, f = p.f, hs = h / 16;
  const int per = (3 * hs / NS + hs + f / (16 * NS) + hs) * MB, total = per * p.layers;
  auto tasks = [&](int phase) __attribute__((always_inline)) { return MB * (phase & 1 ? hs : (phase == TX_QKV ? 3 * hs : f / 16) / NS); };
  const size_t layer_bytes = (size_t)R * 2 * (5 * h + f) + 2 * (size_t)hs * R * 8;
  const unsigned S = R * 32;
  const int first = p.cu[0], end = min(p.cu[1], p.M);

  auto take = [&](int wave) __attribute__((always_inline)) {
    if (threadIdx.x == wave * 64) snext = __hip_atomic_fetch_add(p.ticket, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1;
  };
  // A task of the phase, which is a constant: each has code of its own.
  auto task = [&](auto of, const int layer, const int index) __attribute__((always_inline)) {
    constexpr int phase = decltype(of)::value;
    constexpr bool wide = !(phase & 1);
    const int strip = index / MB * (wide ? NS : 1), m0 = index % MB * 16;
    int lane = threadIdx.x & 63;
    asm volatile("" : "+v"(lane));  // (addresses of every phase kept from task to task would not fit the registers)
    const int tid = w * 64 + lane, fr = lane & 15, fg = lane >> 4;

    // ---- weights ----
    const TextLayer &L = p.L[layer], &P = p.L[max(layer - 1, 0)];
    const int K = phase == TX_DOWN ? f : h, units = K / 64;
    // as many waves as share the units evenly: wave w takes units w, w + nw, ..
    const int nw = units <= TX_WAVES ? units : units <= 2 * TX_WAVES ? (units + 1) / 2 : units <= 3 * TX_WAVES ? (units + 2) / 3 : (units + 3) / 4;
    const bool second = phase == TX_QKV || phase == TX_OUT;  // the norm before this task's operand or residual: the layer before's second
    const bf16_t *g = second ? P.g2 : L.g1, *b = second ? P.b2 : L.b1;
    const bool own = w < (wide ? NS : 1), normed = layer > 0 || phase >= TX_UP;
    u32x2_t ob{0, 0}, og{0, 0}, obb{0, 0};
    if (own) {
      const bf16_t* bias = phase == TX_QKV ? L.bqkv : phase == TX_OUT ? L.bo : phase == TX_UP ? L.c1 : L.c2;
      const int oc = (strip + w) * 16 + 4 * (lane & 3);
      ob = *(const u32x2_t*)(bias + oc);
      if (!wide) {
        og = *(const u32x2_t*)(g + oc);
        obb = *(const u32x2_t*)(b + oc);
      }
    }
    const bf16_t* W = phase == TX_QKV ? L.wqkv : phase == TX_OUT ? L.wo : phase == TX_UP ? L.w1 : L.w2;
    auto weights = [&](int unit, int at, bf16x8_t (&wf)[2]) __attribute__((always_inline)) {
      const bf16_t* row = W + (size_t)(at * 16 + fr) * K + unit * 64 + 8 * fg;
#pragma unroll
      for (int i = 0; i < 2; ++i) wf[i] = *(const bf16x8_t*)(row + 32 * i);
    };

    // ---- activations, as they come ----
    auto at = [&](int l) __attribute__((always_inline)) { return p.ws + l * layer_bytes; };
    const TextMat x = layer ? TextMat{at(layer - 1) + (size_t)(4 * h + f) * R * 2, S, 32} : TextMat{(char*)p.x, 32, (unsigned)h * 2};
    char* base = at(layer);
    const TextMat qkv{base, S, 32}, y{base + (size_t)3 * h * R * 2, S, 32}, mid{base + (size_t)4 * h * R * 2, S, 32};
    float2* st1 = (float2*)(base + (size_t)(5 * h + f) * R * 2);  // [4 rows][strip % 4][strip / 4][row]
    auto pieces = [&](const TextMat& m) __attribute__((always_inline)) {
      return __builtin_amdgcn_make_buffer_rsrc((void*)m.p, (short)0, 0x7fffff00, 0x00020000);
    };
    // 16-B chunk fg + 4 i of a unit's row r: a wave's lanes read whole lines
    auto chunk = [&](const TextMat& m, int i, int r, bool in) __attribute__((always_inline)) {
      return in ? (2 * i + (fg >> 1)) * m.strip + r * m.row + (fg & 1) * 16 : 0x7ffffff0u;
    };
    auto poll = [&](auto read) __attribute__((always_inline)) {
      int n = p.polls;
#pragma clang loop unroll(disable)
      for (; n < 0; ++n) {
        if (!__any(read())) break;
        __builtin_amdgcn_s_sleep(1);
      }
      if (n == 0) sgave = 1;
    };
    const int om = m0 + (lane >> 2), ostrip = strip + (wide ? w : 0);  // the result's row of this thread, and its strip
    const bool out = own && om < end;
    // beside the operand: the residual, and the statistics of four of the rows that are normed here, 16 lanes each
    unsigned long long orr = 0, q[4] = {};
    const bool stats = normed && w < 4;
    auto beside = [&](const TextMat& m) __attribute__((always_inline)) {
      const auto ld = [](const void* a) { return __hip_atomic_load((const unsigned long long*)a, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); };
      if (!wide && out) orr = ld(m.p + strip * m.strip + om * m.row + 8 * (tid & 3));
      if (stats) {
        const float2* st = (second ? (float2*)((char*)st1 - layer_bytes) + hs * R : st1) + (m0 / 4 + w) * hs * 4 + fg;
#pragma unroll
        for (int e = 0; e < 4; ++e) q[e] = ld(st + (e * (hs / 4) + min(fr, hs / 4 - 1)) * 4);  // strip 4 fr + e
      }
    };
    auto missing = [&]() __attribute__((always_inline)) {
      bool no = (layer > 0 || phase == TX_DOWN) && orr == TX_EMPTY;  // (the input is there)
      if (stats && m0 + 4 * w + fg < end) {
#pragma unroll
        for (int e = 0; e < 4; ++e) no |= q[e] == TX_EMPTY;
      }
      return no;
    };
    auto sums = [&](const f32x4_t& acc, int j) __attribute__((always_inline)) { if (w < nw) *(f32x4_t*)&red[w][(16 * j + fr) * 16 + 4 * fg] = acc; };
    auto statistics = [&]() __attribute__((always_inline)) {
      if (!stats) return;
      float2 sq[4];
      float a = 0.f, v = 0.f;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        sq[e] = __builtin_bit_cast(float2, q[e]);
        a += fr < hs / 4 ? sq[e].x : 0.f;
      }
      const float m = tx_sum16(a) / hs;
#pragma unroll
      for (int e = 0; e < 4; ++e) v += fr < hs / 4 ? fmaf(16.f * (sq[e].x - m), sq[e].x - m, sq[e].y) : 0.f;
      v = tx_sum16(v);
      if (fr == 0) {
        smean[4 * w + fg] = m;
        srstd[4 * w + fg] = rsqrtf(v / (16 * hs) + p.eps);
      }
    };

    // ---- weights, activations as they come, the product ----
    if (phase == TX_OUT) {
      f32x4_t acc[1]{f32x4_t{0.f, 0.f, 0.f, 0.f}};
      bf16x8_t wf[1][2] = {}, af[1 + MB][2] = {};
      if (w < units) weights(w, strip, wf[0]);
      asm volatile("" ::: "memory");
      {
        const auto rs = pieces(qkv);
        u32x4_t v[R / 8] = {};
        auto vread = [&]() __attribute__((always_inline)) {
#pragma unroll
          for (int j = 0; j < R / 8; ++j) {  // V, [4 strips][R rows][32 B]
            const int e = j * 64 + lane, r = e / 2 % R;
            v[j] = __builtin_amdgcn_raw_buffer_load_b128(rs, r >= first && r < end ? e * 16 : 0x7ffffff0u, (2 * hs + 4 * w) * S, SC);
          }
        };
        auto vmiss = [&]() __attribute__((always_inline)) {
          bool no = false;
#pragma unroll
          for (int j = 0; j < R / 8; ++j) no |= tx_empty(v[j]);
          return no;
        };
        poll([&] {
          beside(x);
          if (w >= units) return missing();
          u32x4_t u[2 + 2 * MB];
#pragma unroll
          for (int i = 0; i < 2; ++i) u[i] = __builtin_amdgcn_raw_buffer_load_b128(rs, chunk(qkv, i, m0 + fr, m0 + fr >= first && m0 + fr < end), 4 * w * S, SC);
#pragma unroll
          for (int n = 0; n < MB; ++n)
#pragma unroll
            for (int i = 0; i < 2; ++i)
              u[2 + 2 * n + i] = __builtin_amdgcn_raw_buffer_load_b128(rs, chunk(qkv, i, 16 * n + fr, 16 * n + fr >= first && 16 * n + fr < end), (hs + 4 * w) * S, SC);
          if constexpr (MB <= 2) vread();
          bool no = missing();
#pragma unroll
          for (int i = 0; i < 2 + 2 * MB; ++i) {
            no |= tx_empty(u[i]);
            af[i / 2][i % 2] = __builtin_bit_cast(bf16x8_t, u[i]);
          }
          if constexpr (MB <= 2) no |= vmiss();
          return no;
        });
        if (MB > 2 && w < units)  // (all at once does not fit the registers: 64 rows of 768 columns 290 us, 265 so)
          poll([&] {
            vread();
            return vmiss();
          });
#pragma unroll
        for (int j = 0; j < R / 8; ++j) *(u32x4_t*)((char*)red[w] + (j * 64 + lane) * 16) = v[j];
      }
      statistics();
      if (w < units) {
        constexpr int NH = 64 / D, NT = MB, NP = (MB + 1) / 2;  // keys: blocks of 16, and pairs of them
        f32x4_t s[NH][2 * NP];
        bf16x8_t pf[NH][NP];
        float inv[NH];
#pragma unroll
        for (int i = 0; i < NH; ++i) {
          float mx = -INFINITY;
          s[i][2 * NP - 1] = f32x4_t{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
#pragma unroll
          for (int n = 0; n < NT; ++n) {
            s[i][n] = T::mma16(af[1 + n][i], af[0][i], f32x4_t{0.f, 0.f, 0.f, 0.f});
            if (NH == 1) s[i][n] = T::mma16(af[1 + n][1], af[0][1], s[i][n]);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const int key = 16 * n + 4 * fg + e;
              if (key < first || key >= end) s[i][n][e] = -INFINITY;
              mx = fmaxf(mx, s[i][n][e]);
            }
          }
          mx = tx_rows(mx, [](float a, float b) { return fmaxf(a, b); });
          const float mc = mx == -INFINITY ? 0.f : fmaf(-mx, p.c, T::kF16 ? 0.f : -8.f);
          float all = 0.f;
#pragma unroll
          for (int n = 0; n < 2 * NP; ++n)
#pragma unroll
            for (int e = 0; e < 4; ++e) all += s[i][n][e] = __builtin_amdgcn_exp2f(fmaf(s[i][n][e], p.c, mc));
          all = tx_rows(all, [](float a, float b) { return a + b; });
          inv[i] = all > 0.f ? 1.f / all : 0.f;
#pragma unroll
          for (int n = 0; n < NP; ++n) {
            const f32x4_t a = s[i][2 * n], b = s[i][2 * n + 1];
            pf[i][n] = __builtin_bit_cast(bf16x8_t, u32x4_t{T::pack2(a[0], a[1]), T::pack2(a[2], a[3]), T::pack2(b[0], b[1]), T::pack2(b[2], b[3])});
          }
        }
        f32x4_t o[4];  // d = 32 (i / 2) + 8 fg + 4 (i & 1) + e of row fr
        const char* v = (const char*)red[w] + (4 * fg + (fr >> 2)) * 32;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int c = 4 * (i >> 1) + (fr & 3), a = (c >> 1) * R * 32 + (c & 1) * 16 + 8 * (i & 1);
          o[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int n = 0; n < NP; ++n) {
            const s16x4_t lo = lds_read_tr16(v + n * 1024 + a), up = 2 * n + 1 < MB ? lds_read_tr16(v + n * 1024 + 512 + a) : s16x4_t{0, 0, 0, 0};
            o[i] = T::mma16(bf16x8_t{lo[0], lo[1], lo[2], lo[3], up[0], up[1], up[2], up[3]}, pf[NH == 1 ? 0 : i >> 1][n], o[i]);
          }
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const float n = inv[NH == 1 ? 0 : i];
          const f32x4_t a = o[2 * i], b = o[2 * i + 1];
          const u32x4_t q{T::pack2(a[0] * n, a[1] * n), T::pack2(a[2] * n, a[3] * n), T::pack2(b[0] * n, b[1] * n), T::pack2(b[2] * n, b[3] * n)};
          acc[0] = T::mma16(wf[0][i], __builtin_bit_cast(bf16x8_t, q), acc[0]);
        }
      }
      sums(acc[0], 0);
    } else if (phase == TX_DOWN) {
      f32x4_t acc[1]{f32x4_t{0.f, 0.f, 0.f, 0.f}};
      const auto unit = [&](int n) { return w < nw ? w + n * nw : units; };
      bf16x8_t wf[4][2] = {}, af[4][2] = {};
#pragma unroll
      for (int n = 0; n < 4; ++n)
        if (unit(n) < units) weights(unit(n), strip, wf[n]);
      asm volatile("" ::: "memory");
      const auto rs = pieces(mid);
      poll([&] {
        beside(y);
#pragma unroll
        for (int n = 0; n < 4; ++n)
          if (unit(n) < units) {
#pragma unroll
            for (int i = 0; i < 2; ++i)
              af[n][i] = __builtin_bit_cast(bf16x8_t, __builtin_amdgcn_raw_buffer_load_b128(rs, chunk(mid, i, m0 + fr, m0 + fr < end), 4 * unit(n) * S, SC));
          }
        bool no = missing();
#pragma unroll
        for (int n = 0; n < 4; ++n)
          if (unit(n) < units) no |= tx_empty(__builtin_bit_cast(u32x4_t, af[n][0])) || tx_empty(__builtin_bit_cast(u32x4_t, af[n][1]));
        return no;
      });
      statistics();
#pragma unroll
      for (int n = 0; n < 4; ++n)
        if (unit(n) < units) {
#pragma unroll
          for (int i = 0; i < 2; ++i) acc[0] = T::mma16(wf[n][i], af[n][i], acc[0]);
        }
      sums(acc[0], 0);
    } else {
      f32x4_t acc[NS];
#pragma unroll
      for (int j = 0; j < NS; ++j) acc[j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      bf16x8_t wf[NS][2] = {}, af[2] = {};
      float gf[2][8] = {}, bf[2][8] = {};
      if (w < units) {
#pragma unroll
        for (int j = 0; j < NS; ++j) weights(w, strip + j, wf[j]);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const bf16x8_t gi = *(const bf16x8_t*)(g + w * 64 + fg * 8 + 32 * i), bi = *(const bf16x8_t*)(b + w * 64 + fg * 8 + 32 * i);
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            gf[i][e] = T::to_f((bf16_t)gi[e]);
            bf[i][e] = T::to_f((bf16_t)bi[e]);
          }
        }
      }
      asm volatile("" ::: "memory");
      const TextMat m = phase == TX_QKV ? x : y;
      const auto rs = pieces(m);
      poll([&] {
        beside(m);
        if (w >= units) return missing();
#pragma unroll
        for (int i = 0; i < 2; ++i)
          af[i] = __builtin_bit_cast(bf16x8_t, __builtin_amdgcn_raw_buffer_load_b128(rs, chunk(m, i, m0 + fr, m0 + fr < end), 4 * w * m.strip, SC));
        bool no = missing();
        no |= tx_empty(__builtin_bit_cast(u32x4_t, af[0]));
        no |= tx_empty(__builtin_bit_cast(u32x4_t, af[1]));
        return no && layer + phase > 0;  // (the input is there)
      });
      statistics();
      if (normed) tx_barrier();
      if (w < units) {
        if (normed) {
          const float mean = smean[fr], rstd = srstd[fr];
#pragma unroll
          for (int i = 0; i < 2; ++i) {
            const auto norm = [&](int e) __attribute__((always_inline)) { return fmaf((T::to_f((bf16_t)af[i][e]) - mean) * rstd, gf[i][e], bf[i][e]); };
            af[i] = __builtin_bit_cast(bf16x8_t, u32x4_t{T::pack2(norm(0), norm(1)), T::pack2(norm(2), norm(3)),
                                                         T::pack2(norm(4), norm(5)), T::pack2(norm(6), norm(7))});
          }
        }
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < NS; ++j) acc[j] = T::mma16(wf[j][i], af[i], acc[j]);
      }
#pragma unroll
      for (int j = 0; j < NS; ++j) sums(acc[j], j);
    }
    tx_barrier();
    take(TX_WAVES - 1);
    if (!own) return;

    // ---- the result ----
    const float* rd = &red[0][4 * tid];
    f32x4_t v = *(const f32x4_t*)rd;
    int u = 1;
    for (; u + 4 < nw; u += 5) {
      f32x4_t s[5];
#pragma unroll
      for (int j = 0; j < 5; ++j) s[j] = *(const f32x4_t*)(rd + (u + j) * RED);
#pragma unroll
      for (int j = 0; j < 5; ++j) v += s[j];
    }
    for (; u < nw; ++u) v += *(const f32x4_t*)(rd + u * RED);
    const auto val = [](const u32x2_t& o, int e) { return T::to_f((bf16_t)(e & 1 ? o[e >> 1] >> 16 : o[e >> 1] & 0xffff)); };
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] += val(ob, e);
    if (phase == TX_UP) {
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = gelu_erf(v[e]);
    } else if (!wide) {
      const u32x2_t rb = __builtin_bit_cast(u32x2_t, orr);
      const float mean = smean[om - m0], rstd = srstd[om - m0];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float r = val(rb, e);
        v[e] += normed ? T::to_f(T::from_f(fmaf((r - mean) * rstd, val(og, e), val(obb, e)))) : r;
      }
    }
    const u32x2_t o{T::pack2(v[0], v[1]), T::pack2(v[2], v[3])};
    const TextMat sum = layer + 1 < p.layers ? TextMat{base + (size_t)(4 * h + f) * R * 2, S, 32} : TextMat{(char*)p.out, 32, (unsigned)h * 2};
    const TextMat C = phase == TX_QKV ? qkv : phase == TX_OUT ? y : phase == TX_UP ? mid : sum;
    if (out) tx_put(C.p + ostrip * C.strip + om * C.row + 8 * (tid & 3), __builtin_bit_cast(unsigned long long, o));
    if (!wide) {  // statistics of the values as stored
      float z[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) z[e] = val(o, e);
      const float m = tx_sum4((z[0] + z[1]) + (z[2] + z[3])) * (1.f / 16.f);
      float d = 0.f;
#pragma unroll
      for (int e = 0; e < 4; ++e) d = fmaf(z[e] - m, z[e] - m, d);
      d = tx_sum4(d);
      if (out && (tid & 3) == 0) tx_put((phase == TX_OUT ? st1 : st1 + hs * R) + ((om >> 2) * hs + (strip & 3) * (hs / 4) + (strip >> 2)) * 4 + (om & 3), __builtin_bit_cast(unsigned long long, float2{m, d}));
    }
  };
  for (take(0);;) {
    tx_barrier();  // (the task before this one is done with LDS)
    const int t = __builtin_amdgcn_readfirstlane(snext);
    if (t >= total) {
      if (threadIdx.x == 0 && sgave && p.gave_up) __hip_atomic_store(p.gave_up, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      return;
    }
    // ---- the task ----
    const int layer = t / per;
    int index = t - layer * per, phase = TX_QKV;
#pragma unroll
    for (int e = TX_QKV; e < TX_DOWN; ++e)
      if (phase == e && index >= tasks(e)) {
        index -= tasks(e);
        phase = e + 1;
      }
    switch (phase) {
      case TX_QKV: task(std::integral_constant<int, TX_QKV>{}, layer, index); break;
      case TX_OUT: task(std::integral_constant<int, TX_OUT>{}, layer, index); break;
      case TX_UP: task(std::integral_constant<int, TX_UP>{}, layer, index); break;
      default: task(std::integral_constant<int, TX_DOWN>{}, layer, index);
    }
  }
}

// Before the launch: nothing is there, and rows behind the text, which the layers leave out, are zeros.
__global__ void __launch_bounds__(256) enc_text_empty_kernel(u32x4_t* ws, long n, u32x4_t* out, long n_out) {
  for (long i = blockIdx.x * 256l + threadIdx.x; i < n; i += gridDim.x * 256l) ws[i] = u32x4_t{~0u, ~0u, ~0u, ~0u};
  for (long i = blockIdx.x * 256l + threadIdx.x; i < n_out; i += gridDim.x * 256l) out[i] = u32x4_t{0, 0, 0, 0};
}

template <typename T>
__device__ __forceinline__ void tx_load(const bf16_t* p, float (&v)[8]) {
  const bf16x8_t u = *(const bf16x8_t*)p;
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] = T::to_f((bf16_t)u[e]);
}

template <typename T>
__device__ __forceinline__ u32x4_t tx_pack(const float (&v)[8]) {
  return u32x4_t{T::pack2(v[0], v[1]), T::pack2(v[2], v[3]), T::pack2(v[4], v[5]), T::pack2(v[6], v[7])};
}

// LayerNorm of a row of D <= 1024 columns, a wave: lane's columns 8 (lane + 64 i) + e, as the layernorm kernel does it.
template <typename T>
__device__ __forceinline__ void tx_norm(float (&v)[2][8], const bf16_t* g, const bf16_t* b, int lane, int D, float eps) {
  float s = 0.f, var = 0.f;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int e = 0; e < 8; ++e) s += (lane + 64 * i) * 8 < D ? v[i][e] : 0.f;
  const float mean = wave_sum(s) / D;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int e = 0; e < 8; ++e) var += (lane + 64 * i) * 8 < D ? (v[i][e] - mean) * (v[i][e] - mean) : 0.f;
  const float inv = rsqrtf(wave_sum(var) / D + eps);
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    float gv[8], bv[8];
    const int c = min((lane + 64 * i) * 8, D - 8);
    tx_load<T>(g + c, gv);
    tx_load<T>(b + c, bv);
#pragma unroll
    for (int e = 0; e < 8; ++e) v[i][e] = (v[i][e] - mean) * inv * gv[e] + bv[e];
  }
}

// The first of three launches for a text: its embeddings (a block a row) beside the emptied workspace.
template <typename T>
__global__ void __launch_bounds__(256)
enc_text_begin_kernel(const int* ids, const int* positions, const bf16_t* word, const bf16_t* pos, const bf16_t* type, const bf16_t* g,
                      const bf16_t* b, bf16_t* x, int M, int D, float eps, u32x4_t* ws, long n) {
  const int lane = threadIdx.x & 63, row = blockIdx.x;
  if (row >= M) {
    for (long i = (blockIdx.x - M) * 256l + threadIdx.x; i < n; i += (gridDim.x - M) * 256l) ws[i] = u32x4_t{~0u, ~0u, ~0u, ~0u};
    return;
  }
  if (threadIdx.x >= 64) return;
  const size_t wi = (size_t)ids[row] * D, pi = (size_t)positions[row] * D;
  float v[2][8];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    float q[8], t[8];
    const int c = min((lane + 64 * i) * 8, D - 8);
    tx_load<T>(word + wi + c, v[i]);
    tx_load<T>(pos + pi + c, q);
    tx_load<T>(type + c, t);
#pragma unroll
    for (int e = 0; e < 8; ++e) v[i][e] = v[i][e] + q[e] + t[e];
  }
  tx_norm<T>(v, g, b, lane, D, eps);
#pragma unroll
  for (int i = 0; i < 2; ++i)
    if ((lane + 64 * i) * 8 < D) *(u32x4_t*)(x + (size_t)row * D + (lane + 64 * i) * 8) = tx_pack<T>(v[i]);
}

// The last one: the norm behind the layers, the pooling (mode 0: the text's first row, 1: the mean of its rows) and the unit norm, in fp32. Rows and
// sums in the order of the pooling kernels: the same bits.
template <typename T>
__global__ void __launch_bounds__(64 * TX_WAVES)
enc_text_end_kernel(const bf16_t* y, const bf16_t* g, const bf16_t* b, const int* cu, int M, int D, float eps, int mode, float* out) {
  constexpr int NT = 64 * TX_WAVES;
  __shared__ __attribute__((aligned(16))) char smem[64 * 1024 * 2];  // the normed rows, and then each thread's sums
  __shared__ float red[16];
  bf16_t* rows = (bf16_t*)smem;
  float* part = (float*)smem;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, first = min(max(cu[0], 0), M - 1), n = mode ? max(min(cu[1], M) - first, 1) : 1;
  for (int r = w; r < n; r += TX_WAVES) {
    float v[2][8];
#pragma unroll
    for (int i = 0; i < 2; ++i) tx_load<T>(y + (size_t)(first + r) * D + min((lane + 64 * i) * 8, D - 8), v[i]);
    tx_norm<T>(v, g, b, lane, D, eps);
#pragma unroll
    for (int i = 0; i < 2; ++i)
      if ((lane + 64 * i) * 8 < D) *(u32x4_t*)(rows + r * D + (lane + 64 * i) * 8) = tx_pack<T>(v[i]);
  }
  __syncthreads();
  // threads of 8 columns, and each the rows gr, gr + G, ..
  const int nch = D / 8, G = NT / nch, gr = threadIdx.x / nch, c = threadIdx.x % nch;
  float v[8] = {}, ss = 0.f;
  if (gr < G)
    for (int t = gr; t < n; t += G) {
      float a[8];
      tx_load<T>(rows + t * D + c * 8, a);
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] += a[e];
    }
  __syncthreads();
#pragma unroll
  for (int e = 0; e < 8; ++e) part[threadIdx.x * 8 + e] = v[e];
  __syncthreads();
  if (gr == 0) {
    for (int i = 1; i < min(G, n); ++i)
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] += part[(i * nch + c) * 8 + e];
    const float invn = 1.f / (float)n;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      v[e] *= invn;
      ss += v[e] * v[e];
    }
  }
  ss = block_sum(ss, red);
  const float inv = ss > 0.f ? rsqrtf(ss) : 1.f;
  if (gr) return;
#pragma unroll
  for (int e = 0; e < 8; ++e) out[c * 8 + e] = v[e] * inv;
}

// Bytes of da_enc_text's workspace; 0: it does not take such a text.
DA_EXPORT long long da_enc_text_ws(int M, int h, int f, int layers, int D, int f16) {
  if (M < 1 || M > 64 || layers < 1 || layers > TX_LAYERS || h < 64 || h % 64 || h > 64 * TX_WAVES || f < 64 || f % 64 || f > 256 * TX_WAVES ||
      (D != 64 && (D != 32 || f16)))
    return 0;
  const long long R = (M + 15) / 16 * 16;
  return layers * (R * 2 * (5ll * h + f) + 2 * (h / 16) * R * 8) + 256;  // (and the ticket)
}

// Workgroups: as many as two neighbouring products have tasks, whose weights travel while the product before is taken; each has a CU to itself, so
// that with 256 nothing else runs until the last task. us, 256 / 192 / 144 workgroups, 12 layers of 768, 16 rows 157 / 157 / 160 (144 of two
// products), 32 rows 180 / 178 / 223 (192), 64 rows 253 / 279 / 382; of 384, 32 rows 143 / 142 / 140 (144), 48 162 / 162 / 159 (144), 64 168 / 164 /
// 182 (192). Wider ones take all: their weights are longer on the way (24 of 1024, 16 rows 369 / 391 / 440, 32 446 / 545 / 631).
// Beside decode steps (of a 3.8B, one row, 1.72 ms alone; questions of 21 tokens and 768 columns 5 ms apart / one upon another; the launches one by one):
// a step 1.80 / 6.8 ms with 256, 1.77 / 3.3 with 192 (1.76 / 1.95), a question 247 / 222 us, 251 / 219 (597 / 573). Of 1024 columns: a step 1.90 / 15.1 ms
// with 256, 1.85 / 4.0 with 192 (1.81 / 2.13), a question 498 / 478 us, 623 / 608 (1346 / 1324).
static int enc_text_grid(int M, int h, int f, int ns) {
  const int mb = (M + 15) / 16, out = h / 16 * mb, qkv = 3 * out / ns, up = f / 16 * mb / ns;
  const int two = out + (qkv > up ? qkv : up);
  return h > 768 || two > 256 ? 256 : two < 96 ? 96 : (two + 15) / 16 * 16;
}

// x [M, h] through the layers (pointers of TextLayer each, of the host): out [M, h] is the last layer's sum before its norm. One text, rows
// cu[0] .. cu[1] - 1.
static int enc_text(const void* x, const void* const* layers, int n, void* out, void* ws, const int* cu, int M, int h, int f, int D, float eps,
                    float c, int f16, int* gave_up, int polls, hipStream_t s) {
  const long long bytes = da_enc_text_ws(M, h, f, n, D, f16);
  TextArgs a{};
  std::memcpy(a.L, layers, n * sizeof(TextLayer));
  a.x = (const bf16_t*)x; a.out = (bf16_t*)out; a.ws = (char*)ws; a.ticket = (int*)((char*)ws + bytes - 256); a.cu = cu;
  a.gave_up = gave_up; a.polls = -polls;
  a.M = M; a.h = h; a.f = f; a.layers = n; a.eps = eps; a.c = c;
  // strips a task: with four fewer tasks read a block's activations and take its norm, with two a task has fewer weights (us, four / two: 32 rows
  // of 1024 columns, 24 layers 484 / 555, of 768, 12 209 / 216, of 512, 8 126 / 121, of 384, 12 178 / 168; 64 rows of 768 290 / 334, of 384
  // 194 / 204; 16 rows of 768 198 / 173, with one 191)
  const int ns = M <= 16 || (M <= 32 && h <= 512) ? 2 : 4, grid = enc_text_grid(M, h, f, ns);
#define ENC_TEXT(T, DD)                                                                 \
  do {                                                                                  \
    if (M <= 16) enc_text_kernel<T, 1, DD, 2><<<grid, 64 * TX_WAVES, 0, s>>>(a);        \
    else if (M > 48) enc_text_kernel<T, 4, DD, 4><<<grid, 64 * TX_WAVES, 0, s>>>(a);    \
    else if (M > 32) enc_text_kernel<T, 3, DD, 4><<<grid, 64 * TX_WAVES, 0, s>>>(a);    \
    else if (ns == 2) enc_text_kernel<T, 2, DD, 2><<<grid, 64 * TX_WAVES, 0, s>>>(a);   \
    else enc_text_kernel<T, 2, DD, 4><<<grid, 64 * TX_WAVES, 0, s>>>(a);                \
  } while (0)
  if (D == 32) ENC_TEXT(BF16T, 32);
  else if (f16) ENC_TEXT(F16T, 64);
  else ENC_TEXT(BF16T, 64);
#undef ENC_TEXT
  return (int)hipGetLastError();
}

DA_EXPORT int da_enc_text(const void* x, const void* const* layers, int n, void* out, void* ws, const int* cu, int M, int h, int f, int D,
                         float eps, float c, int f16, int* gave_up, int polls, void* stream) {
  const long long bytes = da_enc_text_ws(M, h, f, n, D, f16);
  if (!bytes || !x || !layers || !out || !ws || !cu) return (int)hipErrorInvalidValue;
  enc_text_empty_kernel<<<512, 256, 0, (hipStream_t)stream>>>((u32x4_t*)ws, bytes / 16, (u32x4_t*)out, M * h / 8);
  return enc_text(x, layers, n, out, ws, cu, M, h, f, D, eps, c, f16, gave_up, polls, (hipStream_t)stream);
}

// The whole encoder of such a text: ids and positions [M] to its pooled unit vector, out fp32 [h]. emb: word, position and type tables, their
// norm's gain and shift. x, y [M, h]: scratch. Three launches behind one call want no graph, whose end the next call's
// copy waits 18 us for, nor a text filled up to a length: a question 218 -> 200 us.
DA_EXPORT int da_enc_text_pooled(const void* ids, const void* positions, const void* const* emb, const void* const* layers, int n, void* x, void* y,
                                void* ws, const int* cu, int M, int h, int f, int D, float eps, float c, int mode, void* out, int f16,
                                int* gave_up, int polls, void* stream) {
  const long long bytes = da_enc_text_ws(M, h, f, n, D, f16);
  if (!bytes || !ids || !positions || !emb || !layers || !x || !y || !ws || !cu || !out) return (int)hipErrorInvalidValue;
  hipStream_t s = (hipStream_t)stream;
  const bf16_t *const *e = (const bf16_t* const*)emb, *const *last = (const bf16_t* const*)layers + (size_t)12 * (n - 1);
  const auto begin = f16 ? enc_text_begin_kernel<F16T> : enc_text_begin_kernel<BF16T>;
  begin<<<M + 512, 256, 0, s>>>((const int*)ids, (const int*)positions, e[0], e[1], e[2], e[3], e[4], (bf16_t*)x, M, h, eps, (u32x4_t*)ws, bytes / 16);
  const int err = enc_text(x, layers, n, y, ws, cu, M, h, f, D, eps, c, f16, gave_up, polls, s);
  if (err) return err;
  const auto end = f16 ? enc_text_end_kernel<F16T> : enc_text_end_kernel<BF16T>;
  end<<<1, 64 * TX_WAVES, 0, s>>>((const bf16_t*)y, last[10], last[11], cu, M, h, eps, mode, (float*)out);
  return (int)hipGetLastError();
}

// The device's address of pinned host memory.
DA_EXPORT int da_host_address(void* host, void** out) { return (int)hipHostGetDevicePointer(out, host, 0); }
