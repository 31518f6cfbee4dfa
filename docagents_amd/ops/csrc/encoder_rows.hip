// Encoder products for few rows (a question: <= 64 tokens), with the LayerNorms between them inside: five launches a layer,
// four where attention is inside the product behind it.
//
//   C[M, N] = epi(LN(A)[M, K] . W[N, K]^T + bias)      epi: none / GELU
//   C[M, N] = A . W^T + bias + LN(R)                   and the row statistics that the next LN needs
//
// A post-norm layer's LayerNorm sits between two products and its output is read twice, as the next product's operand and
// as the residual after it. Here no launch writes it: the product that makes the sum y also writes, for each row and 16
// columns, their mean and sum of squared deviations; its readers merge those (K / 16 pairs a row: the pairwise variance
// formula of Chan, Golub and LeVeque, no cancellation) and normalise y as they load it, rounded to bf16 like the row that
// the layernorm kernel stores.
//
// What bounds it is latency: 12 layers' 170 MB are 35 us at HBM's rate, a launch is 4 - 5. So a workgroup is a strip of
// 16 columns (48 - 256 of them) whose up to 16 waves take K in units of 64 in turn, and the waves' sums meet in LDS once. A unit
// arrives by LDS-DMA, 128 B of every row, into a stage that is the wave's own: a CU has 256 requests on their way, and
// operands straight in MFMA layout are requests of 64 B, twice as many. A wave waits for its own transfers only; the statistics
// are asked for first and merged while the weights are on their way.
// 21 rows of 12 layers of 768 x 3072 columns, us a launch, operands straight to the MFMA / by LDS-DMA: K = 3072 8.7 / 6.2, a norm
// on A 6.3 / 5.4 (without GELU) and 6.7 / 5.9 (with it), K = 768 4.2 / 4.3; the question 375 -> 333 us, 60 tokens through 24
// layers of 1024 in fp16 1028 -> 926, 16 + 20 through 384 columns 315 -> 311. A dk product, a norm, or a split-K product with
// its reduce took 5.2 / 7.1, 4.6 and 9.7.
#include "gemm.h"

typedef __attribute__((address_space(3))) void* lds_ptr_t;

struct EncRowsArgs {
  const bf16_t *A, *W, *bias, *resid;
  bf16_t* C;
  const float* st;        // [64 rows][64 parts] (mean, squared deviations) of the rows that are normalised; null: none are
  const bf16_t *g, *b;    // gain and shift of that norm
  float* st_out;          // RESID: the same of the rows of C, a part per 16 columns
  int M, N, K, lda, ldc, ldr, parts;
  float eps;
  const int* cu;  // attention: the text's first row and its end
  float c;        // and log2(e) times the scale of the scores
};

// The waves' stages (ST of each) and, after the last unit, their sums share LDS: up to enc_waves(FM) waves.
constexpr int enc_waves(int fm) { return fm == 4 ? 12 : 16; }
constexpr int enc_stages(int fm) { return fm == 1 ? 2 : 1; }

// Attention inside the product that takes its output (D != 0: heads of D; A is then q, k and v beside one another, one text of
// KR rows at most): a unit of 64 k is a head of 64 or two of 32, so its wave attends for the block's 16 rows and the result is
// its MFMA operand as it stands. S^T = K Q^T leaves a lane keys 16 t + 4 fg + e of its row, which is P's operand if V's rows
// come in that order, and V's columns are read so that a lane of O^T has 8 in a row. Scores and weights as in the attention
// kernels: the maximum and the sums in fp32, weights rounded to the type (bf16: of 2^-8 times them, so that sums of the largest
// values stay in fp32). Rows outside the text read as zero.
// All strips do the same attention over again. What it costs is its operands (10 KB a wave at 32 rows, which other dies have just
// written), so they come by LDS-DMA, and only the text's: straight to the MFMA the question took as long as with a launch
// between, 64 rows 10 % longer. Texts that share blocks had to take turns with V (a NaN of one reaches another through weights
// of zero), 6 us a layer for seven: one text only. One of 21 tokens through 12 layers of 768: 333 -> 302 us, of 20 through 384
// (heads of 32) 278 -> 246, of 60 there 310 -> 285, of 20 through 24 of 1024 811 -> 760.
template <typename T, int FM, bool LNA, int EPI, int D = 0, int KR = 0, int UNITS = 0>
__global__ void __launch_bounds__(64 * enc_waves(FM))
enc_rows_kernel(EncRowsArgs p) {
  constexpr int ROWS = FM * 16, SLD = 20, ST = enc_stages(FM), A_BYTES = ROWS * 128, STAGE = A_BYTES + 2048;
  constexpr int PA = 2 * FM, P = PA + 2;  // LDS-DMA instructions of a stage
  constexpr bool WIDE = UNITS > 12;  // (W straight to registers, the statistics in LDS after the sums: 160 KB are full)
  constexpr int RING = D ? KR * 256 + (WIDE ? 2048 : 4096) : ST * STAGE;  // a wave's stages, or its K, V, Q and W
  static_assert(ROWS * SLD * 4 <= RING, "the sums fit the stages");
  static_assert(!D || (FM == 1 && !LNA), "attention: 16 rows a block");
  __shared__ __attribute__((aligned(16))) char smem[(D ? UNITS : enc_waves(FM)) * RING];
  __shared__ float sstat[WIDE ? 1 : 2 * ROWS];
  float *smean = WIDE ? (float*)smem + 16 * ROWS * SLD : sstat, *srstd = smean + ROWS;
  float (*red)[ROWS][SLD] = (float (*)[ROWS][SLD])smem;
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), nw = blockDim.x >> 6;
  const int fr = lane & 15, fg = lane >> 4;
  const int n0 = blockIdx.x * 16, units = p.K / 64, rows = p.M, m0 = blockIdx.y * ROWS;
  int first = 0, end = 0;  // the text (attention)
  if constexpr (D != 0) {
    first = p.cu[0];
    end = min(p.cu[1], rows);
  }
  {  // this block's rows
    p.M -= m0;
    if (!D) p.A += (size_t)m0 * p.lda;
    p.C += (size_t)m0 * p.ldc;
    if (p.resid) p.resid += (size_t)m0 * p.ldr;
    if (p.st) p.st += m0 * 128;
    if (p.st_out) p.st_out += m0 * 128;
  }

  // ---- requests: statistics (16 lanes a row, 4 parts each) and the epilogue's operands, then the product's ----
  const int sl = lane & 15;
  f32x4_t s0, s1;
  auto stats_load = [&](int r) __attribute__((always_inline)) {
    const f32x4_t* q = (const f32x4_t*)(p.st + (size_t)min(r, p.M - 1) * 128 + sl * 8);
    s0 = q[0];
    s1 = q[1];
  };
  auto stats_merge = [&](int r) __attribute__((always_inline)) {
    const float mean[4] = {s0[0], s0[2], s1[0], s1[2]}, dev[4] = {s0[1], s0[3], s1[1], s1[3]};
    float a = 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) a += sl * 4 + e < p.parts ? mean[e] : 0.f;
#pragma unroll
    for (int x = 8; x; x >>= 1) a += __shfl_xor(a, x, 64);
    const float m = a / p.parts;
    float v = 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) v += sl * 4 + e < p.parts ? fmaf(16.f * (mean[e] - m), mean[e] - m, dev[e]) : 0.f;
#pragma unroll
    for (int x = 8; x; x >>= 1) v += __shfl_xor(v, x, 64);
    if (sl == 0 && r < ROWS) {
      smean[r] = m;
      srstd[r] = rsqrtf(v / (16 * p.parts) + p.eps);
    }
  };
  if (p.st) stats_load(4 * w + fg);
  const int om = tid >> 2, oc = n0 + 4 * (tid & 3);  // the output row and columns of this thread (tid < 4 * ROWS)
  const bool out = om < p.M && tid < 4 * ROWS;
  u32x2_t ob{0, 0}, orr{0, 0}, og{0, 0}, obb{0, 0};
  if (out) {
    if (p.bias) ob = *(const u32x2_t*)(p.bias + oc);
    if constexpr (EPI == EPI_RESID) {
      orr = *(const u32x2_t*)(p.resid + (size_t)om * p.ldr + oc);
      if (p.st && FM < 4) {
        og = *(const u32x2_t*)(p.g + oc);
        obb = *(const u32x2_t*)(p.b + oc);
      }
    }
  }
  asm volatile("" ::: "memory");
  const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc((void*)p.A, (short)0, 0x7fffff00, 0x00020000);
  const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc((void*)(p.W + (size_t)n0 * p.K), (short)0, 0x7fffff00, 0x00020000);
  char* ring = smem + w * RING;
  constexpr int NT = D ? KR / 16 : 1;
  bf16x8_t aw[2];
  if constexpr (D != 0) {  // unit w; rows outside the text read as zero
    if constexpr (WIDE) {
#pragma unroll
      for (int h = 0; h < 2; ++h) aw[h] = *(const bf16x8_t*)(p.W + (size_t)(n0 + fr) * p.K + w * 64 + 32 * h + 8 * fg);
    } else {
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int r = 8 * j + (lane >> 3);
        const unsigned at = (unsigned)r * (unsigned)(p.K * 2) + (((lane & 7) ^ ((r >> 1) & 7)) << 4);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, (lds_ptr_t)(ring + KR * 256 + 2048 + j * 1024), 16, at, w * 128, 0, 0);
      }
    }
    asm volatile("" ::: "memory");
    auto row = [&](int r, int at) __attribute__((always_inline)) { return r >= first && r < end ? (unsigned)r * (unsigned)(p.lda * 2) + at : 0x7ffffff0u; };
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int r = 8 * j + (lane >> 3);
      const unsigned at = row(m0 + r, ((lane & 7) ^ ((r >> 1) & 7)) << 4);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (lds_ptr_t)(ring + KR * 256 + j * 1024), 16, at, w * 128, 0, 0);
    }
#pragma unroll
    for (int j = 0; j < KR / 8; ++j) {
      const int r = 8 * j + (lane >> 3);
      const unsigned at = row(r, ((lane & 7) ^ ((r >> 1) & 7)) << 4);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (lds_ptr_t)(ring + j * 1024), 16, at, p.K * 2 + w * 128, 0, 0);
    }
    asm volatile("" ::: "memory");
#pragma unroll
    for (int j = 0; j < KR / 8; ++j) {  // (last, for the wait: V's chunk c of row r at slot c ^ ((r & 2) << 1))
      const int r = 8 * j + (lane >> 3);
      const unsigned at = row(r, ((lane & 7) ^ ((r & 2) << 1)) << 4);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (lds_ptr_t)(ring + KR * 128 + j * 1024), 16, at, p.K * 4 + w * 128, 0, 0);
    }
  }
  // ---- the wave's units w, w + nw, ..: row r's 16-B chunk c of 64 k at slot c ^ (r >> 1 & 7) of its 128 B ----
  unsigned ao[8], wo[2];  // rows past M: past the resource's end, which reads as zero
#pragma unroll
  for (int j = 0; j < PA; ++j) {
    const int r = 8 * j + (lane >> 3), c = (lane & 7) ^ ((r >> 1) & 7);
    ao[j] = r < p.M ? (unsigned)r * (unsigned)(p.lda * 2) + c * 16 : 0x7ffffff0u;
  }
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int r = 8 * j + (lane >> 3), c = (lane & 7) ^ ((r >> 1) & 7);
    wo[j] = (unsigned)r * (unsigned)(p.K * 2) + c * 16;
  }
  auto ask = [&](int u, int slot) __attribute__((always_inline)) {
    char* base = ring + slot * STAGE;
#pragma unroll
    for (int j = 0; j < 2; ++j)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, (lds_ptr_t)(base + A_BYTES + j * 1024), 16, wo[j], u * 128, 0, 0);
#pragma unroll
    for (int j = 0; j < PA; ++j)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (lds_ptr_t)(base + j * 1024), 16, ao[j & 7], u * 128, 0, 0);
  };
  bf16x8_t gf[2], bf[2];
  auto norm_load = [&](int u) __attribute__((always_inline)) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      gf[h] = *(const bf16x8_t*)(p.g + u * 64 + fg * 8 + 32 * h);
      bf[h] = *(const bf16x8_t*)(p.b + u * 64 + fg * 8 + 32 * h);
    }
  };
  if constexpr (LNA) norm_load(min(w, units - 1));
#pragma unroll
  for (int i = 0; i < ST; ++i)
    if (!D && w + i * nw < units) ask(w + i * nw, i);
  if (p.st && !WIDE) {
    asm volatile("" ::: "memory");
    stats_merge(4 * w + fg);
    for (int r = 4 * (w + nw) + fg; r - fg < ROWS; r += 4 * nw) {
      stats_load(r);
      stats_merge(r);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // (the transfers stay on their way)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  }
  f32x4_t acc[FM];
#pragma unroll
  for (int i = 0; i < FM; ++i) acc[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  if constexpr (D != 0) {
    constexpr int NH = 64 / D;
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(KR / 8) : "memory");  // everything but V
    __builtin_amdgcn_sched_barrier(0);
    const int at[2] = {fr * 128 + ((fg ^ ((fr >> 1) & 7)) << 4), fr * 128 + (((4 + fg) ^ ((fr >> 1) & 7)) << 4)};
    bf16x8_t aq[2], ak[4][2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if constexpr (!WIDE) aw[h] = *(const bf16x8_t*)(ring + KR * 256 + 2048 + at[h]);
      aq[h] = *(const bf16x8_t*)(ring + KR * 256 + at[h]);
#pragma unroll
      for (int t = 0; t < NT; ++t) ak[t][h] = *(const bf16x8_t*)(ring + t * 2048 + at[h]);
    }
    f32x4_t s[2][4];
    bf16x8_t pf[2][2];
    float inv[2];
#pragma unroll
    for (int h = 0; h < NH; ++h) {
      float mx = -INFINITY;
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        s[h][t] = T::mma16(ak[t][h], aq[h], f32x4_t{0.f, 0.f, 0.f, 0.f});
        if (NH == 1) s[h][t] = T::mma16(ak[t][1], aq[1], s[h][t]);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int key = 16 * t + 4 * fg + e;
          if (key < first || key >= end) s[h][t][e] = -INFINITY;
          mx = fmaxf(mx, s[h][t][e]);
        }
      }
      mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
      mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
      const float mc = mx == -INFINITY ? 0.f : fmaf(-mx, p.c, T::kF16 ? 0.f : -8.f);
      float sum = 0.f;
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int e = 0; e < 4; ++e) sum += s[h][t][e] = __builtin_amdgcn_exp2f(fmaf(s[h][t][e], p.c, mc));
      sum += __shfl_xor(sum, 16, 64);
      sum += __shfl_xor(sum, 32, 64);
      inv[h] = sum > 0.f ? 1.f / sum : 0.f;
#pragma unroll
      for (int t = 0; t < NT; t += 2)
        pf[h][t / 2] = __builtin_bit_cast(bf16x8_t, u32x4_t{T::pack2(s[h][t][0], s[h][t][1]), T::pack2(s[h][t][2], s[h][t][3]),
                                                            T::pack2(s[h][t + 1][0], s[h][t + 1][1]), T::pack2(s[h][t + 1][2], s[h][t + 1][3])});
    }
    f32x4_t o[4];  // d = 32 (i / 2) + 8 fg + 4 (i & 1) + e of row fr
#pragma unroll
    for (int i = 0; i < 4; ++i) o[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // V
    __builtin_amdgcn_sched_barrier(0);
    const char* v = ring + KR * 128 + (4 * fg + (fr >> 2)) * 128;
#pragma unroll
    for (int t = 0; t < NT; t += 2)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int at = ((4 * (i >> 1) + (fr & 3)) ^ ((fr >> 3) << 2)) * 16 + 8 * (i & 1);
        const s16x4_t lo = lds_read_tr16(v + t * 2048 + at), up = lds_read_tr16(v + (t + 1) * 2048 + at);
        o[i] = T::mma16(bf16x8_t{lo[0], lo[1], lo[2], lo[3], up[0], up[1], up[2], up[3]}, pf[NH == 1 ? 0 : i >> 1][t / 2], o[i]);
      }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const float n = inv[NH == 1 ? 0 : h];
      const f32x4_t a = o[2 * h], b = o[2 * h + 1];
      const u32x4_t x{T::pack2(a[0] * n, a[1] * n), T::pack2(a[2] * n, a[3] * n), T::pack2(b[0] * n, b[1] * n), T::pack2(b[2] * n, b[3] * n)};
      acc[0] = T::mma16(aw[h], __builtin_bit_cast(bf16x8_t, x), acc[0]);
    }
  }
  const int sw = (fr >> 1) & 7;
  const int co[2] = {(fg ^ sw) << 4, ((4 + fg) ^ sw) << 4};
#pragma unroll 1
  for (int u = D ? units : w, slot = 0; u < units; u += nw) {
    if (LNA && u != w) norm_load(u);
    // this unit is in: everything but the stage behind it (with a norm: everything)
    if (!LNA && ST > 1 && u + nw < units) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(P * (ST - 1)) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    const char* s = ring + slot * STAGE + fr * 128;
    bf16x8_t wf[2], af[2][FM];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      wf[h] = *(const bf16x8_t*)(s + A_BYTES + co[h]);
#pragma unroll
      for (int i = 0; i < FM; ++i) af[h][i] = *(const bf16x8_t*)(s + i * 2048 + co[h]);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // and read: its stage is free
    __builtin_amdgcn_sched_barrier(0);
    if (u + ST * nw < units) ask(u + ST * nw, slot);
    slot = slot + 1 == ST ? 0 : slot + 1;
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < FM; ++i) {
        bf16x8_t a = af[h][i];
        if constexpr (LNA) {
          const float mean = smean[16 * i + fr], rstd = srstd[16 * i + fr];
          u32x4_t y;
#pragma unroll
          for (int e = 0; e < 4; ++e)
            y[e] = T::pack2(fmaf((T::to_f((bf16_t)a[2 * e]) - mean) * rstd, T::to_f((bf16_t)gf[h][2 * e]), T::to_f((bf16_t)bf[h][2 * e])),
                            fmaf((T::to_f((bf16_t)a[2 * e + 1]) - mean) * rstd, T::to_f((bf16_t)gf[h][2 * e + 1]),
                                 T::to_f((bf16_t)bf[h][2 * e + 1])));
          a = __builtin_bit_cast(bf16x8_t, y);
        }
        acc[i] = T::mma16(wf[h], a, acc[i]);  // (W first: a lane has 4 columns of a row)
      }
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < FM; ++i) *(f32x4_t*)&red[w][16 * i + fr][4 * fg] = acc[i];
  if (WIDE && p.st) stats_merge(4 * w + fg);  // (13 waves or more: all rows)
  __syncthreads();
  if (tid >= 4 * ROWS) return;  // (whole waves)
  if (EPI == EPI_RESID && FM == 4 && out && p.st) {  // (no registers for them before)
    og = *(const u32x2_t*)(p.g + oc);
    obb = *(const u32x2_t*)(p.b + oc);
  }
  f32x4_t v = *(const f32x4_t*)&red[0][om][4 * (tid & 3)];
  for (int x = 1; x < nw; ++x) v += *(const f32x4_t*)&red[x][om][4 * (tid & 3)];
  float y[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    auto half = [&](const u32x2_t& q) { return T::to_f((bf16_t)(e & 1 ? q[e >> 1] >> 16 : q[e >> 1] & 0xffff)); };
    y[e] = v[e] + half(ob);
    if constexpr (EPI == EPI_GELU) y[e] = gelu_erf(y[e]);
    if constexpr (EPI == EPI_RESID) {
      float r = half(orr);
      if (p.st) r = T::to_f(T::from_f(fmaf((r - smean[om]) * srstd[om], half(og), half(obb))));
      y[e] += r;
    }
  }
  const u32x2_t o{T::pack2(y[0], y[1]), T::pack2(y[2], y[3])};
  if (out) *(u32x2_t*)(p.C + (size_t)om * p.ldc + oc) = o;
  if constexpr (EPI == EPI_RESID) {  // of the values as stored
    float q[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) q[e] = T::to_f((bf16_t)(e & 1 ? o[e >> 1] >> 16 : o[e >> 1] & 0xffff));
    float s = (q[0] + q[1]) + (q[2] + q[3]);
    s += __shfl_xor(s, 1, 64);
    s += __shfl_xor(s, 2, 64);
    const float m = s * (1.f / 16.f);
    float d = 0.f;
#pragma unroll
    for (int e = 0; e < 4; ++e) d = fmaf(q[e] - m, q[e] - m, d);
    d += __shfl_xor(d, 1, 64);
    d += __shfl_xor(d, 2, 64);
    if (out && (tid & 3) == 0) *(float2*)(p.st_out + (size_t)om * 128 + blockIdx.x * 2) = float2{m, d};
  }
}

template <typename T, int FM>
static int enc_rows_launch(const EncRowsArgs& a, int epi, hipStream_t s) {
  // as many waves as share the units of 64 k evenly; at least FM (4 threads an output row)
  const int units = a.K / 64, per = (units + enc_waves(FM) - 1) / enc_waves(FM);
  const dim3 grid(a.N / 16, (a.M + FM * 16 - 1) / (FM * 16)), block(max((units + per - 1) / per, FM) * 64);
#define ENC_ROWS(LNA, E) enc_rows_kernel<T, FM, LNA, E><<<grid, block, 0, s>>>(a)
  if (epi == EPI_RESID) ENC_ROWS(false, EPI_RESID);
  else if (epi == EPI_GELU && a.st) ENC_ROWS(true, EPI_GELU);
  else if (epi == EPI_BIAS && a.st) ENC_ROWS(true, EPI_BIAS);
  else if (epi == EPI_BIAS) ENC_ROWS(false, EPI_BIAS);
  else return (int)hipErrorInvalidValue;
#undef ENC_ROWS
  return (int)hipGetLastError();
}

template <typename T>
static int enc_rows_rows(const EncRowsArgs& a, int epi, hipStream_t s) {
  // the smallest row blocks whose workgroups still fit the CUs in one round: a CU's share of A is what it waits for
  // (K = 3072, 32 rows: 8.5 us in two blocks, 10.9 in one; 144 and 192 strips in two blocks 6.6 and 7.3 vs 5.9 and 6.9)
  const int strips = a.N / 16, blocks = (a.M + 15) / 16;
  if (strips * blocks <= 256) return enc_rows_launch<T, 1>(a, epi, s);
  return a.M <= 32 || strips * ((blocks + 1) / 2) <= 256 ? enc_rows_launch<T, 2>(a, epi, s) : enc_rows_launch<T, 4>(a, epi, s);
}

template <typename T, int D>
static int enc_attn_rows(const EncRowsArgs& a, hipStream_t s) {
  const dim3 grid(a.N / 16, (a.M + 15) / 16);
  if (a.M > 32) enc_rows_kernel<T, 1, false, EPI_RESID, D, 64, 6><<<grid, a.K, 0, s>>>(a);
  else if (a.K <= 768) enc_rows_kernel<T, 1, false, EPI_RESID, D, 32, 12><<<grid, a.K, 0, s>>>(a);  // (a wave a unit)
  else enc_rows_kernel<T, 1, false, EPI_RESID, D, 32, 16><<<grid, a.K, 0, s>>>(a);
  return (int)hipGetLastError();
}

// epi BIAS / GELU (st: the norm of A's rows, over K columns; GELU only with it) / RESID (st: the norm of resid's rows,
// over N columns; st_out is written). 1 <= M <= 64, K % 64 == 0, N % 16 == 0, a normed width of at most 1024; bf16 or fp16 throughout.
DA_EXPORT int da_enc_rows(const void* A, int lda, const void* W, void* C, int ldc, const void* bias, const void* resid,
                         int ldr, int M, int N, int K, int epi, const float* st, const void* g, const void* b, float eps,
                         float* st_out, int f16, void* stream) {
  const int width = epi == EPI_RESID ? N : K;
  if (M < 1 || M > 64 || K < 64 || K % 64 || N < 16 || N % 16 || lda % 8 || ldc % 4 || (st && (!g || !b || width > 1024 || width % 16)))
    return (int)hipErrorInvalidValue;
  if (epi == EPI_RESID && (!resid || ldr % 4 || !st_out || N > 1024)) return (int)hipErrorInvalidValue;
  if (2ll * ((M - 1) * (long long)lda + K) > 0x7ffff000ll || 32ll * K > 0x7ffff000ll) return (int)hipErrorInvalidValue;  // (32-bit offsets)
  EncRowsArgs a{(const bf16_t*)A, (const bf16_t*)W, (const bf16_t*)bias, (const bf16_t*)resid, (bf16_t*)C, st,
                (const bf16_t*)g, (const bf16_t*)b, st_out, M, N, K, lda, ldc, ldr, width / 16, eps};
  hipStream_t s = (hipStream_t)stream;
  return f16 ? enc_rows_rows<F16T>(a, epi, s) : enc_rows_rows<BF16T>(a, epi, s);
}

// RESID with A the attention of K / D heads of D (64, and 32 in bf16) over the one text of rows cu[0] .. cu[1] - 1: qkv holds q, k and v, K
// columns each. M <= 32, K <= 1024 or M <= 64, K <= 384 (LDS); the rest as above.
DA_EXPORT int da_enc_attn_rows(const void* qkv, int lda, const void* W, void* C, int ldc, const void* bias, const void* resid, int ldr,
                              int M, int N, int K, int D, const int* cu, float c, const float* st, const void* g,
                              const void* b, float eps, float* st_out, int f16, void* stream) {
  if (M < 1 || M > (K > 384 ? 32 : 64) || K < 64 || K % 64 || K > 1024 || N < 16 || N % 16 || N > 1024 || lda % 8 || lda < 3 * K || ldc % 4 || ldr % 4 ||
      lda > (1 << 22) || (D != 64 && (D != 32 || f16)) || !cu || !resid || !st_out || (st && (!g || !b)))
    return (int)hipErrorInvalidValue;
  EncRowsArgs a{(const bf16_t*)qkv, (const bf16_t*)W, (const bf16_t*)bias, (const bf16_t*)resid, (bf16_t*)C, st,
                (const bf16_t*)g, (const bf16_t*)b, st_out, M, N, K, lda, ldc, ldr, N / 16, eps, cu, c};
  hipStream_t s = (hipStream_t)stream;
  if (D == 32) return enc_attn_rows<BF16T, 32>(a, s);
  return f16 ? enc_attn_rows<F16T, 64>(a, s) : enc_attn_rows<BF16T, 64>(a, s);
}
