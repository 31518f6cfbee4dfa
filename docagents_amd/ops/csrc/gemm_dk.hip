// Decode GEMM for 1 <= M <= 64 rows in one launch (gemm_dk), and products of more rows in blocks of 32 or 64 (da_gemm_dk_rows).
//
//   C[M, N'] = epi( rownorm(A)[M, K] . W[N, K]^T )
//
// A workgroup owns 16 FN columns of the result and all of K: its waves take K-steps of 64 in turn (wave w: w, w + NW, ...),
// each with a ring of stages of its own, and their sums meet in LDS once, so the epilogue (bias / residual / gated) runs in
// the same launch. What bounds it is HBM: W is read once, and beside it the L2s' share of A, 16 FM rows for 16 FN of W.
//
// A stage is the rows' 128 B of a K-step, brought by LDS-DMA in whole lines (operands straight in MFMA layout are 64-B
// requests, which cost a CU as much as 128). Nothing in a ring is shared: a wave waits for its own transfers only, reads
// the fragments, sends the next transfers into the same slot and multiplies, and there is no barrier before the sums.
// Two workgroups of <= 80 KB fit a CU; more stages in fewer of them are slower (8192 x 4096, 16 rows: 12.2 us at two
// stages of four waves, 12.4 at three, 12.9 at six).
//
// Columns of a tile: the fewest times 16 for one round of 256 workgroups, up to 64 (from 16385 columns on, in rounds of
// two workgroups a CU). us at 4 / 16 / 32 rows, before (register-staged tiles with a barrier every 256 of K, and streaming
// tiles of all waves above 8192 columns) -> now:
//   3072 x 3072  7.2 / 8.1 / 8.6 -> 5.7 / 6.7 / 8.5      4096 x 4096   9.2 / 9.6 / 10.7 -> 7.7 / 8.5 / 10.5
//   3072 x 8192  12.6 / 14.9 / 17.5 -> 10.8 / 12.3 / 15.7  4096 x 14336 22.8 / 25.2 / 32.7 -> 20.1 / 23.0 / 29.5
//   6144 x 4096  11.5 / 12.1 / 15.7 -> 10.6 / 11.2 / 13.4  9216 x 3072  14.0 / 15.2 / 16.8 -> 11.3 / 12.2 / 14.7
//   5184 x 4096  13.4 / 15.8 / 18.1 -> 9.7 / 10.9 / 13.1   12608 x 4096 19.4 / 19.8 / 21.3 -> 17.9 / 18.5 / 20.7
//   16384 x 3072 19.3 / 19.2 / 19.7 -> 17.7 / 18.1 / 19.8  28672 x 4096 40.1 / 40.4 / 40.6 -> 38.5 / 39.2 / 41.4
//
// Where K is a multiple of 2048, the tiles of an XCD begin at K-steps of their own: all at the same columns of
// rows a multiple of 4 KB apart, they ask the same few channels at a time (8192 x 4096, 4 rows: 13.7 us without, 12.1 with;
// 4096 x 14336: 21.8 and 20.1; 2 rows, K = 2048: 4096 columns 6.4 and 5.4, 28672 22.4 and 20.0, 128256 83.5 and 74.7, of up to 2048
// columns 1 % longer, which begin together; K = 3072 gains nothing).
//
// Deferred RMSNorm: the decode layer's norms ride here instead of in launches of their own. The producer of the residual
// stream (EPI_RESID) writes, next to x, per-(workgroup, row) sums of squares of its bf16 output slice (ssq_out
// [parts][64]); the consumer reads x itself as A and scales its sums by rsqrt(sum_parts / norm_k + eps) (the RMSNorm gains
// are folded into W at load, models/llama.py).
#include "gemm.h"

typedef __attribute__((address_space(3))) void* lds_ptr_t;

struct DkArgs {
  const bf16_t* A; const bf16_t* W; bf16_t* C;
  const bf16_t* bias; const bf16_t* resid;
  const float* ssq_in;  // nullable: [ssq_parts][64] partial sums of squares of A's rows
  float* ssq_out;       // EPI_RESID (nullable): [N / ssq_bn][64] sums of squares of the output rows, by ssq_bn columns
  float* ws;            // SPLIT: the workgroups' sums, and a counter per tile that is 0 between launches
  int* cnt;
  int splits, ssq_bn;
  int M, N, K, lda, ldc, ldr, ssq_parts, norm_k;
  float eps;
  int relu;  // EPI_SWIGLU: the gate's activation is relu, not silu
  RopeArgs rope;  // EPI_ROPE
};

// The values of four neighbours, as two words.
template <typename T> __device__ __forceinline__ f32x4_t unpack4(const u32x2_t& u) {
  return f32x4_t{T::to_f((bf16_t)(u[0] & 0xffff)), T::to_f((bf16_t)(u[0] >> 16)), T::to_f((bf16_t)(u[1] & 0xffff)), T::to_f((bf16_t)(u[1] >> 16))};
}

// ST stages of a wave's ring, each BM rows of A and BN of W; row r's 16-B chunk c at slot c ^ (r >> 1 & 7), so that the 16
// rows of a fragment read land on all banks
// SPLIT: K by `splits` workgroups as well. Each leaves its sums and counts; the last to come, which nobody waits for, adds them up
// in order and has the epilogue: 2.5 us that a long K repays, where few columns leave CUs idle or workgroups read all of A for few
// columns each. The sums go past the XCDs' L2s (sc1) to where all of them see them. us, whole -> split:
//   2 / 8 / 16 / 32 rows, tiles of 16 columns by 4: 320 x 8192 8.1 / 9.1 / 10.9 / 14.2 -> 6.2 / 6.6 / 6.9 / 7.7, 128 x 4096 5.1 / 5.9 /
//     6.7 / 8.5 -> 5.1 / 5.2 / 5.4 / 6.0, 768 x 3072 at 24 / 32 7.2 / 7.7 -> 6.3 / 6.5; of 32 by 4: 1536 x 6144 at 2 / 8 / 16 / 32
//     7.6 / 8.6 / 9.7 / 13.0 -> 7.8 / 8.1 / 8.4 / 9.2, 2048 x 8192 10.2 / 9.8 / 11.3 / 14.8 -> 10.0 / 10.0 / 10.1 / 10.6
//   32 / 24 / 17 rows, tiles of 64 columns by 4 or 5: 4096 x 14336 29.6 / 27.3 / 26.6 -> 25.9 / 25.1 / 25.5, 3072 x 8192 16.2 / 14.9 /
//     15.3 -> 15.3 / 15.1 / 14.9; not 4096 x 8192 (16.8 -> 17.9), 4096 x 4096 (11.0 -> 11.0) or 512 x 2048 (5.8 -> 5.8), nor 33 rows
//     and more, whose streaming tiles share A (4096 x 14336, 64: 28.1, 31.7).
// ROWS: more than one block of BM rows (gridDim.y of them; W's lines are worth a place in the caches then). The blocks of a column
// tile are neighbours on one XCD.
template <int FM, int FN, int NW, int ST, int EPI, typename T, bool ROWS, bool SPLIT>
__global__ void __launch_bounds__(64 * NW)
gemm_dk_kernel(DkArgs p) {
  constexpr int BM = 16 * FM, BN = 16 * FN, A_BYTES = BM * 128, STAGE = A_BYTES + BN * 128;
  constexpr int PA = BM / 8, PW = BN / 8, P = PA + PW;  // LDS-DMA instructions of a stage
  constexpr int SLD = BN + 4, RED = NW * BM * SLD * 4;
  constexpr int RING = NW * ST * STAGE, SUMS = RED + NW * 64 * 4;
  static_assert(P * ST < 64 && PA <= 8 && PW <= 16, "tile");
  __shared__ __attribute__((aligned(16))) char smem[RING > SUMS ? RING : SUMS];
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int fr = lane & 15, fg = lane >> 4;
  int tile = SPLIT ? blockIdx.x / p.splits : blockIdx.x;
  const int first = SPLIT ? blockIdx.x % p.splits * NW + w : w, every = SPLIT ? NW * p.splits : NW;  // this wave's K-steps
  if constexpr (ROWS) {
    const int t = xcd_remap(blockIdx.y * gridDim.x + blockIdx.x, gridDim.x * gridDim.y), m0 = t % (int)gridDim.y * BM;
    tile = t / (int)gridDim.y;
    p.M -= m0;
    p.A += (size_t)m0 * p.lda;
    p.C += (size_t)m0 * p.ldc;
    if (EPI == EPI_RESID) p.resid += (size_t)m0 * p.ldr;
  }
  const int n0 = tile * BN, nk = p.K / 64;

  // deferred norm: thread = (part, 4 rows), 8 parts each on their way before the ring's first stages
  constexpr int RQ = FM == 3 ? 16 : BM / 4, PL = 64 * NW / RQ;  // row quads (a power of two), parts at a time
  f32x4_t sq[8];
  if (p.ssq_in)
#pragma unroll
    for (int j = 0; j < 8; ++j)
      sq[j] = *(const f32x4_t*)(p.ssq_in + (size_t)min(tid / RQ + j * PL, p.ssq_parts - 1) * 64 + tid % RQ * 4);

  // rotation: this thread's pieces of the result (their heads, positions and slots), cos and sin on their way before the ring too
  constexpr int BNO = EPI == EPI_SWIGLU ? BN / 2 : BN;  // output columns of the tile
  constexpr int CPR = BNO / 4;                          // 4-column pieces of a row
  constexpr int RI = EPI == EPI_ROPE ? (BM * CPR + 64 * NW - 1) / (64 * NW) : 1;
  [[maybe_unused]] int rpos[RI], rslot[RI];
  [[maybe_unused]] f32x4_t rcs[RI];
  if constexpr (EPI == EPI_ROPE) {
#pragma unroll
    for (int i = 0; i < RI; ++i) {
      const int m = min((tid + i * 64 * NW) / CPR, p.M - 1);
      rpos[i] = p.rope.pos[m];
      rslot[i] = p.rope.slot[m];
    }
#pragma unroll
    for (int i = 0; i < RI; ++i)  // (columns of v: not used)
      rcs[i] = *(const f32x4_t*)(p.rope.cs + (size_t)min(max(rpos[i], 0), p.rope.max_seq - 1) * p.rope.D +
                                 (n0 + (tid + i * 64 * NW) % CPR * 4) % p.rope.D);
  }

  unsigned ao[8], wo[16];  // rows past the operands': past the resource's end, which reads as zero
#pragma unroll
  for (int j = 0; j < PA; ++j) {
    const int r = 8 * j + (lane >> 3), c = (lane & 7) ^ ((r >> 1) & 7);
    ao[j] = r < p.M ? (unsigned)r * (unsigned)(p.lda * 2) + c * 16 : 0x7ffffff0u;
  }
#pragma unroll
  for (int j = 0; j < PW; ++j) {
    const int r = 8 * j + (lane >> 3), c = (lane & 7) ^ ((r >> 1) & 7);
    wo[j] = n0 + r < p.N ? (unsigned)r * (unsigned)(p.K * 2) + c * 16 : 0x7ffffff0u;
  }
  const char* Wt = (const char*)p.W + (size_t)n0 * p.K * 2;
  char* ring = smem + w * ST * STAGE;
  const int rot = nk % 32 == 0 && (nk > 32 || p.N > 2048) ? (tile >> 3) * 4 % nk : 0;  // the K-step that this tile begins with
  const int mine = max(nk - first + every - 1, 0) / every;              // of this wave
  auto issue = [&](int i, int slot) __attribute__((always_inline)) {  // (past the wave's last: no transfer)
    int step = first + i * every + rot;
    step = step >= nk ? step - nk : step;
    const int n = i < mine ? 0x7fffff00 : 0;
    const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc((void*)p.A, (short)0, n, 0x00020000);
    const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc((void*)Wt, (short)0, n, 0x00020000);
    char* base = ring + slot * STAGE;
#pragma unroll
    for (int j = 0; j < PW; ++j)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, (lds_ptr_t)(base + A_BYTES + j * 1024), 16, wo[j & 15], step * 128, 0, ROWS ? 0 : 2);
#pragma unroll
    for (int j = 0; j < PA; ++j)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (lds_ptr_t)(base + j * 1024), 16, ao[j & 7], step * 128, 0, 0);
  };
#pragma unroll
  for (int i = 0; i < ST; ++i) issue(i, i);

  f32x4_t ss{0.f, 0.f, 0.f, 0.f};  // lanes < RQ: this wave's sums of rows 4 lane .. + 3
  if (p.ssq_in) {
#pragma unroll
    for (int j = 0; j < 8; ++j) ss += tid / RQ + j * PL < p.ssq_parts ? sq[j] : f32x4_t{0.f, 0.f, 0.f, 0.f};
    for (int q0 = tid / RQ + 8 * PL; q0 < p.ssq_parts; q0 += 4 * PL) {
#pragma unroll
      for (int j = 0; j < 4; ++j) sq[j] = *(const f32x4_t*)(p.ssq_in + (size_t)min(q0 + j * PL, p.ssq_parts - 1) * 64 + tid % RQ * 4);
#pragma unroll
      for (int j = 0; j < 4; ++j) ss += q0 + j * PL < p.ssq_parts ? sq[j] : f32x4_t{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int o = RQ; o < 64; o <<= 1)
#pragma unroll
      for (int e = 0; e < 4; ++e) ss[e] += __shfl_xor(ss[e], o, 64);
  }

  f32x4_t acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const int sw = (fr >> 1) & 7;
  const int co[2] = {(fg ^ sw) << 4, ((4 + fg) ^ sw) << 4};
  int slot = 0;
#pragma unroll 1
  for (int i = 0; i < mine; ++i) {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(P * (ST - 1)) : "memory");  // stage i is in
    __builtin_amdgcn_sched_barrier(0);
    bf16x8_t af[2][FM], wf[2][FN];
    const char* s = ring + slot * STAGE + fr * 128;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int j = 0; j < FN; ++j) wf[h][j] = *(const bf16x8_t*)(s + A_BYTES + j * 2048 + co[h]);
#pragma unroll
      for (int q = 0; q < FM; ++q) af[h][q] = *(const bf16x8_t*)(s + q * 2048 + co[h]);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // and read: its slot is free
    __builtin_amdgcn_sched_barrier(0);
    issue(i + ST, slot);
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int q = 0; q < FM; ++q)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[q][j] = T::mma16(wf[h][j], af[h][q], acc[q][j]);  // (W first: a lane has 4 columns of a row)
    slot = slot + 1 == ST ? 0 : slot + 1;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (transfers past the end write zeros)
  __syncthreads();
  // ---- the waves' sums, added in wave order (the rings are free now) ----
  float (*red)[BM][SLD] = (float (*)[BM][SLD])smem;
  float* sums = (float*)(smem + RED);
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) *(f32x4_t*)&red[w][16 * i + fr][16 * j + 4 * fg] = acc[i][j];
  if (p.ssq_in && lane < RQ) *(f32x4_t*)(sums + w * 64 + lane * 4) = ss;
  __syncthreads();

  if constexpr (SPLIT) {  // (a thread's pieces here are its pieces below)
    static_assert(EPI != EPI_SWIGLU && !ROWS, "split");
    constexpr int IT = (BM * CPR + 64 * NW - 1) / (64 * NW);  // (threads past the last piece: that one again)
    constexpr unsigned TB = IT * 64 * NW * 16;
    f32x4_t v[IT];
#pragma unroll
    for (int i = 0; i < IT; ++i) {
      const int t = min(tid + i * 64 * NW, BM * CPR - 1);
      v[i] = *(const f32x4_t*)&red[0][t / CPR][t % CPR * 4];
#pragma unroll
      for (int x = 1; x < NW; ++x) v[i] += *(const f32x4_t*)&red[x][t / CPR][t % CPR * 4];
    }
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc((void*)p.ws, (short)0, gridDim.x * TB, 0x00020000);
    const unsigned at = tid * 16u;
#pragma unroll
    for (int i = 0; i < IT; ++i)
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, v[i]), rs, at + i * 1024 * NW, blockIdx.x * TB, 16);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's stores are done; then every wave's
    __syncthreads();
    int* last = (int*)(smem + RED);
    if (tid == 0) *last = __hip_atomic_fetch_add(p.cnt + tile, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == p.splits - 1;
    __syncthreads();
    if (!*(volatile int*)last) return;
    if (tid == 0) __hip_atomic_store(p.cnt + tile, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
    for (int i = 0; i < IT; ++i) v[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    for (int q0 = 0; q0 < p.splits; q0 += 4) {
      u32x4_t x[4][IT];
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int i = 0; i < IT; ++i)
          x[q][i] = __builtin_amdgcn_raw_buffer_load_b128(rs, at + i * 1024 * NW, (tile * p.splits + min(q0 + q, p.splits - 1)) * TB, 16);
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (q0 + q < p.splits)
#pragma unroll
          for (int i = 0; i < IT; ++i) v[i] += __builtin_bit_cast(f32x4_t, x[q][i]);
    }
#pragma unroll
    for (int i = 0; i < IT; ++i) {
      const int t = tid + i * 64 * NW;
      if (t < BM * CPR) *(f32x4_t*)&red[0][t / CPR][t % CPR * 4] = v[i];
    }
  }
  static_assert(EPI != EPI_RESID || ROWS || (CPR & (CPR - 1)) == 0, "a row's pieces meet by lane exchange");
  if constexpr (EPI == EPI_ROPE) {  // rotated as the kernel behind a product does it (the same bits): the rounded values in fp32, and rounded again
    const RopeArgs& R = p.rope;
    const int qw = R.H * R.D, kw = R.Hkv * R.D;
#pragma unroll
    for (int i = 0; i < RI; ++i) {
      const int t = tid + i * 64 * NW, m = t / CPR, c = t % CPR * 4, gn = n0 + c;
      if (t >= BM * CPR || m >= p.M || gn >= p.N) continue;
      float inv = 1.f;
      if (p.ssq_in) {
        float v = 0.f;
#pragma unroll
        for (int x = 0; x < NW; ++x) v += sums[x * 64 + m];
        inv = rsqrtf(v / p.norm_k + p.eps);
      }
      f32x4_t v = *(const f32x4_t*)&red[0][m][c];
#pragma unroll
      for (int x = 1; x < NW; ++x) v += *(const f32x4_t*)&red[x][m][c];
      u32x2_t o{T::pack2(v[0] * inv, v[1] * inv), T::pack2(v[2] * inv, v[3] * inv)};
      const int kind = gn < qw ? 0 : gn < qw + kw ? 1 : 2, rel = gn - (kind == 0 ? 0 : kind == 1 ? qw : qw + kw);
      if (kind < 2) {
        const f32x4_t x = unpack4<T>(o), cs = rcs[i];
        o = u32x2_t{T::pack2(fmaf(x[0], cs[0], -(x[1] * cs[1])), fmaf(x[1], cs[0], x[0] * cs[1])),
                    T::pack2(fmaf(x[2], cs[2], -(x[3] * cs[3])), fmaf(x[3], cs[2], x[2] * cs[3]))};
      }
      if (kind > 0) {
        DA_ASSERT(rpos[i] >= 0 && rpos[i] < R.max_seq && rslot[i] >= 0);
        bf16_t* cache = kind == 1 ? R.kc : R.vc;
        *(u32x2_t*)(cache + (((size_t)rslot[i] * R.Hkv + rel / R.D) * R.max_seq + rpos[i]) * R.D + rel % R.D) = o;
        if (!R.kv_out) continue;
      }
      *(u32x2_t*)(p.C + (size_t)m * p.ldc + gn) = o;
    }
    return;
  }
#pragma unroll 1
  for (int t = tid; t < BM * CPR; t += 64 * NW) {
    const int m = t / CPR, c = t % CPR * 4;
    float inv = 1.f;
    if (p.ssq_in) {
      float v = 0.f;
#pragma unroll
      for (int x = 0; x < NW; ++x) v += sums[x * 64 + m];
      inv = rsqrtf(v / p.norm_k + p.eps);
    }
    auto total = [&](int col) {
      f32x4_t v = *(const f32x4_t*)&red[0][m][col];
#pragma unroll
      for (int x = 1; x < (SPLIT ? 1 : NW); ++x) v += *(const f32x4_t*)&red[x][m][col];
      return v;
    };
    auto bias4 = [&](int col) {  // columns of the product
      return p.bias ? unpack4<T>(*(const u32x2_t*)(p.bias + col)) : f32x4_t{0.f, 0.f, 0.f, 0.f};
    };
    const int gn = EPI == EPI_SWIGLU ? n0 / 2 + c : n0 + c;
    const bool ok = m < p.M && gn < (EPI == EPI_SWIGLU ? p.N / 2 : p.N);
    f32x4_t v{0.f, 0.f, 0.f, 0.f};
    if constexpr (EPI == EPI_SWIGLU) {
      const int gc = (c >> 4) * 32 + (c & 15);
      if (ok) {
        const f32x4_t g = total(gc), u = total(gc + 16), bg = bias4(n0 + gc), bu = bias4(n0 + gc + 16);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = gate_act(fmaf(g[e], inv, bg[e]), p.relu) * fmaf(u[e], inv, bu[e]);
      }
    } else if (ok) {
      const f32x4_t x = total(c), b = bias4(gn);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = fmaf(x[e], inv, b[e]);
      if constexpr (EPI == EPI_GELU) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = gelu_erf(v[e]);
      }
      if constexpr (EPI == EPI_RESID) v += unpack4<T>(*(const u32x2_t*)(p.resid + (size_t)m * p.ldr + gn));
    }
    const u32x2_t o{T::pack2(v[0], v[1]), T::pack2(v[2], v[3])};
    if (ok) *(u32x2_t*)(p.C + (size_t)m * p.ldc + gn) = o;
    if constexpr (EPI == EPI_RESID && !ROWS) {
      if (p.ssq_out) {  // sum of squares of the bf16 values the stream now holds
        const f32x4_t x = unpack4<T>(o);
        float q = (x[0] * x[0] + x[1] * x[1]) + (x[2] * x[2] + x[3] * x[3]);
        if (!ok) q = 0.f;
#pragma unroll
        for (int x = 1; x < CPR; x <<= 1)
          if (x < p.ssq_bn / 4) q += __shfl_xor(q, x, 64);
        if (c % p.ssq_bn == 0 && m < p.M && gn < p.N) p.ssq_out[(size_t)(gn / p.ssq_bn) * 64 + m] = q;
      }
    }
  }
}

// 16-column groups of a tile (a residual's row sums meet by lane exchange: a power of two; gated columns come in 32s)
static int dk_fn(int N, int epi) {
  const int fn = min(4, (N / 16 + 255) / 256);
  if (epi == EPI_SWIGLU) return fn <= 2 ? 2 : 4;
  return epi == EPI_RESID && fn == 3 ? 4 : fn;
}

template <int FM, int FN, int EPI>
static int dk_launch3(const DkArgs& a, hipStream_t s) {
  // four waves, as many stages as leave a CU room for two workgroups; at least two, of which one is read
  constexpr int STAGE = (FM + FN) * 2048, FIT = 81920 / (4 * STAGE), ST = FIT < 2 ? 2 : FIT > 4 ? 4 : FIT;
  gemm_dk_kernel<FM, FN, 4, ST, EPI, BF16T, false, false><<<(a.N + 16 * FN - 1) / (16 * FN), 256, 0, s>>>(a);
  return (int)hipGetLastError();
}

template <int FM, int FN>
static int dk_split(const DkArgs& a, int epi, hipStream_t s) {
  constexpr int STAGE = (FM + FN) * 2048, FIT = 81920 / (4 * STAGE), ST = FIT < 2 ? 2 : FIT > 4 ? 4 : FIT;
  const int blocks = (a.N + 16 * FN - 1) / (16 * FN) * a.splits;
  if (epi == EPI_RESID) gemm_dk_kernel<FM, FN, 4, ST, EPI_RESID, BF16T, false, true><<<blocks, 256, 0, s>>>(a);
  else if (epi == EPI_NONE || epi == EPI_BIAS) gemm_dk_kernel<FM, FN, 4, ST, EPI_NONE, BF16T, false, true><<<blocks, 256, 0, s>>>(a);
  else return (int)hipErrorInvalidValue;
  return (int)hipGetLastError();
}

template <int FM>
static int dk_launch1(const DkArgs& a, int epi, hipStream_t s) {
  const int fn = dk_fn(a.N, epi);
  switch (epi) {
    case EPI_NONE: case EPI_BIAS:
      return fn == 1   ? dk_launch3<FM, 1, EPI_NONE>(a, s)
             : fn == 2 ? dk_launch3<FM, 2, EPI_NONE>(a, s)
             : fn == 3 ? dk_launch3<FM, 3, EPI_NONE>(a, s) : dk_launch3<FM, 4, EPI_NONE>(a, s);
    case EPI_RESID:
      return fn == 1   ? dk_launch3<FM, 1, EPI_RESID>(a, s)
             : fn == 2 ? dk_launch3<FM, 2, EPI_RESID>(a, s) : dk_launch3<FM, 4, EPI_RESID>(a, s);
    case EPI_SWIGLU: return fn == 2 ? dk_launch3<FM, 2, EPI_SWIGLU>(a, s) : dk_launch3<FM, 4, EPI_SWIGLU>(a, s);
    case EPI_ROPE:
      return fn == 1   ? dk_launch3<FM, 1, EPI_ROPE>(a, s)
             : fn == 2 ? dk_launch3<FM, 2, EPI_ROPE>(a, s)
             : fn == 3 ? dk_launch3<FM, 3, EPI_ROPE>(a, s) : dk_launch3<FM, 4, EPI_ROPE>(a, s);
    default: return (int)hipErrorInvalidValue;
  }
}

// Number of ssq parts a RESID launch of width N writes (the consumer's ssq_parts).
DA_EXPORT int da_gemm_dk_parts(int N) {
  const int bn = 16 * dk_fn(N, EPI_RESID);
  return (N + bn - 1) / bn;
}

// epi: EPI_NONE / EPI_BIAS / EPI_RESID / EPI_SWIGLU. ssq_in (nullable): deferred RMSNorm of A's rows
// over ssq_parts parts (norm over norm_k columns, eps); ssq_out (nullable, EPI_RESID only):
// [da_gemm_dk_parts(N)][64] floats. 1 <= M <= 64, K % 64 == 0, N % 16 == 0 (SwiGLU: N % 32 == 0).
// splits > 0 (up to 32 rows, not SwiGLU, no ssq_in): tiles of 16 fn columns (fn 1, 2 or, from 17 rows on, 4), K by as many
// workgroups; ws: da_gemm_dk_ws bytes, cnt: a zero per tile.
DA_EXPORT size_t da_gemm_dk_ws(int N, int fn, int splits) {
  return (size_t)((N + 16 * fn - 1) / (16 * fn)) * splits * (fn == 4 ? 8192 : 4096);
}

DA_EXPORT int da_gemm_dk(const void* A, int lda, const void* W, void* C, int ldc, const void* bias,
                         const void* resid, int ldr, int M, int N, int K, int epi, const float* ssq_in, int ssq_parts,
                         int norm_k, float eps, float* ssq_out, int fn, int splits, void* ws, void* cnt, void* stream) {
  if (M < 1 || M > 64 || K < 64 || K % 64 || N < 16 || N % 16 || lda % 8 || ldc % 8) return (int)hipErrorInvalidValue;
  const int relu = epi == EPI_REGLU;
  if (relu) epi = EPI_SWIGLU;
  if (epi == EPI_SWIGLU && N % 32) return (int)hipErrorInvalidValue;
  if (epi == EPI_RESID && (!resid || ldr % 8)) return (int)hipErrorInvalidValue;
  if (ssq_out && epi != EPI_RESID) return (int)hipErrorInvalidValue;
  if (ssq_in && (ssq_parts < 1 || norm_k < 1 || !(eps > 0.f))) return (int)hipErrorInvalidValue;
  const int ssq_fn = dk_fn(N, epi);
  if (splits < 0 || splits > 64 ||
      (splits && (M > 32 || ssq_in || !ws || !cnt || (fn != 1 && fn != 2 && fn != 4) || (ssq_out && (ssq_fn > fn || N % (16 * ssq_fn))))))
    return (int)hipErrorInvalidValue;
  // a tile's rows within the resource's reach
  if (2ll * ((M - 1) * (long long)lda + K) > 0x7ffff000ll || 32ll * (splits ? fn : ssq_fn) * K > 0x7ffff000ll ||
      (splits && da_gemm_dk_ws(N, fn, splits) > 0x7ffff000u))
    return (int)hipErrorInvalidValue;
  DkArgs a{};
  a.A = (const bf16_t*)A; a.W = (const bf16_t*)W; a.C = (bf16_t*)C;
  a.bias = (const bf16_t*)bias; a.resid = (const bf16_t*)resid;
  a.ssq_in = ssq_in; a.ssq_out = ssq_out;
  a.M = M; a.N = N; a.K = K; a.lda = lda; a.ldc = ldc; a.ldr = ldr;
  a.ssq_parts = ssq_parts; a.norm_k = norm_k; a.eps = eps; a.relu = relu;
  a.ws = (float*)ws; a.cnt = (int*)cnt; a.splits = splits; a.ssq_bn = 16 * ssq_fn;
  hipStream_t s = (hipStream_t)stream;
  if (splits && M <= 16) return fn == 1 ? dk_split<1, 1>(a, epi, s) : fn == 2 ? dk_split<1, 2>(a, epi, s) : (int)hipErrorInvalidValue;
  if (splits) return fn == 1 ? dk_split<2, 1>(a, epi, s) : fn == 2 ? dk_split<2, 2>(a, epi, s) : dk_split<2, 4>(a, epi, s);
  if (M <= 16) return dk_launch1<1>(a, epi, s);
  if (M <= 32) return dk_launch1<2>(a, epi, s);
  if (M <= 48) return dk_launch1<3>(a, epi, s);
  return dk_launch1<4>(a, epi, s);
}

// The QKV projection: rows rotated by their positions (interleaved pairs), k and v to the cache (and, with kv_out, to C too).
// ssq_in as above. A launch behind the product read the result and wrote it again, 2.8 - 5.2 us a layer; here positions, cosines and
// sines of a thread's pieces arrive beside the weights, and the epilogue takes 0.5 - 0.7 us longer (64 x 6144 x 4096 17.3 + 4.8 -> 18.0).
// A step of an 8B at 2 / 11 / 26 / 62 rows 3025 / 3157 / 3831 / 6027 -> 2983 / 3104 / 3791 / 5962 us.
DA_EXPORT int da_gemm_dk_rope(const void* A, int lda, const void* W, void* C, int ldc, int M, int N, int K, const float* ssq_in,
                             int ssq_parts, int norm_k, float eps, const void* pos, const void* slot, const void* cos_sin,
                             void* k_cache, void* v_cache, int H, int Hkv, int D, int max_seq, int kv_out, void* stream) {
  if (M < 1 || M > 64 || K < 64 || K % 64 || N < 16 || N % 16 || lda % 8 || ldc % 8 || D < 8 || D % 8 || N != (H + 2 * Hkv) * D ||
      !pos || !slot || !cos_sin || !k_cache || !v_cache || max_seq < 1 || (ssq_in && (ssq_parts < 1 || norm_k < 1 || !(eps > 0.f))))
    return (int)hipErrorInvalidValue;
  if (2ll * ((M - 1) * (long long)lda + K) > 0x7ffff000ll || 128ll * K > 0x7ffff000ll) return (int)hipErrorInvalidValue;
  DkArgs a{};
  a.A = (const bf16_t*)A; a.W = (const bf16_t*)W; a.C = (bf16_t*)C;
  a.ssq_in = ssq_in; a.ssq_parts = ssq_parts; a.norm_k = norm_k; a.eps = eps;
  a.M = M; a.N = N; a.K = K; a.lda = lda; a.ldc = ldc;
  a.rope = RopeArgs{(const int*)pos, (const int*)slot, (const float*)cos_sin, (bf16_t*)k_cache, (bf16_t*)v_cache, H, Hkv, D, max_seq,
                    kv_out ? 1 : 0};
  hipStream_t s = (hipStream_t)stream;
  if (M <= 16) return dk_launch1<1>(a, EPI_ROPE, s);
  if (M <= 32) return dk_launch1<2>(a, EPI_ROPE, s);
  if (M <= 48) return dk_launch1<3>(a, EPI_ROPE, s);
  return dk_launch1<4>(a, EPI_ROPE, s);
}

template <int FM, int FN, int ST, typename T>
static int dk_rows(const DkArgs& a, int epi, hipStream_t s) {
  const dim3 grid((a.N + 16 * FN - 1) / (16 * FN), (a.M + 16 * FM - 1) / (16 * FM));
#define DK_ROWS(E) gemm_dk_kernel<FM, FN, 4, ST, E, T, true, false><<<grid, 256, 0, s>>>(a)
  switch (epi) {
    case EPI_NONE: case EPI_BIAS: DK_ROWS(EPI_NONE); break;
    case EPI_GELU: DK_ROWS(EPI_GELU); break;
    case EPI_RESID: DK_ROWS(EPI_RESID); break;
    case EPI_SWIGLU:
      if constexpr (FN % 2 == 0 && !T::kF16) {
        DK_ROWS(EPI_SWIGLU);
        break;
      }
      return (int)hipErrorInvalidValue;
    default: return (int)hipErrorInvalidValue;
  }
#undef DK_ROWS
  return (int)hipGetLastError();
}

template <typename T>
static int dk_rows_tile(const DkArgs& a, int epi, int tile, hipStream_t s) {
  switch (tile) {
    case 20: return dk_rows<2, 1, 3, T>(a, epi, s);
    case 21: return dk_rows<2, 2, 2, T>(a, epi, s);
    case 22: return dk_rows<4, 2, 2, T>(a, epi, s);
    case 23: return dk_rows<4, 3, 2, T>(a, epi, s);
    case 24: return dk_rows<4, 4, 2, T>(a, epi, s);
    case 25: return dk_rows<4, 6, 2, T>(a, epi, s);
    default: return (int)hipErrorInvalidValue;
  }
}

// More rows than a block, by tiles of their own (kernels.py, _DK_TILES): 20 = 32x16, 21 = 32x32, 22 = 64x32, 23 = 64x48, 24 = 64x64,
// 25 = 64x96. epi: NONE / BIAS / GELU / RESID, bf16 also SWIGLU / REGLU (N % 32 == 0; not tiles 20 and 23). K % 64 == 0, N % 8 == 0,
// bf16 or fp16 (f16) throughout.
DA_EXPORT int da_gemm_dk_rows(const void* A, int lda, const void* W, void* C, int ldc, const void* bias, const void* resid, int ldr,
                              int M, int N, int K, int epi, int tile, int f16, void* stream) {
  const int relu = epi == EPI_REGLU;
  if (relu) epi = EPI_SWIGLU;
  if (M < 1 || M > 65535 * 32 || K < 64 || K % 64 || N < 8 || N % 8 || lda % 8 || ldc % 4 || (epi == EPI_SWIGLU && N % 32) ||
      (epi == EPI_RESID && (!resid || ldr % 4)))
    return (int)hipErrorInvalidValue;
  if (2ll * (63 * (long long)lda + K) > 0x7ffff000ll || 2ll * 96 * K > 0x7ffff000ll) return (int)hipErrorInvalidValue;
  DkArgs a{};
  a.A = (const bf16_t*)A; a.W = (const bf16_t*)W; a.C = (bf16_t*)C;
  a.bias = (const bf16_t*)bias; a.resid = (const bf16_t*)resid;
  a.M = M; a.N = N; a.K = K; a.lda = lda; a.ldc = ldc; a.ldr = ldr; a.relu = relu;
  return f16 ? dk_rows_tile<F16T>(a, epi, tile, (hipStream_t)stream) : dk_rows_tile<BF16T>(a, epi, tile, (hipStream_t)stream);
}
