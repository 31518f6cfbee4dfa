// bf16 GEMM on gfx950 MFMA with fused epilogues.
//
//   C[M, N] = epi( A[M, K] · W[N, K]^T )       (nn.Linear layout: both operands K-contiguous)
//
// Design (MI355X-first):
//  * v_mfma_f32_16x16x32_bf16, 4 waves per workgroup, each wave owns a (BM/WM)x(BN/WN) sub-tile
//    indexed by fragment repeat (acc[FM][FN]), never by wave position.
//  * BK = 64, double-buffered LDS with register-staged prefetch (issue global loads for tile t+1
//    before the MFMAs of tile t, write them to the other LDS buffer after: Guideline 15 / T14).
//  * LDS rows are 128 B; 16-B chunks XOR-swizzled by ((row>>1)&7) so the 16 rows read by one
//    ds_read_b128 lane group land on 16 distinct slots of the 256-B bank row (conflict-free).
//  * bijective XCD remap + grouped-M tile order so neighbouring tiles share an XCD L2 (T1).
//  * epilogue staged through LDS in fp32, then 16-B coalesced stores with bias / GELU / SwiGLU /
//    residual fused (the reference outsources all of this to OpenAI).
//  * split-K writes fp32 partials; gemm_splitk_reduce applies the same epilogue.
#include "gemm.h"

#include <type_traits>

template <int BM, int BN, int WM, int WN, int EPI, int PF = 1>
__global__ void __launch_bounds__(256)
gemm_bf16_kernel(GemmArgs p) {
  // PF = k-tiles in flight in registers. PF = 1: the classic register-staged double buffer (one
  // tile ahead). Decode-sized tiles (M <= 64) stream weights and are latency-bound at PF = 1 —
  // one 16-KB W tile per workgroup in flight, ~6 dependent HBM round trips per split — so they
  // keep PF tiles (up to 72 KB per workgroup) requested ahead of the MFMAs (Little's law).
  // (Weight fragments loaded straight into the MFMA B registers, skipping LDS, lost on every arm
  // measured: half-line requests, profiles/r3/rejected_r3.txt.)
  constexpr int BK = 64;
  constexpr int TM = BM / WM, TN = BN / WN;
  constexpr int FM = TM / 16, FN = TN / 16;
  constexpr int A_BYTES = BM * BK * 2, B_BYTES = BN * BK * 2;
  constexpr int LA = BM * 8 / 256, LB = BN * 8 / 256;  // 16-B loads per thread per tile
  static_assert(WM * WN == 4, "4 waves");
  static_assert(LA >= 1 && LB >= 1, "tile too small");
  constexpr int STAGE_FLOATS = 4 * TM * (TN + 4);
  constexpr int LDS_MAIN = 2 * (A_BYTES + B_BYTES);
  constexpr int LDS_BYTES = LDS_MAIN > STAGE_FLOATS * 4 ? LDS_MAIN : STAGE_FLOATS * 4;
  __shared__ __attribute__((aligned(16))) char smem[LDS_BYTES];

  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int wm = wid / WN, wn = wid % WN;

  // ---- tile scheduling: XCD remap, then grouped-M ordering ----
  const int ntm = (p.M + BM - 1) / BM, ntn = (p.N + BN - 1) / BN;
  const int nwg = ntm * ntn;
  const int t = xcd_remap(blockIdx.x, nwg);
  constexpr int GROUP = 8;
  const int gid = t / (GROUP * ntn);
  const int first_m = gid * GROUP;
  const int gsz = min(ntm - first_m, GROUP);
  const int tin = t % (GROUP * ntn);
  const int tm = first_m + tin % gsz, tn = tin / gsz;
  const int m0 = tm * BM, n0 = tn * BN;

  const int kbeg = blockIdx.z * p.k_per_split;
  const int nk = p.k_per_split / BK;

  // ---- global -> register staging (PF slots) ----
  u32x4_t ra[PF][LA], rb[PF][LB];
  const int fr = lane & 15, fg = lane >> 4;
  // Rows past M / N are clamped, not branched around: they only feed accumulators whose outputs
  // are never stored, and branch-free loads keep the compiler's vmcnt waits counted (a load
  // under a divergent branch makes every later wait a full vmcnt(0) drain).
  auto gload = [&](u32x4_t (&xa)[LA], u32x4_t (&xb)[LB], int kt) {
    const int k0 = kbeg + kt * BK;
#pragma unroll
    for (int i = 0; i < LA; ++i) {
      const int idx = tid + 256 * i, r = idx >> 3, c = idx & 7;
      xa[i] = *(const u32x4_t*)(p.A + (size_t)min(m0 + r, p.M - 1) * p.lda + k0 + c * 8);
    }
#pragma unroll
    for (int i = 0; i < LB; ++i) {
      const int idx = tid + 256 * i, r = idx >> 3, c = idx & 7;
      xb[i] = *(const u32x4_t*)(p.W + (size_t)min(n0 + r, p.N - 1) * p.K + k0 + c * 8);
    }
  };
  auto lstore = [&](const u32x4_t (&xa)[LA], const u32x4_t (&xb)[LB], int buf) {
    char* sa = smem + buf * (A_BYTES + B_BYTES);
    char* sb = sa + A_BYTES;
#pragma unroll
    for (int i = 0; i < LA; ++i) {
      const int idx = tid + 256 * i, r = idx >> 3, c = idx & 7;
      *(u32x4_t*)(sa + r * 128 + ((c ^ ((r >> 1) & 7)) << 4)) = xa[i];
    }
#pragma unroll
    for (int i = 0; i < LB; ++i) {
      const int idx = tid + 256 * i, r = idx >> 3, c = idx & 7;
      *(u32x4_t*)(sb + r * 128 + ((c ^ ((r >> 1) & 7)) << 4)) = xb[i];
    }
  };

  f32x4_t acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  // Loads are issued unconditionally (tile index clamped to nk - 1: the redundant tail loads hit
  // L2) so every vmcnt wait below stays counted; compute / LDS stores sit under uniform branches.
  const int kl = nk > 0 ? nk - 1 : 0;
#pragma unroll
  for (int u = 0; u < PF; ++u) {
    gload(ra[u], rb[u], min(u, kl));
    asm volatile("" ::: "memory");  // keep issue order = tile order (counted waits stay short)
  }
  if (nk > 0) lstore(ra[0], rb[0], 0);
  __syncthreads();

  for (int kt0 = 0; kt0 < nk; kt0 += PF) {
#pragma unroll
    for (int u = 0; u < PF; ++u) {
      const int kt = kt0 + u;
      const int cur = kt & 1;
      // slot u held tile kt, already copied to LDS: refill it PF tiles ahead
      if (PF > 1 || kt + 1 < nk) gload(ra[u], rb[u], min(kt + PF, kl));
      if (kt < nk) {
        const char* sa = smem + cur * (A_BYTES + B_BYTES);
        const char* sb = sa + A_BYTES;
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
          const int c = kk * 4 + fg;
          bf16x8_t af[FM], bfr[FN];
#pragma unroll
          for (int i = 0; i < FM; ++i) {
            const int r = wm * TM + i * 16 + fr;
            af[i] = *(const bf16x8_t*)(sa + r * 128 + ((c ^ ((r >> 1) & 7)) << 4));
          }
#pragma unroll
          for (int j = 0; j < FN; ++j) {
            const int r = wn * TN + j * 16 + fr;
            bfr[j] = *(const bf16x8_t*)(sb + r * 128 + ((c ^ ((r >> 1) & 7)) << 4));
          }
#pragma unroll
          for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j) acc[i][j] = mfma16(af[i], bfr[j], acc[i][j]);
        }
      }
      if (kt >= nk) continue;
      if (kt + 1 < nk) lstore(ra[(u + 1) % PF], rb[(u + 1) % PF], cur ^ 1);
      // LDS writes visible + buffer reads done; a raw barrier, NOT __syncthreads(): its fence
      // drains vmcnt and would cancel the PF - 1 tiles still in flight
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
    }
  }

  // ---- epilogue: stage fp32 tile of this wave in LDS, then coalesced 16-B stores ----
  float* st = (float*)smem + wid * TM * (TN + 4);
  constexpr int SLD = TN + 4;
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q) st[(i * 16 + fg * 4 + q) * SLD + j * 16 + fr] = acc[i][j][q];
  __syncthreads();

  const int row0 = m0 + wm * TM, col0 = n0 + wn * TN;
  if constexpr (EPI == EPI_SWIGLU) {
    // output tile TM x TN/2; chunk of 8 outputs; TN/16 chunks per row
    constexpr int CPR = TN / 16;
    constexpr int RPI = 64 / CPR;
    const int oc = (lane % CPR) * 8;          // output col within wave tile
    const int grp = oc / 16, within = oc % 16;  // gate cols 32*grp+within.., up cols +16
    const int ncols_out = p.N / 2;
    const int gout = col0 / 2 + oc;
    for (int rr = lane / CPR; rr < TM; rr += RPI) {
      const int gm = row0 + rr;
      if (gm >= p.M || gout >= ncols_out) continue;
      const float* srow = st + rr * SLD + grp * 32 + within;
      const bf16_t* gb = p.bias ? p.bias + col0 + grp * 32 + within : nullptr;
      unsigned packed[4];
#pragma unroll
      for (int e = 0; e < 8; e += 2) {
        float g0 = srow[e], g1 = srow[e + 1], u0 = srow[16 + e], u1 = srow[16 + e + 1];
        if (gb) {
          g0 += bf2f(gb[e]);
          g1 += bf2f(gb[e + 1]);
          u0 += bf2f(gb[16 + e]);
          u1 += bf2f(gb[16 + e + 1]);
        }
        packed[e / 2] = pack_bf2(gate_act(g0, p.relu) * u0, gate_act(g1, p.relu) * u1);
      }
      *(u32x4_t*)(p.C + (size_t)gm * p.ldc + gout) = u32x4_t{packed[0], packed[1], packed[2], packed[3]};
    }
  } else {
    constexpr int CPR = TN / 8;
    constexpr int RPI = 64 / CPR;
    const int cc = (lane % CPR) * 8;
    const int gn = col0 + cc;
    for (int rr = lane / CPR; rr < TM; rr += RPI) {
      const int gm = row0 + rr;
      if (gm >= p.M || gn >= p.N) continue;
      const float* srow = st + rr * SLD + cc;
      float v[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = srow[e];
      if constexpr (EPI == EPI_PARTIAL) {
        float* dst = p.ws + ((size_t)blockIdx.z * p.M + gm) * p.N + gn;
        *(f32x4_t*)dst = f32x4_t{v[0], v[1], v[2], v[3]};
        *(f32x4_t*)(dst + 4) = f32x4_t{v[4], v[5], v[6], v[7]};
        continue;
      }
      if (p.bias) {
        u32x4_t b = *(const u32x4_t*)(p.bias + gn);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          v[2 * e] += bf2f((bf16_t)(b[e] & 0xffff));
          v[2 * e + 1] += bf2f((bf16_t)(b[e] >> 16));
        }
      }
      if constexpr (EPI == EPI_GELU) {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = gelu_erf(v[e]);
      }
      if constexpr (EPI == EPI_RESID) {
        u32x4_t r = *(const u32x4_t*)(p.resid + (size_t)gm * p.ldr + gn);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          v[2 * e] += bf2f((bf16_t)(r[e] & 0xffff));
          v[2 * e + 1] += bf2f((bf16_t)(r[e] >> 16));
        }
      }
      *(u32x4_t*)(p.C + (size_t)gm * p.ldc + gn) =
          u32x4_t{pack_bf2(v[0], v[1]), pack_bf2(v[2], v[3]), pack_bf2(v[4], v[5]), pack_bf2(v[6], v[7])};
    }
  }
}

// ------------------------------------------------------------------------------------------
// Weight-streaming product (2 rows to some 1000: decoding, short prompts, short texts; bf16, and fp16 for the encoders).
// K in stages of 64; tiles of 32 x 128, 64 x 128, 64 x 64, 128 x 64, 128 x 128 and 192 x 128, four or eight waves.
//  * A stage (8 - 24 KB of A, 8 or 16 KB of W) arrives by LDS-DMA in a ring that fills LDS. What a CU can have on its way
//    beyond the L2 is 32 KB whatever is asked for (57 GB/s from HBM or the last-level cache, 142 GB/s from L2; loads into
//    registers the same), and A's pieces wait in that queue behind W's, so the tile's bytes per product bound it, not the
//    ring's depth.
//  * A stage's two halves of 32 are read from LDS one ahead of the MFMAs, across the barrier, and the next stage's LDS-DMA
//    instructions lie between the MFMAs (16 address cycles each: behind the barrier, all together, every wave's MFMAs waited
//    for them). 1024 x 1024 x 4096 in 128 x 128 tiles 37 -> 31 (halves) -> 26 us (pieces), 256 x 4096 x 1024 in 64 x 64 8.4 -> 7.6.
//  * One workgroup per CU walks units (tile, K split) b, b + G, ...; the ring runs on across units, so the next one's
//    weights are on their way during this one's epilogue. Past the last unit the pieces are issued against an empty
//    resource (no traffic): the counted waits stay the same to the end.
//  * NT, one row block (W is read once): a tile of columns begins at a K-step of its own (its number, round K). Workgroups that
//    all read the same columns of rows a power of two apart ask the same few channels at a time: 64 x 28672 x 4096 46.6 ->
//    40.3 us (5.8 TB/s; a kernel that only loads that much takes 38), 64 x 128256 x 4096 197 -> 189. The order of a sum depends
//    on its column only. With more row blocks it gained nothing, and sums are in the phase-split kernel's order.
//  * W is the MFMA's A operand, so a lane holds 4 consecutive columns of a row and stores them without staging.
//  * nrm: the rows of A are the raw residual stream, and the result's rows are scaled by rsqrt(sum of the parts'
//    squares / norm_k + eps) (gemm_dk.hip); the parts are added up while the first stages are on their way.
constexpr int WS_LDS = 160 * 1024;

struct WsNorm {
  const float* ssq;  // [parts][64]; null: none
  int parts, norm_k;
  float eps;
};

template <int BM, int BN, int WGM, int WGN, int EPI, bool NT, typename T>
__global__ void __launch_bounds__(64 * WGM * WGN)
gemm_ws_kernel(GemmArgs p, WsNorm nrm, int splits) {
  constexpr int NW = WGM * WGN, A_BYTES = BM * 128, STAGE = A_BYTES + BN * 128;
  constexpr bool NORM = BM <= 64 && EPI != EPI_PARTIAL;
  constexpr int SCALES = NORM ? (NW + 1) * BM * 4 : 0;                 // the rows' scales, and each wave's part of the sums
  constexpr int ST = (WS_LDS - SCALES) / STAGE < 10 ? (WS_LDS - SCALES) / STAGE : 10;  // stages of the ring
  constexpr int PA = BM / 8 / NW, PW = BN / 8 / NW;  // LDS-DMA instructions of a wave per stage
  constexpr int P = PA + PW, PH = P / 2;  // of them beside a stage's first half
  constexpr int FM = BM / WGM / 16, FN = BN / WGN / 16, WROWS = FM * 16, WCOLS = FN * 16;
  static_assert(PA >= 1 && PA <= 4 && PW >= 1 && PW <= 4 && FN % 2 == 0 && ST >= 3 && P * (ST - 2) < 64, "tile");
  typedef __attribute__((address_space(3))) void* lds_ptr_t;
  __shared__ __attribute__((aligned(16))) char smem[ST * STAGE + SCALES];
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = w / WGN, wn = w % WGN;
  const int fr = lane & 15, fg = lane >> 4;
  const int ntm = (p.M + BM - 1) / BM, ntn = (p.N + BN - 1) / BN, units = ntm * ntn * splits;
  const int nk = p.k_per_split / 64, G = gridDim.x;
  const int mine = (units - (int)blockIdx.x + G - 1) / G;  // units of this workgroup (>= 1)

  // unit -> (first row, first column, split); row blocks of one W tile are neighbours on one XCD
  auto unit_of = [&](int i, int& m0, int& n0, int& sp) __attribute__((always_inline)) {
    const int t = xcd_remap((int)blockIdx.x + i * G, units);
    m0 = t % ntm * BM;
    n0 = t / ntm % ntn * BN;
    sp = t / (ntm * ntn);
  };

  // ---- the ring's writing side: stage `ik` of unit `iu` is next ----
  __amdgpu_buffer_rsrc_t ra, rw;
  unsigned ao[4], wo[4];  // row w * 8 * PA + j * 8 + lane / 8 of A (PW: of W), 16-B chunk swizzled by (row >> 1) & 7
  int iu = 0, ik = 0, pos = 0, slot = 0;  // pos: the K-step that stage ik holds
  auto open = [&]() __attribute__((always_inline)) {  // resources and offsets of unit iu
    int m0, n0, sp;
    unit_of(iu, m0, n0, sp);
    pos = NT ? n0 / BN % nk : 0;
    const int n = iu < mine ? 0x7ffffff0 : 0;
    ra = __builtin_amdgcn_make_buffer_rsrc(
        (void*)((const char*)p.A + (size_t)m0 * p.lda * 2 + (size_t)sp * p.k_per_split * 2), (short)0, n, 0x00020000);
    rw = __builtin_amdgcn_make_buffer_rsrc(
        (void*)((const char*)p.W + (size_t)n0 * p.K * 2 + (size_t)sp * p.k_per_split * 2), (short)0, n, 0x00020000);
#pragma unroll
    for (int j = 0; j < PA; ++j) {
      const int r = w * 8 * PA + j * 8 + (lane >> 3), c = (lane & 7) ^ ((r >> 1) & 7);
      ao[j] = (unsigned)(min(m0 + r, p.M - 1) - m0) * (unsigned)(p.lda * 2) + c * 16;
    }
#pragma unroll
    for (int j = 0; j < PW; ++j) {
      const int r = w * 8 * PW + j * 8 + (lane >> 3), c = (lane & 7) ^ ((r >> 1) & 7);
      wo[j] = (unsigned)(min(n0 + r, p.N - 1) - n0) * (unsigned)(p.K * 2) + c * 16;
    }
  };
  auto piece = [&](int j) __attribute__((always_inline)) {  // the wave's j-th of PA + PW instructions of a stage
    char* base = smem + slot * STAGE;
    if (j < PA)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (lds_ptr_t)(base + (w * PA + j) * 1024), 16, ao[j & 3], pos * 128, 0, 0);
    else
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, (lds_ptr_t)(base + A_BYTES + (w * PW + j - PA) * 1024), 16, wo[(j - PA) & 3],
                                               pos * 128, 0, NT ? 2 : 0);
  };
  auto next_stage = [&]() __attribute__((always_inline)) {
    slot = slot + 1 == ST ? 0 : slot + 1;
    pos = pos + 1 == nk ? 0 : pos + 1;
    if (++ik == nk) {
      ik = 0;
      ++iu;
      open();
    }
  };
  // this wave's pieces of the stage that is read next are in (newer ones: ST - 3 whole stages and PH pieces); after the
  // barrier everyone's are, and what was read before it may be written
  auto landed = [&](auto newer) __attribute__((always_inline)) {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(decltype(newer)::value) : "memory");
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
  };
  // the rows' sums of squares: thread = (part, 4 rows), 8 parts each on their way before the ring's first stages
  [[maybe_unused]] float* scale = (float*)(smem + ST * STAGE);
  [[maybe_unused]] f32x4_t sq[8];
  constexpr int RQ = BM / 4, PL = 64 * NW / RQ;  // row quads, parts at a time
  if constexpr (NORM)
    if (nrm.ssq)
#pragma unroll
      for (int j = 0; j < 8; ++j)
        sq[j] = *(const f32x4_t*)(nrm.ssq + (size_t)min(tid / RQ + j * PL, nrm.parts - 1) * 64 + tid % RQ * 4);
  open();
#pragma unroll 1
  for (int i = 0; i < ST - 1; ++i) {
#pragma unroll
    for (int j = 0; j < P; ++j) piece(j);
    next_stage();
  }
  if constexpr (NORM)
    if (nrm.ssq) {
      f32x4_t s{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < 8; ++j) s += tid / RQ + j * PL < nrm.parts ? sq[j] : f32x4_t{0.f, 0.f, 0.f, 0.f};
      for (int q = tid / RQ + 8 * PL; q < nrm.parts; q += PL) s += *(const f32x4_t*)(nrm.ssq + (size_t)q * 64 + tid % RQ * 4);
#pragma unroll
      for (int o = RQ; o < 64; o <<= 1)
#pragma unroll
        for (int e = 0; e < 4; ++e) s[e] += __shfl_xor(s[e], o, 64);
      if (lane < RQ) *(f32x4_t*)(scale + (w + 1) * BM + lane * 4) = s;
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      if (tid < BM) {
        float t = 0.f;
#pragma unroll
        for (int i = 1; i <= NW; ++i) t += scale[i * BM + tid];
        scale[tid] = rsqrtf(t / nrm.norm_k + nrm.eps);  // (visible at the first stage's barrier)
      }
    }

  int rd = 0;  // the slot that is read next
  const int sw = (fr >> 1) & 7;
  const int co[2] = {(fg ^ sw) << 4, ((4 + fg) ^ sw) << 4};
  bf16x8_t af[2][FM], wf[2][FN];  // fragments of a stage's halves: one is read while the other is multiplied
  auto read = [&](auto half) __attribute__((always_inline)) {
    constexpr int H = decltype(half)::value;
    const char* sa = smem + rd * STAGE + wm * WROWS * 128 + fr * 128 + co[H];
    const char* sb = smem + rd * STAGE + A_BYTES + wn * WCOLS * 128 + fr * 128 + co[H];
#pragma unroll
    for (int j = 0; j < FN; ++j) wf[H][j] = *(const bf16x8_t*)(sb + j * 2048);
#pragma unroll
    for (int i = 0; i < FM; ++i) af[H][i] = *(const bf16x8_t*)(sa + i * 2048);
  };
  f32x4_t acc[FM][FN];
  // MFMAs of a half with pieces of the next stage between them (together at the barrier the waves would wait for the
  // address unit, 16 cycles an instruction, with their MFMAs behind them)
  auto multiply = [&](auto half) __attribute__((always_inline)) {
    constexpr int H = decltype(half)::value, J0 = H ? PH : 0, NJ = H ? P - PH : PH;
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        acc[i][j] = T::mma16(wf[H][j], af[H][i], acc[i][j]);
#pragma unroll
        for (int q = 0; q < NJ; ++q)
          if (i * FN + j == (q + 1) * FM * FN / (NJ + 1) - 1 + (NJ + 1 > FM * FN)) {
            __builtin_amdgcn_sched_barrier(0);
            piece(J0 + q);
            __builtin_amdgcn_sched_barrier(0);
          }
      }
  };
  using H0 = std::integral_constant<int, 0>;
  using H1 = std::integral_constant<int, 1>;
  landed(std::integral_constant<int, P * (ST - 2)>{});  // stage 0
  read(H0{});
  for (int u = 0; u < mine; ++u) {
    int m0, n0, sp;
    unit_of(u, m0, n0, sp);
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) acc[i][j] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    for (int kt = 0; kt < nk; ++kt) {
      read(H1{});
      multiply(H0{});
      rd = rd + 1 == ST ? 0 : rd + 1;
      landed(std::integral_constant<int, P * (ST - 3) + PH>{});
      read(H0{});
      multiply(H1{});
      next_stage();
    }
    // ---- row m0 + WROWS wm + 16 i + fr, columns col + 16 j + 4 fg .. + 3 ----
    const int col = n0 + wn * WCOLS + 4 * fg;
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      const int m = m0 + wm * WROWS + i * 16 + fr;
      if (m >= p.M) continue;
      float inv = 1.f;
      if constexpr (NORM)
        if (nrm.ssq) inv = scale[wm * WROWS + i * 16 + fr];  // (one row block: up to 64 rows)
      if constexpr (EPI == EPI_SWIGLU) {
#pragma unroll
        for (int j = 0; j < FN; j += 2) {
          const int oc = n0 / 2 + wn * (WCOLS / 2) + j * 8 + 4 * fg, gc = col + 16 * j;
          if (oc >= p.N / 2) continue;
          float v[4];
#pragma unroll
          for (int q = 0; q < 4; ++q)
            v[q] = gate_act(fmaf(acc[i][j][q], inv, p.bias ? T::to_f(p.bias[gc + q]) : 0.f), p.relu) *
                   fmaf(acc[i][j + 1][q], inv, p.bias ? T::to_f(p.bias[gc + 16 + q]) : 0.f);
          *(u32x2_t*)(p.C + (size_t)m * p.ldc + oc) = u32x2_t{T::pack2(v[0], v[1]), T::pack2(v[2], v[3])};
        }
      } else {
#pragma unroll
        for (int j = 0; j < FN; ++j) {
          const int gn = col + 16 * j;
          if (gn >= p.N) continue;
          if constexpr (EPI == EPI_PARTIAL) {
            *(f32x4_t*)(p.ws + ((size_t)sp * p.M + m) * p.N + gn) = acc[i][j];
          } else {
            float v[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) v[q] = fmaf(acc[i][j][q], inv, p.bias ? T::to_f(p.bias[gn + q]) : 0.f);
            if constexpr (EPI == EPI_GELU) {
#pragma unroll
              for (int q = 0; q < 4; ++q) v[q] = gelu_erf(v[q]);
            }
            if constexpr (EPI == EPI_RESID) {
              const u32x2_t r = *(const u32x2_t*)(p.resid + (size_t)m * p.ldr + gn);
#pragma unroll
              for (int q = 0; q < 2; ++q) {
                v[2 * q] += T::to_f((bf16_t)(r[q] & 0xffff));
                v[2 * q + 1] += T::to_f((bf16_t)(r[q] >> 16));
              }
            }
            *(u32x2_t*)(p.C + (size_t)m * p.ldc + gn) = u32x2_t{T::pack2(v[0], v[1]), T::pack2(v[2], v[3])};
          }
        }
      }
    }
  }
  // the pieces issued past the end write zeros into LDS: in before the workgroup (and its LDS) goes
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

// Split-K reduction + epilogue. One thread per 8 output elements (16-B stores).
// ssq_in (nullable): deferred RMSNorm of the product's rows — the A rows were the raw residual
// stream, so by linearity out[m, :] = inv[m] * (A W^T)[m, :], inv[m] = rsqrt(sum_p ssq_in[p][m] /
// norm_k + eps) over the producer's `parts` row sums ([parts][64] floats; gains folded into W).
template <typename T = BF16T>
__global__ void __launch_bounds__(256)
gemm_splitk_reduce(const float* __restrict__ ws, int splits, int M, int N, int epi,
                   const bf16_t* __restrict__ bias, const bf16_t* __restrict__ resid, int ldr,
                   bf16_t* __restrict__ C, int ldc, const float* __restrict__ ssq_in = nullptr, int parts = 0,
                   int norm_k = 1, float eps = 0.f, int relu = 0) {
  const int nout = (epi == EPI_SWIGLU) ? N / 2 : N;
  const int chunks = nout / 8;
  const size_t total = (size_t)M * chunks;
  for (size_t idx = blockIdx.x * (size_t)blockDim.x + threadIdx.x; idx < total;
       idx += (size_t)gridDim.x * blockDim.x) {
    const int m = (int)(idx / chunks), oc = (int)(idx % chunks) * 8;
    float inv = 1.f;
    if (ssq_in) {  // a handful of L2-resident floats per row (fixed summation order)
      inv = rsqrtf(sum_strided(ssq_in + m, parts, 64) / norm_k + eps);
    }
    float v[8];
    if (epi == EPI_SWIGLU) {
      const int grp = oc / 16, within = oc % 16;
      const int gc = grp * 32 + within;
      float g[8], u[8];
      sum_rows8(ws + (size_t)m * N + gc, splits, (size_t)M * N, g);
      sum_rows8(ws + (size_t)m * N + gc + 16, splits, (size_t)M * N, u);
#pragma unroll
      for (int e = 0; e < 8; ++e)
        v[e] = gate_act(fmaf(g[e], inv, bias ? T::to_f(bias[gc + e]) : 0.f), relu) *
               fmaf(u[e], inv, bias ? T::to_f(bias[gc + 16 + e]) : 0.f);
    } else {
      sum_rows8(ws + (size_t)m * N + oc, splits, (size_t)M * N, v);
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] *= inv;
      if (bias) {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] += T::to_f(bias[oc + e]);
      }
      if (epi == EPI_GELU) {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = gelu_erf(v[e]);
      }
      if (epi == EPI_RESID) {
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] += T::to_f(resid[(size_t)m * ldr + oc + e]);
      }
    }
    *(u32x4_t*)(C + (size_t)m * ldc + oc) =
        u32x4_t{T::pack2(v[0], v[1]), T::pack2(v[2], v[3]), T::pack2(v[4], v[5]), T::pack2(v[6], v[7])};
  }
}

// ------------------------------------------------------------------------------------------
// GEMV (M = 1: the batch-1 decode step that sets cache-miss latency). Pure weight streaming:
// every wave instruction loads 1 KiB of ONE weight row (64 lanes x 16 B, fully coalesced,
// non-temporal), R rows x U k-blocks of loads are in flight per wave before any FMA, the 8-wide
// dot products accumulate in fp32 per lane and each row is reduced across the wave once.
// The activation row (K bf16) is read through the caches (every wave reads the same vector).
// EPI_SWIGLU: a wave owns 2 gate rows and their 2 up rows (16-row interleave) -> 2 outputs.
// KS = 2: two neighbouring waves of a workgroup split a row's K range (long rows on narrow
// matrices: the K=8192 down projection has 3072 rows, one 16 KiB row per wave was two dependent
// HBM round trips at U=8) and combine their partial sums through LDS.
template <int EPI, int R, int U, int KS = 1>
__global__ void __launch_bounds__(256)
gemv_kernel(GemmArgs p) {
  static_assert(EPI != EPI_SWIGLU || R == 4, "SwiGLU waves own 2 gate + 2 up rows");
  static_assert(KS == 1 || KS == 2, "KS");
  const int lane = threadIdx.x & 63;
  const int wv = blockIdx.x * 4 + (threadIdx.x >> 6);  // global wave index
  const int wg = wv / KS, ks = wv % KS;                 // row group, K part
  int rows[R];
  if constexpr (EPI == EPI_SWIGLU) {
    const int g = wg >> 3, t = wg & 7;
#pragma unroll
    for (int r = 0; r < R; ++r) rows[r] = g * 32 + 2 * t + (r & 1) + (r >> 1) * 16;
  } else {
#pragma unroll
    for (int r = 0; r < R; ++r) rows[r] = wg * R + r;
  }
  if (KS == 1 && rows[0] >= p.N) return;  // KS = 2: every wave reaches the LDS exchange below
  const bf16_t* wr[R];
#pragma unroll
  for (int r = 0; r < R; ++r) wr[r] = p.W + (size_t)min(rows[r], p.N - 1) * p.K + lane * 8;
  const bf16_t* ar = p.A + lane * 8;
  const bf16_t* gr = p.gamma ? p.gamma + lane * 8 : nullptr;
  // fused RMSNorm: eps > 0 (gamma null = unit gain: the decoder folds RMSNorm gains into the
  // following weights at load, so the GEMV streams no gain vector)
  const bool rms = p.eps > 0.f;
  const int nkb = p.K / 512;
  const int kb0 = ks * nkb / KS, kb1 = (ks + 1) * nkb / KS;
  float acc[R];
#pragma unroll
  for (int r = 0; r < R; ++r) acc[r] = 0.f;
  float ss = 0.f;  // fused RMSNorm: sum of squares of the raw input row (the wave's K range)
  for (int kb = kb0; kb < kb1; kb += U) {
    u32x4_t wv[U][R], av[U], gv[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = min(kb + u, kb1 - 1) * 512;
#pragma unroll
      for (int r = 0; r < R; ++r) wv[u][r] = __builtin_nontemporal_load((const u32x4_t*)(wr[r] + k));
      av[u] = *(const u32x4_t*)(ar + k);
      if (gr) gv[u] = *(const u32x4_t*)(gr + k);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (kb + u >= kb1) break;
      float a[8];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        a[2 * e] = bf2f((bf16_t)(av[u][e] & 0xffff));
        a[2 * e + 1] = bf2f((bf16_t)(av[u][e] >> 16));
      }
      if (rms) {
#pragma unroll
        for (int e = 0; e < 4; ++e) ss = fmaf(a[2 * e], a[2 * e], fmaf(a[2 * e + 1], a[2 * e + 1], ss));
      }
      if (gr) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          a[2 * e] *= bf2f((bf16_t)(gv[u][e] & 0xffff));
          a[2 * e + 1] *= bf2f((bf16_t)(gv[u][e] >> 16));
        }
      }
#pragma unroll
      for (int r = 0; r < R; ++r)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          acc[r] = fmaf(bf2f((bf16_t)(wv[u][r][e] & 0xffff)), a[2 * e], acc[r]);
          acc[r] = fmaf(bf2f((bf16_t)(wv[u][r][e] >> 16)), a[2 * e + 1], acc[r]);
        }
    }
  }
#pragma unroll
  for (int r = 0; r < R; ++r) acc[r] = wave_sum(acc[r]);
  if (rms) ss = wave_sum(ss);
  if constexpr (KS == 2) {
    __shared__ float xch[4][R + 1];
    const int w = threadIdx.x >> 6;
    if (lane == 0) {
#pragma unroll
      for (int r = 0; r < R; ++r) xch[w][r] = acc[r];
      xch[w][R] = ss;
    }
    __syncthreads();
    if (ks != 0 || rows[0] >= p.N) return;
#pragma unroll
    for (int r = 0; r < R; ++r) acc[r] += xch[w + 1][r];
    ss += xch[w + 1][R];
  }
  if (rms) {
    const float inv = rsqrtf(ss / p.K + p.eps);
#pragma unroll
    for (int r = 0; r < R; ++r) acc[r] *= inv;
  }
  if (lane != 0) return;
  if constexpr (EPI == EPI_SWIGLU) {
    const int g = wg >> 3, t = wg & 7;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int o = g * 16 + 2 * t + j;
      if (o >= p.N / 2) continue;
      const float gb = p.bias ? bf2f(p.bias[rows[j]]) : 0.f, ub = p.bias ? bf2f(p.bias[rows[2 + j]]) : 0.f;
      p.C[o] = f2bf(gate_act(acc[j] + gb, p.relu) * (acc[2 + j] + ub));
    }
  } else {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int n = rows[r];
      if (n >= p.N) continue;
      float v = acc[r];
      if (p.bias) v += bf2f(p.bias[n]);
      if constexpr (EPI == EPI_GELU) v = gelu_erf(v);
      if constexpr (EPI == EPI_RESID) v += bf2f(p.resid[n]);
      p.C[n] = f2bf(v);
    }
  }
}

template <int R, int U, int KS = 1>
static int launch_gemv_r(const GemmArgs& a, int epi, hipStream_t s) {
  const int waves = (a.N + R - 1) / R * KS;
  dim3 grid((waves + 3) / 4), block(256);
  switch (epi) {
    case EPI_NONE: gemv_kernel<EPI_NONE, R, U, KS><<<grid, block, 0, s>>>(a); break;
    case EPI_BIAS: gemv_kernel<EPI_BIAS, R, U, KS><<<grid, block, 0, s>>>(a); break;
    case EPI_GELU: gemv_kernel<EPI_GELU, R, U, KS><<<grid, block, 0, s>>>(a); break;
    case EPI_RESID: gemv_kernel<EPI_RESID, R, U, KS><<<grid, block, 0, s>>>(a); break;
    default: return (int)hipErrorInvalidValue;
  }
  return (int)hipGetLastError();
}

// K-blocks (512 elements = 1 KiB per row) in flight per row: the whole row when it is short
// (K = 3072: 6 blocks, one round of loads and no clamped duplicate loads), 8 per round otherwise.
static int gemv_u(int K, int /*R*/) {
  const int nkb = K / 512;
  if (nkb <= 4) return 4;
  if (nkb == 6) return 6;
  // 8, not the whole row at K = 8192: at U = 16 the compiler sinks the loads to their uses
  // (28 VGPRs, one block in flight) and the down projection drops to ~3 TB/s (measured)
  return 8;
}

template <int R>
static int launch_gemv_ru(const GemmArgs& a, int epi, hipStream_t s) {
  switch (gemv_u(a.K, R)) {
    case 6: return launch_gemv_r<R, 6>(a, epi, s);
    case 8: return launch_gemv_r<R, 8>(a, epi, s);
    default: return launch_gemv_r<R, 4>(a, epi, s);
  }
}

// Rows per wave: enough waves (>= ~4 per SIMD) that the loads in flight cover HBM latency on
// narrow matrices, 4 rows per wave (more bytes per wave) on wide ones.
static int launch_gemv(const GemmArgs& a, int epi, hipStream_t s) {
  if (a.M != 1 || a.K % 512 || a.N % 4) return (int)hipErrorInvalidValue;
  if (epi == EPI_SWIGLU) {
    dim3 grid((a.N / 4 + 3) / 4), block(256);
    switch (gemv_u(a.K, 4)) {
      case 6: gemv_kernel<EPI_SWIGLU, 4, 6><<<grid, block, 0, s>>>(a); break;
      case 8: gemv_kernel<EPI_SWIGLU, 4, 8><<<grid, block, 0, s>>>(a); break;
      default: gemv_kernel<EPI_SWIGLU, 4, 4><<<grid, block, 0, s>>>(a); break;
    }
    return (int)hipGetLastError();
  }
  if (a.N >= 16384) return launch_gemv_ru<4>(a, epi, s);
  if (a.N >= 8192) return launch_gemv_ru<2>(a, epi, s);
  // long rows on a narrow matrix (down projection, K = 8192): two waves per row, 8 blocks each
  if (a.K >= 8192 && a.K % 1024 == 0) return launch_gemv_r<1, 8, 2>(a, epi, s);
  return launch_gemv_ru<1>(a, epi, s);
}

template <int BM, int BN, int WM, int WN, int PF = 1>
static int launch_tile(const GemmArgs& a, int epi, int splits, hipStream_t s) {
  const int ntm = (a.M + BM - 1) / BM, ntn = (a.N + BN - 1) / BN;
  dim3 grid(ntm * ntn, 1, splits), block(256);
  switch (splits > 1 ? (int)EPI_PARTIAL : epi) {
    case EPI_NONE: gemm_bf16_kernel<BM, BN, WM, WN, EPI_NONE, PF><<<grid, block, 0, s>>>(a); break;
    case EPI_BIAS: gemm_bf16_kernel<BM, BN, WM, WN, EPI_BIAS, PF><<<grid, block, 0, s>>>(a); break;
    case EPI_GELU: gemm_bf16_kernel<BM, BN, WM, WN, EPI_GELU, PF><<<grid, block, 0, s>>>(a); break;
    case EPI_SWIGLU: gemm_bf16_kernel<BM, BN, WM, WN, EPI_SWIGLU, PF><<<grid, block, 0, s>>>(a); break;
    case EPI_RESID: gemm_bf16_kernel<BM, BN, WM, WN, EPI_RESID, PF><<<grid, block, 0, s>>>(a); break;
    case EPI_PARTIAL: gemm_bf16_kernel<BM, BN, WM, WN, EPI_PARTIAL, PF><<<grid, block, 0, s>>>(a); break;
    default: return (int)hipErrorInvalidValue;
  }
  return (int)hipGetLastError();
}

template <int BM, int BN, int WGM, int WGN, bool NT, typename T = BF16T>
static int launch_ws_tile(const GemmArgs& a, int epi, int splits, const WsNorm& nrm, hipStream_t s) {
  const long units = (long)((a.M + BM - 1) / BM) * ((a.N + BN - 1) / BN) * splits;
  if (units > 0x7fffffffL || a.k_per_split % 64 || a.k_per_split < 64) return (int)hipErrorInvalidValue;
  const dim3 grid((unsigned)min(units, 256L)), block(64 * WGM * WGN);
#define WS_LAUNCH(E) gemm_ws_kernel<BM, BN, WGM, WGN, E, NT, T><<<grid, block, 0, s>>>(a, nrm, splits)
  switch (splits > 1 ? (int)EPI_PARTIAL : epi) {
    case EPI_NONE: WS_LAUNCH(EPI_NONE); break;
    case EPI_BIAS: WS_LAUNCH(EPI_BIAS); break;
    case EPI_GELU: WS_LAUNCH(EPI_GELU); break;
    case EPI_SWIGLU:
      if constexpr (T::kF16) return (int)hipErrorInvalidValue;
      else WS_LAUNCH(EPI_SWIGLU);
      break;
    case EPI_RESID: WS_LAUNCH(EPI_RESID); break;
    case EPI_PARTIAL: WS_LAUNCH(EPI_PARTIAL); break;
    default: return (int)hipErrorInvalidValue;
  }
#undef WS_LAUNCH
  return (int)hipGetLastError();
}

// 64 x 64 tiles: (8192, 16384] columns without splits (_dk_splits, _auto_splits). Narrower products have to be split either
// way, and the wider tile then moves less of A: 64 x 8192 x 4096 22.8 us at four splits vs 24.0 at two of 64 x 64. Splits are
// short, and eight waves fill and drain faster: with the reduce, 64 x 4096 x 4096 14.4 us vs 15.8 with four (8 splits), x 14336
// 28.5 / 30.2, 64 x 6144 x 4096 18.2 / 18.9 (4); unsplit 64 x 28672 x 4096 42.9 / 40.3.
// Up to 32 rows only products of more than 16384 columns come here (kernels.py, _dk_streams).
// W is read once where there is one row block only: not worth a place in the caches then.
static int launch_ws(const GemmArgs& a, int epi, int splits, const WsNorm& nrm, hipStream_t s) {
  if (a.M <= 32 && splits == 1 && a.N > 16384) return launch_ws_tile<32, 128, 1, 4, true>(a, epi, splits, nrm, s);
  if (a.M <= 64) {
    if (splits > 1) return launch_ws_tile<64, 128, 2, 4, true>(a, epi, splits, nrm, s);
    return a.N <= 16384 ? launch_ws_tile<64, 64, 2, 2, true>(a, epi, splits, nrm, s)
                        : launch_ws_tile<64, 128, 1, 4, true>(a, epi, splits, nrm, s);
  }
  return a.M <= 128 ? launch_ws_tile<128, 128, 2, 4, true>(a, epi, splits, nrm, s)
                    : launch_ws_tile<128, 128, 2, 4, false>(a, epi, splits, nrm, s);
}

// The streaming kernel's offsets into a tile's rows are 32 bits wide (_dk_splits draws the same line).
static bool ws_spans(const GemmArgs& a) { return max(a.K, a.lda) < 1 << 22; }

// The tiles of more than 64 rows (kernels.py, _row_tile): 14 = 128x128, 15 = 128x64, 16 = 64x64, 17 = 64x128, 18 = 192x128.
template <typename T>
static int launch_ws_rows(const GemmArgs& a, int epi, int tile, int splits, hipStream_t s) {
  if (!ws_spans(a)) return (int)hipErrorInvalidValue;
  switch (tile) {
    case 14:
      return a.M <= 128 ? launch_ws_tile<128, 128, 2, 4, true, T>(a, epi, splits, WsNorm{}, s)
                        : launch_ws_tile<128, 128, 2, 4, false, T>(a, epi, splits, WsNorm{}, s);
    case 15: return launch_ws_tile<128, 64, 4, 2, false, T>(a, epi, splits, WsNorm{}, s);
    case 16: return launch_ws_tile<64, 64, 2, 2, false, T>(a, epi, splits, WsNorm{}, s);
    case 17: return launch_ws_tile<64, 128, 2, 4, false, T>(a, epi, splits, WsNorm{}, s);
    case 18: return launch_ws_tile<192, 128, 4, 2, false, T>(a, epi, splits, WsNorm{}, s);
    default: return (int)hipErrorInvalidValue;
  }
}

// K splits of up to 64 rows: the ring's fill and drain cost what four stages gain over the register-staged 64x128 tile with 4
// k-tiles in flight. 64 rows, weights from HBM, register / ring us, with the reduce: 768 x 768 8.0 / 8.6 (3 stages a split), 1024
// x 1024 8.7 / 9.1 (4), 768 x 3072 10.2 / 9.8 (6), 3072 x 3072 14.5 / 13.6 (6), 4096 x 4096 15.6 / 14.5 (8), 6144 x 4096 18.8 /
// 17.2 (16), 5120 x 5120 22.9 / 20.6 (20), 4096 x 14336 29.7 / 28.3 (28). Unsplit products are faster on the ring at every
// length (64 x 12288 x 768 9.9 / 9.3).
static bool ws_pays(const GemmArgs& a, int splits) {
  return ws_spans(a) && (a.M > 64 || splits == 1 || a.k_per_split >= 6 * 64);
}

// Decode tiles: 64x128 by the rule above, else 4 k-tiles in flight per workgroup.
template <int BM, int BN>
static int launch_decode_tile(const GemmArgs& a, int epi, int splits, hipStream_t s) {
  if (BM == 64 && ws_pays(a, splits)) return launch_ws(a, epi, splits, WsNorm{}, s);
  return launch_tile<BM, BN, 1, 4, 4>(a, epi, splits, s);
}

// Split-K reduction fused with the residual add AND the next RMSNorm (decode layers, M <= 64):
// one workgroup per row sums the fp32 partials, adds bias + residual, writes the new residual
// stream row C, then normalises that (bf16-rounded) row: H = C * rsqrt(mean(C^2) + eps) * gamma.
// Replaces reduce + rmsnorm (two launches, two passes over the row) with one.
__global__ void __launch_bounds__(256)
splitk_reduce_resid_rmsnorm(const float* __restrict__ ws, int splits, int M, int N, const bf16_t* __restrict__ bias,
                            const bf16_t* __restrict__ resid, int ldr, bf16_t* __restrict__ C, int ldc,
                            const bf16_t* __restrict__ gamma, float eps, bf16_t* __restrict__ H, int ldh) {
  constexpr int MAXC = 4;  // N <= 8 * 256 * 4 = 8192
  __shared__ float red[16];
  const int m = blockIdx.x;
  const int nch = N / 8;
  float v[MAXC][8];
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < MAXC; ++i) {
    const int c = threadIdx.x + 256 * i;
    if (c >= nch) continue;
    const int oc = c * 8;
    sum_rows8(ws + (size_t)m * N + oc, splits, (size_t)M * N, v[i]);  // 8 splits' loads in flight
    const u32x4_t r = *(const u32x4_t*)(resid + (size_t)m * ldr + oc);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      v[i][2 * e] += bf2f((bf16_t)(r[e] & 0xffff)) + (bias ? bf2f(bias[oc + 2 * e]) : 0.f);
      v[i][2 * e + 1] += bf2f((bf16_t)(r[e] >> 16)) + (bias ? bf2f(bias[oc + 2 * e + 1]) : 0.f);
    }
    u32x4_t o;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      o[e] = pack_bf2(v[i][2 * e], v[i][2 * e + 1]);
      v[i][2 * e] = bf2f((bf16_t)(o[e] & 0xffff));       // normalise what the stream holds (bf16)
      v[i][2 * e + 1] = bf2f((bf16_t)(o[e] >> 16));
      ss += v[i][2 * e] * v[i][2 * e] + v[i][2 * e + 1] * v[i][2 * e + 1];
    }
    *(u32x4_t*)(C + (size_t)m * ldc + oc) = o;
  }
  const float inv = rsqrtf(block_sum(ss, red) / N + eps);
#pragma unroll
  for (int i = 0; i < MAXC; ++i) {
    const int c = threadIdx.x + 256 * i;
    if (c >= nch) continue;
    const u32x4_t g = *(const u32x4_t*)(gamma + c * 8);
    u32x4_t o;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      o[e] = pack_bf2(v[i][2 * e] * inv * bf2f((bf16_t)(g[e] & 0xffff)),
                      v[i][2 * e + 1] * inv * bf2f((bf16_t)(g[e] >> 16)));
    *(u32x4_t*)(H + (size_t)m * ldh + c * 8) = o;
  }
}

// C = resid + A.W^T (+ bias) and H = RMSNorm(C) * gamma in two launches (split-K GEMM + fused
// reduce). M <= 64 (decode), N % 8 == 0, N <= 8192. ws holds splits * M * N floats.
DA_EXPORT int da_gemm_resid_rmsnorm(const void* A, int lda, const void* W, void* C, int ldc, const void* bias,
                                    const void* resid, int ldr, int M, int N, int K, int tile, int splits, void* ws,
                                    const void* gamma, float eps, void* Hout, int ldh, void* stream) {
  hipStream_t s = (hipStream_t)stream;
  if (K % 64 || N % 8 || N > 8192 || lda % 8 || ldc % 8 || ldh % 8 || !ws || !gamma || !resid || !Hout)
    return (int)hipErrorInvalidValue;
  if (splits < 1 || (K / 64) % splits || M > 128 || (M > 64 && tile != 9)) return (int)hipErrorInvalidValue;
  if (M == 0) return 0;
  GemmArgs a{};
  a.A = (const bf16_t*)A; a.W = (const bf16_t*)W; a.C = (bf16_t*)C;
  a.bias = nullptr; a.resid = nullptr; a.ws = (float*)ws;
  a.M = M; a.N = N; a.K = K; a.lda = lda; a.ldc = ldc; a.ldr = ldr; a.k_per_split = K / splits;
  // tile 9 (65..128 rows): one 128x64 weight-streaming tile per 64 weight rows
  const int err = tile == 9   ? launch_tile<128, 64, 2, 2, 4>(a, EPI_PARTIAL, splits, s)
                  : tile == 2 ? launch_decode_tile<64, 128>(a, EPI_PARTIAL, splits, s)
                              : launch_decode_tile<32, 128>(a, EPI_PARTIAL, splits, s);
  if (err) return err;
  splitk_reduce_resid_rmsnorm<<<M, 256, 0, s>>>((const float*)ws, splits, M, N, (const bf16_t*)bias,
                                                (const bf16_t*)resid, ldr, (bf16_t*)C, ldc, (const bf16_t*)gamma, eps,
                                                (bf16_t*)Hout, ldh);
  DA_LAUNCH_CHECK();
}

// Split-K reduce of a residual-producing decode GEMM (33..64 rows) in the gemm_dk layer structure:
// C = resid + sum of the partials (+ bias), and per-row sums of squares of the bf16 rows C holds,
// one per 512-column part ([N / 512][64] floats: a consumer reads N / 512 floats per row). One wave
// per (row, 512 columns): no norm here, so no workgroup has to see a whole row — 64 rows x 6
// blocks instead of the 64 row-workgroups of splitk_reduce_resid_rmsnorm, whose 98 KB of partials
// per row was read by one CU.
__global__ void __launch_bounds__(64)
splitk_reduce_resid_ssq(const float* __restrict__ ws, int splits, int M, int N, const bf16_t* __restrict__ bias,
                        const bf16_t* __restrict__ resid, int ldr, bf16_t* __restrict__ C, int ldc,
                        float* __restrict__ ssq_out) {
  const int m = blockIdx.y, lane = threadIdx.x;
  const int oc = blockIdx.x * 512 + lane * 8;
  float v[8];
  sum_rows8(ws + (size_t)m * N + oc, splits, (size_t)M * N, v);
  const u32x4_t r = *(const u32x4_t*)(resid + (size_t)m * ldr + oc);
  u32x4_t o;
  float sq = 0.f;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const float lo = v[2 * e] + bf2f((bf16_t)(r[e] & 0xffff)) + (bias ? bf2f(bias[oc + 2 * e]) : 0.f);
    const float hi = v[2 * e + 1] + bf2f((bf16_t)(r[e] >> 16)) + (bias ? bf2f(bias[oc + 2 * e + 1]) : 0.f);
    o[e] = pack_bf2(lo, hi);
    const float bl = bf2f((bf16_t)(o[e] & 0xffff)), bh = bf2f((bf16_t)(o[e] >> 16));
    sq += bl * bl + bh * bh;  // what the stream now holds (bf16)
  }
  *(u32x4_t*)(C + (size_t)m * ldc + oc) = o;
  sq = wave_sum(sq);
  if (lane == 0) ssq_out[(size_t)blockIdx.x * 64 + m] = sq;
}

// gemm_dk's contract (DkArgs semantics, csrc/gemm_dk.hip) for 33..64 rows, and up to 32 without splits, on the streaming
// tiles: epi NONE / BIAS / SWIGLU with an optional deferred norm of A's rows (ssq_in: the raw
// residual stream as A, the row scale applied in the reduce, or without splits in the epilogue), or EPI_RESID with optional per-part
// sums of squares out (ssq_out: [N / 512][64]). splits 1: no reduce (not with ssq_out); else ws holds
// splits * M * N floats.
DA_EXPORT int da_gemm_dk_splitk(const void* A, int lda, const void* W, void* C, int ldc, const void* bias,
                                const void* resid, int ldr, int M, int N, int K, int epi, const float* ssq_in,
                                int ssq_parts, int norm_k, float eps, float* ssq_out, void* ws, int splits,
                                void* stream) {
  hipStream_t s = (hipStream_t)stream;
  if (M < 1 || M > 64 || K % 64 || N % 16 || lda % 8 || ldc % 8 || (splits > 1 && !ws) || splits < 1 || (K / 64) % splits)
    return (int)hipErrorInvalidValue;
  const int relu = epi == EPI_REGLU;
  if (relu) epi = EPI_SWIGLU;
  if (epi == EPI_SWIGLU && N % 32) return (int)hipErrorInvalidValue;
  if (epi == EPI_RESID && (!resid || ldr % 8 || ssq_in)) return (int)hipErrorInvalidValue;
  if (ssq_out && (epi != EPI_RESID || N % 512)) return (int)hipErrorInvalidValue;
  if (ssq_in && (ssq_parts < 1 || norm_k < 1 || !(eps > 0.f))) return (int)hipErrorInvalidValue;
  if (epi != EPI_NONE && epi != EPI_BIAS && epi != EPI_SWIGLU && epi != EPI_RESID) return (int)hipErrorInvalidValue;
  GemmArgs a{};
  a.A = (const bf16_t*)A; a.W = (const bf16_t*)W; a.C = (bf16_t*)C;
  a.ws = (float*)ws;
  a.M = M; a.N = N; a.K = K; a.lda = lda; a.ldc = ldc; a.ldr = ldr; a.k_per_split = K / splits;
  if (splits == 1) {  // wide products: the epilogue in the same launch
    if (ssq_out || !ws_spans(a)) return (int)hipErrorInvalidValue;
    a.bias = (const bf16_t*)bias; a.resid = (const bf16_t*)resid; a.relu = relu;
    return launch_ws(a, epi, 1, WsNorm{ssq_in, ssq_parts, norm_k, eps}, s);
  }
  const int err = launch_decode_tile<64, 128>(a, EPI_PARTIAL, splits, s);
  if (err) return err;
  if (epi == EPI_RESID && ssq_out) {
    splitk_reduce_resid_ssq<<<dim3(N / 512, M), 64, 0, s>>>((const float*)ws, splits, M, N, (const bf16_t*)bias,
                                                            (const bf16_t*)resid, ldr, (bf16_t*)C, ldc, ssq_out);
    DA_LAUNCH_CHECK();
  }
  const int nout = (epi == EPI_SWIGLU) ? N / 2 : N;
  const size_t work = (size_t)M * (nout / 8);
  const int blocks = (int)((work + 255) / 256);
  gemm_splitk_reduce<BF16T><<<blocks, 256, 0, s>>>((const float*)ws, splits, M, N, epi, (const bf16_t*)bias,
                                             (const bf16_t*)resid, ldr, (bf16_t*)C, ldc, ssq_in, ssq_parts, norm_k,
                                             eps, relu);
  DA_LAUNCH_CHECK();
}

// A . W^T left as `splits` fp32 partials [splits][M][N] in ws (splits = 1: the product itself) for a consumer
// that sums them in its own pass. Decode-sized tiles: 2 = 64x128, 3 = 32x128, 9 = 128x64, 15 = 128x64 streaming.
DA_EXPORT int da_gemm_partials(const void* A, int lda, const void* W, int M, int N, int K, int tile, int splits,
                               void* ws, void* stream) {
  if (M < 1 || K % 64 || N % 8 || lda % 8 || splits < 1 || (K / 64) % splits || !ws) return (int)hipErrorInvalidValue;
  GemmArgs a{};
  a.A = (const bf16_t*)A; a.W = (const bf16_t*)W; a.ws = (float*)ws;
  a.M = M; a.N = N; a.K = K; a.lda = lda; a.ldc = N; a.k_per_split = K / splits;
  hipStream_t s = (hipStream_t)stream;
  switch (tile) {
    case 2: return launch_decode_tile<64, 128>(a, EPI_PARTIAL, splits, s);
    case 3: return launch_decode_tile<32, 128>(a, EPI_PARTIAL, splits, s);
    case 9: return launch_tile<128, 64, 2, 2, 4>(a, EPI_PARTIAL, splits, s);
    case 15: return ws_spans(a) ? launch_ws_tile<128, 64, 4, 2, false>(a, EPI_PARTIAL, splits, WsNorm{}, s) : (int)hipErrorInvalidValue;
    default: return (int)hipErrorInvalidValue;
  }
}

// Prefill QKV projection with RoPE + KV-cache write fused into the epilogue (gemm8p EPI_ROPE);
// M >= 256 (the phase-split kernel), N == (H + 2 Hkv) * D, D % 8 == 0. kv_out = 0: the k / v
// columns of C are left unwritten (cache only).
DA_EXPORT int da_gemm_rope(const void* A, int lda, const void* W, void* C, int ldc, int M, int N, int K,
                           const void* pos, const void* slot, const void* cos_sin, void* k_cache, void* v_cache,
                           int H, int Hkv, int D, int max_seq, int kv_out, void* stream) {
  if (K % 64 || K < 128 || N % 8 || lda % 8 || ldc % 8 || D % 8 || M < 256) return (int)hipErrorInvalidValue;
  if (N != (H + 2 * Hkv) * D || !pos || !slot || !cos_sin || !k_cache || !v_cache) return (int)hipErrorInvalidValue;
  GemmArgs a{};
  a.A = (const bf16_t*)A; a.W = (const bf16_t*)W; a.C = (bf16_t*)C;
  a.M = M; a.N = N; a.K = K; a.lda = lda; a.ldc = ldc; a.k_per_split = K;
  a.rope = RopeArgs{(const int*)pos, (const int*)slot, (const float*)cos_sin, (bf16_t*)k_cache, (bf16_t*)v_cache,
                    H, Hkv, D, max_seq, kv_out ? 1 : 0};
  // the row-tile height of fewer rounds: a single round of 256-row tiles on more than half of the chip beats two of 128-row ones (us,
  // 256 rows only from 256 tiles on -> this: 1400 x 9216 x 3072 96 -> 69, 1792 96 -> 76, 1400 x 6144 x 4096 104 -> 75, 2048 116 -> 81)
  return launch_gemm8p(a, EPI_ROPE, (hipStream_t)stream, gemm8p_pick_bm(M, N, K, EPI_ROPE));
}

// Tile selection: big tiles when the grid fills 256 CUs, skinny tiles (+ split-K) for decode-sized M.
// tile: 0 = auto, 1 = 128x128, 2 = weight-streaming 64x128 / 128x128, 3 = 32x128, 4 / 7 = 256x256 phase-split (gemm8p),
// 6 = GEMV (M = 1), 8 = 128x128 PF4, 9 = 128x64 PF4, 10 = 128x256 phase-split (gemm8p), 11 = 64x128 PF4,
// 13 = 256x256 four-wave (gemm4w), 14 - 18 = weight-streaming 128x128, 128x64, 64x64, 64x128, 192x128 (launch_ws_rows).
DA_EXPORT int da_gemm_bf16(const void* A, int lda, const void* W, void* C, int ldc,
                           const void* bias, const void* resid, int ldr,
                           int M, int N, int K, int epi, int tile, int splits, void* ws,
                           const void* rms_gamma, float rms_eps, void* tail_ws, void* tail_cnt, void* stream) {
  hipStream_t s = (hipStream_t)stream;
  if (K % 64 || N % 8 || lda % 8 || ldc % 8) return (int)hipErrorInvalidValue;
  const int relu = epi == EPI_REGLU;
  if (relu) epi = EPI_SWIGLU;
  if (epi == EPI_SWIGLU && N % 32) return (int)hipErrorInvalidValue;
  if (splits < 1) splits = 1;
  if ((K / 64) % splits) return (int)hipErrorInvalidValue;
  if (splits > 1 && ws == nullptr) return (int)hipErrorInvalidValue;
  GemmArgs a{};
  a.A = (const bf16_t*)A; a.W = (const bf16_t*)W; a.C = (bf16_t*)C;
  a.bias = (const bf16_t*)bias; a.resid = (const bf16_t*)resid; a.ws = (float*)ws;
  a.M = M; a.N = N; a.K = K; a.lda = lda; a.ldc = ldc; a.ldr = ldr; a.k_per_split = K / splits;
  a.gamma = (const bf16_t*)rms_gamma; a.eps = rms_eps; a.relu = relu;
  if (tail_ws && tail_cnt) { a.tail_ws = (float*)tail_ws; a.tail_cnt = (int*)tail_cnt; }
  if ((rms_gamma || rms_eps > 0.f) && tile != 6) return (int)hipErrorInvalidValue;  // fused RMSNorm: GEMV only
  if (tile == 0) {
    // decode-sized M: 32x128 / weight-streaming tiles (+ split-K, chosen by the caller), to 639 rows;
    // from 640 rows the phase-split kernel with the row-tile height of fewer workgroup waves (gemm8p_pick_bm; 32-layer Phi-3
    // chain and single-GEMM sweeps: bench/midm_chain.py, bench/gemm_ab.py, profiles/r2, r3)
    if (M <= 32) tile = 3;
    else if (M < 640 || splits > 1) tile = 2;
    else if (K < 128) tile = 1;
    else tile = gemm8p_pick_bm(M, N, K, epi) == 256 ? 7 : 10;
  }
  if (tile == 4 || tile == 7 || tile == 10) {
    if (splits != 1 || K < 128) return (int)hipErrorInvalidValue;
    return launch_gemm8p(a, epi, s, tile == 10 ? 128 : 256);
  }
  if (tile == 13) {
    if (splits != 1 || K < 128) return (int)hipErrorInvalidValue;
    return launch_gemm4w(a, epi, s);
  }
  if (tile == 6) return launch_gemv(a, epi, s);
  int err;
  switch (tile) {
    case 1: err = launch_tile<128, 128, 2, 2>(a, epi, splits, s); break;
    case 2: err = launch_decode_tile<64, 128>(a, epi, splits, s); break;
    case 3: err = launch_decode_tile<32, 128>(a, epi, splits, s); break;
    case 8: err = launch_tile<128, 128, 2, 2, 4>(a, epi, splits, s); break;   // mid-M weight streaming
    case 9: err = launch_tile<128, 64, 2, 2, 4>(a, epi, splits, s); break;
    case 11: err = launch_tile<64, 128, 1, 4, 4>(a, epi, splits, s); break;
    case 14: case 15: case 16: case 17: case 18: err = launch_ws_rows<BF16T>(a, epi, tile, splits, s); break;
    default: return (int)hipErrorInvalidValue;
  }
  if (err || splits == 1) return err;
  const int nout = (epi == EPI_SWIGLU) ? N / 2 : N;
  const size_t work = (size_t)M * (nout / 8);
  int blocks = (int)((work + 255) / 256);
  if (blocks > 4096) blocks = 4096;
  gemm_splitk_reduce<BF16T><<<blocks, 256, 0, s>>>((const float*)ws, splits, M, N, epi, a.bias, a.resid, ldr,
                                             a.C, ldc, nullptr, 0, 1, 0.f, relu);
  DA_LAUNCH_CHECK();
}

// fp16 product for the encoder's DTYPE=fp16 path: C = epi(A W^T), A [M, K] / W [N, K] / C / bias / resid fp16, fp32
// accumulation; epi NONE / BIAS / GELU / RESID. tile: 0 = the phase-split kernel with the row-tile height of fewer workgroup
// waves, 7 / 10 = that with 256 / 128 rows, 14 - 18 as da_gemm_bf16.
DA_EXPORT int da_gemm_f16(const void* A, int lda, const void* W, void* C, int ldc, const void* bias,
                          const void* resid, int ldr, int M, int N, int K, int epi, int tile, int splits, void* ws,
                          void* tail_ws, void* tail_cnt, void* stream) {
  hipStream_t s = (hipStream_t)stream;
  if (M < 1 || K % 64 || K < 128 || N % 8 || lda % 8 || ldc % 8) return (int)hipErrorInvalidValue;
  if (epi != EPI_NONE && epi != EPI_BIAS && epi != EPI_GELU && epi != EPI_RESID) return (int)hipErrorInvalidValue;
  if (epi == EPI_RESID && (!resid || ldr % 8)) return (int)hipErrorInvalidValue;
  if (splits < 1 || (K / 64) % splits || (splits > 1 && !ws)) return (int)hipErrorInvalidValue;
  GemmArgs a{};
  a.A = (const bf16_t*)A; a.W = (const bf16_t*)W; a.C = (bf16_t*)C; a.ws = (float*)ws;
  a.bias = (const bf16_t*)bias; a.resid = (const bf16_t*)resid;
  a.M = M; a.N = N; a.K = K; a.lda = lda; a.ldc = ldc; a.ldr = ldr; a.k_per_split = K / splits;
  if (tile == 0 || tile == 7 || tile == 10) {
    if (splits != 1) return (int)hipErrorInvalidValue;
    if (tail_ws && tail_cnt) { a.tail_ws = (float*)tail_ws; a.tail_cnt = (int*)tail_cnt; }
    return launch_gemm8p(a, 100 + epi, s, tile == 7 ? 256 : tile == 10 ? 128 : gemm8p_pick_bm(M, N, K, epi));
  }
  const int err = launch_ws_rows<F16T>(a, epi, tile, splits, s);
  if (err || splits == 1) return err;
  const int blocks = (int)min(((size_t)M * (N / 8) + 255) / 256, (size_t)4096);
  gemm_splitk_reduce<F16T><<<blocks, 256, 0, s>>>((const float*)ws, splits, M, N, epi, a.bias, a.resid, ldr, a.C, ldc, nullptr,
                                                  0, 1, 0.f, 0);
  DA_LAUNCH_CHECK();
}
