// Attention kernels for gfx950.
//
// 1) flash_attn_v2: packed (varlen) prefill attention, bidirectional (BERT encoder)
//    or causal with GQA (Llama-3 / Phi-3 prefill, N6/N7), optionally over a shared-prefix head in
//    the KV cache. Online softmax in fp32, bf16 MFMA 32x32x16, "swapped" S^T = K.Q^T formulation
//    (details above the kernel).
//
// 2) decode attention (one new token per sequence) over the KV cache [slot, Hkv, max_seq, D]:
//    split-KV ("flash-decoding") so a batch of long contexts fills all 256 CUs; fp32 partials
//    (unnormalised O, running max, running sum) merged by decode_combine.
#include "common.h"

#include <cstdlib>

// Floating-point contraction only within one expression (a*b + c -> fma), never across statements:
// with the HIP default (fast) the backend fuses differently depending on the surrounding code, and
// the decode attention inlined into the persistent batch-1 kernel (decode_b1.hip) then differed from
// decode_attn_kernel by one bf16 ulp on some heads (measured on the MI355X, bench/b1_diverge.py).
// Both files pin the same rule, so the two compute the same bits by construction.
#pragma clang fp contract(on)

// ------------------------------------------------------------------------------------------
// flash_attn_v2: 32x32x16 MFMA, 4 waves x 32 queries (128 queries per workgroup), 64-key tiles
// double-buffered in LDS with register staging (tile t+1's global loads are in flight while tile t
// is computed; one barrier per tile).
//   S^T[key][q] = K·Q^T : A = K rows from LDS (16-B pad per row -> conflict-free ds_read_b128),
//                         B = Q^T from registers (loaded once per wave).
//   lane l owns query l&31; its 32 keys of a 64-key tile sit in the two S^T accumulators, the
//   other 32 in lane l^32 -> row max / row sum need ONE v_permlane32_swap each.
//   O^T[d][q] += V^T·P^T : B = P^T straight from the S^T registers (k index permuted), A = V^T
//                         fetched from the row-major V tile with ds_read_b64_tr_b16 (hardware
//                         transpose; row stride chosen so the 4-row x 2-group reads are
//                         bank-conflict-free).
//   scale·log2(e) is folded into the exp2 argument (one FMA per score); the O rescale is skipped
//   when no lane's running max moved; causal tiles past a wave's last query are skipped by that
//   wave (it still stages tiles and joins the barrier).
template <int D, int NW = 4, int QH = 1>
struct FA2Cfg {
  static constexpr int KT = 64, QW = 32 * QH, QB = QW * NW, NT = 64 * NW;
  static constexpr int KSTR = D * 2 + 16;                                         // bytes
  static constexpr int VSTR = (D == 64) ? 192 : (D == 128) ? 320 : D * 2;         // bytes
  static constexpr int KBUF = KT * KSTR, VBUF = KT * VSTR;
  static constexpr int CPR = D / 8, LPT = (KT * CPR + NT - 1) / NT;
  static constexpr int SMEM = 2 * (KBUF + VBUF);
};

// Shared-prefix keys (pre.len > 0): every sequence's keys are [pre.len prefix keys | its own keys];
// the prefix K/V live once in a KV-cache slot ([Hkv][max_seq][D]: head stride pre.hstride, row
// stride D), RoPE already applied. Query i of a sequence sits at key position pre.len + i (causal
// mask bottom-right aligned), so a batch whose prompts share a system-prompt head prefills that
// head once and only the suffixes here.
struct FaPrefix {
  const bf16_t* k;
  const bf16_t* v;
  long long hstride;
  int len;
  int rev;  // dispatch order (set by the launcher): bit 0 causal longest-first, bit 1 XCD-grouped
  // own keys from the KV cache (pipelined D = 96 kernel; null: from the k / v views): sequence b's
  // keys at cache[kv_slot[cu[b]], hk, kv_pos[cu[b]] + j, :] (slot_stride = Hkv * max_seq * D,
  // head stride hstride), rows D apart — the QKV epilogue then stores k / v to the cache only
  const int* kv_slot;
  const int* kv_pos;
  const bf16_t* kc;
  const bf16_t* vc;
  long long slot_stride;
};

// The (query block, head, sequence) a flash workgroup works on, from its place in the dispatch
// order. rev bit 0 (causal): the longest query blocks (most keys) first, so the kernel's tail is
// made of short blocks (longest-processing-time-first packing). rev bit 1: the query blocks of one
// (sequence, kv head) pair all run on one XCD. Workgroups are dealt round-robin over the 8 XCDs
// (linear ids g and g + 8 share one: observed dispatch, relied on for speed only), and every block
// of a pair re-reads that pair's K / V rows; grid order put a pair's blocks on all 8 XCDs, so each
// XCD's L2 fetched the same rows. Grouped, the pair's rows are fetched into one L2 and re-read
// there (pair-major per XCD: a few pairs' rows live at a time).
struct FaBlock {
  int qb, h, b;
};
__device__ __forceinline__ FaBlock fa_block(int rev, int causal, int G) {
  const int X = gridDim.x, Y = gridDim.y, Z = gridDim.z;
  const bool lpt = causal && (rev & 1);
  if ((rev & 2) && G >= 1 && Y % G == 0 && ((Y / G) * Z) % 8 == 0) {
    const int g = blockIdx.x + X * (blockIdx.y + Y * blockIdx.z);
    const int xcd = g & 7, s = g >> 3;
    const int per = X * G;                         // workgroups of one (sequence, kv head) pair
    const int pair = (s / per) * 8 + xcd, r = s % per;
    const int qi = r / G, gh = r % G;               // all G heads' longest blocks first
    const int hkv = Y / G;
    return FaBlock{lpt ? X - 1 - qi : qi, (pair % hkv) * G + gh, pair / hkv};
  }
  return FaBlock{lpt ? X - 1 - (int)blockIdx.x : (int)blockIdx.x, (int)blockIdx.y, (int)blockIdx.z};
}

// QH = 32-query halves per wave. QH = 2: each K fragment read from LDS feeds the S MFMAs of both
// halves and each transposed V fragment the O MFMAs of both, so LDS read bytes per FLOP halve (at
// QH = 1 the LDS reads of a tile take as long as its MFMAs); the two halves' softmax VALU work is
// independent of the other half's MFMAs, so the scheduler overlaps them inside one wave.
template <int D, int NW, int QH, typename T = BF16T>
__global__ void __launch_bounds__(64 * NW, QH == 1 ? 8 / NW : 1)
flash_attn_v2_kernel(const bf16_t* __restrict__ q, const bf16_t* __restrict__ k, const bf16_t* __restrict__ v,
                     int ldq, int ldk, int ldv, const int* __restrict__ cu, int H, int Hkv, int causal,
                     float c, bf16_t* __restrict__ o, int ldo, FaPrefix pre) {
  using C = FA2Cfg<D, NW, QH>;
  constexpr int KT = C::KT, NDS = D / 16, NDB = D / 32, CPR = C::CPR, LPT = C::LPT, NT = C::NT;
  constexpr bool EVEN = (KT * CPR) % NT == 0;  // every thread stages exactly LPT chunks
  extern __shared__ __attribute__((aligned(16))) char smem[];

  const FaBlock fb = fa_block(pre.rev, causal, H / Hkv);  // dispatch order: see fa_block
  const int b = fb.b, h = fb.h, qb = fb.qb;
  const int s0 = cu[b], L = cu[b + 1] - s0;
  const int q0 = qb * C::QB;
  if (q0 >= L) return;
  const int hk = h / (H / Hkv);
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int qr = lane & 31, hi = lane >> 5;
  const int wq0 = q0 + wid * C::QW;
  int qi[QH];
  bool qvalid[QH];
  bf16x8_t qf[QH][NDS];
  f32x16_t oacc[QH][NDB];
  float m_run[QH], l_part[QH];
#pragma unroll
  for (int j = 0; j < QH; ++j) {
    qi[j] = wq0 + 32 * j + qr;
    qvalid[j] = qi[j] < L;
#pragma unroll
    for (int ds = 0; ds < NDS; ++ds) {
      if (qvalid[j]) qf[j][ds] = *(const bf16x8_t*)(q + (size_t)(s0 + qi[j]) * ldq + h * D + ds * 16 + hi * 8);
      else qf[j][ds] = bf16x8_t{0, 0, 0, 0, 0, 0, 0, 0};
    }
#pragma unroll
    for (int i = 0; i < NDB; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) oacc[j][i][r] = 0.f;
    m_run[j] = -INFINITY;
    l_part[j] = 0.f;
  }

  const int P = pre.len, Lk = P + L;  // keys: [prefix | own]; own query i is key P + i
  const int kv_end = causal ? min(Lk, P + q0 + C::QB) : Lk;
  const int wave_end = causal ? min(Lk, P + wq0 + C::QW) : Lk;
  const int ntiles = (kv_end + KT - 1) / KT;

  const bf16_t* kbase_p = k + (size_t)s0 * ldk + hk * D;
  const bf16_t* vbase_p = v + (size_t)s0 * ldv + hk * D;
  if (pre.kv_slot) {  // own keys in the cache (the launcher passes ldk = ldv = D)
    const size_t off = (size_t)pre.kv_slot[s0] * pre.slot_stride + (size_t)hk * pre.hstride + (size_t)pre.kv_pos[s0] * D;
    kbase_p = pre.kc + off;
    vbase_p = pre.vc + off;
  }
  const bf16_t* kpre = pre.k + hk * pre.hstride;
  const bf16_t* vpre = pre.v + hk * pre.hstride;
  u32x4_t kst[LPT], vst[LPT];
  // Own-key tiles (all keys >= P) load through buffer resources rebuilt per tile on the scalar unit
  // (base = the tile's first key, num_records = the bytes left in the sequence: keys past the end
  // read 0), with fixed per-lane 32-bit offsets: no per-load 64-bit address math, bounds compare or
  // exec-mask branch (those were ~90 of the ~285 vector instructions of a tile).
  unsigned koff[LPT], voff[LPT];
#pragma unroll
  for (int i = 0; i < LPT; ++i) {
    const int idx = tid + NT * i, r = idx / CPR, cc = idx % CPR;
    const bool in = EVEN || idx < KT * CPR;
    koff[i] = in ? (unsigned)(r * ldk * 2 + cc * 16) : 0x80000000u;
    voff[i] = in ? (unsigned)(r * ldv * 2 + cc * 16) : 0x80000000u;
  }
  auto load_tile = [&](int t) {
    const int k0 = t * KT;
    if (k0 >= P) {
      const int o0 = k0 - P;
      const __amdgpu_buffer_rsrc_t rk = __builtin_amdgcn_make_buffer_rsrc(
          (void*)(kbase_p + (size_t)o0 * ldk), (short)0, (L - o0) * ldk * 2, 0x00020000);
      const __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc(
          (void*)(vbase_p + (size_t)o0 * ldv), (short)0, (L - o0) * ldv * 2, 0x00020000);
#pragma unroll
      for (int i = 0; i < LPT; ++i) {
        kst[i] = __builtin_amdgcn_raw_buffer_load_b128(rk, koff[i], 0, 0);
        vst[i] = __builtin_amdgcn_raw_buffer_load_b128(rv, voff[i], 0, 0);
      }
      return;
    }
#pragma unroll
    for (int i = 0; i < LPT; ++i) {
      const int idx = tid + NT * i, r = idx / CPR, cc = idx % CPR, key = t * KT + r;
      if ((EVEN || idx < KT * CPR) && key < Lk) {
        if (key >= P) {
          kst[i] = *(const u32x4_t*)(kbase_p + (size_t)(key - P) * ldk + cc * 8);
          vst[i] = *(const u32x4_t*)(vbase_p + (size_t)(key - P) * ldv + cc * 8);
        } else {
          kst[i] = *(const u32x4_t*)(kpre + (size_t)key * D + cc * 8);
          vst[i] = *(const u32x4_t*)(vpre + (size_t)key * D + cc * 8);
        }
      } else {
        kst[i] = u32x4_t{0, 0, 0, 0};
        vst[i] = u32x4_t{0, 0, 0, 0};
      }
    }
  };
  auto store_tile = [&](int buf) {
    char* sK = smem + buf * (C::KBUF + C::VBUF);
    char* sV = sK + C::KBUF;
#pragma unroll
    for (int i = 0; i < LPT; ++i) {
      const int idx = tid + NT * i, r = idx / CPR, cc = idx % CPR;
      if (EVEN || idx < KT * CPR) {
        *(u32x4_t*)(sK + r * C::KSTR + cc * 16) = kst[i];
        *(u32x4_t*)(sV + r * C::VSTR + cc * 16) = vst[i];
      }
    }
  };

  load_tile(0);
  store_tile(0);
  __syncthreads();

  for (int t = 0; t < ntiles; ++t) {
    const int cur = t & 1;
    if (t + 1 < ntiles) load_tile(t + 1);
    const int kb = t * KT;
    if (kb < wave_end) {
      const char* sK = smem + cur * (C::KBUF + C::VBUF);
      const char* sV = sK + C::KBUF;
      f32x16_t sacc[QH][2];
      // all K fragments of the tile first, then the MFMAs with the two 32-key halves interleaved:
      // one LDS round trip per tile instead of one per MFMA, and back-to-back MFMAs never depend
      // on each other (a fragment-at-a-time loop serialises LDS latency + MFMA latency 12 times).
      // D = 128 (16 fragments) batches per 32-key half, which keeps it within 256 VGPRs.
#pragma unroll
      for (int j = 0; j < QH; ++j)
#pragma unroll
        for (int hh = 0; hh < 2; ++hh)
#pragma unroll
          for (int r = 0; r < 16; ++r) sacc[j][hh][r] = 0.f;
      if constexpr (NDS <= 6) {
        bf16x8_t kfr[2][NDS];
#pragma unroll
        for (int hh = 0; hh < 2; ++hh)
#pragma unroll
          for (int ds = 0; ds < NDS; ++ds)
            kfr[hh][ds] = *(const bf16x8_t*)(sK + (hh * 32 + qr) * C::KSTR + ds * 32 + hi * 16);
#pragma unroll
        for (int ds = 0; ds < NDS; ++ds)
#pragma unroll
          for (int hh = 0; hh < 2; ++hh)
#pragma unroll
            for (int j = 0; j < QH; ++j) sacc[j][hh] = T::mma32(kfr[hh][ds], qf[j][ds], sacc[j][hh]);
        // pin that order: the register-pressure scheduler otherwise re-serialises read -> MFMA pairs
        __builtin_amdgcn_sched_group_barrier(0x100, 2 * NDS, 0);       // DS reads
        __builtin_amdgcn_sched_group_barrier(0x008, 2 * NDS * QH, 0);  // MFMAs
      } else {
#pragma unroll
        for (int hh = 0; hh < 2; ++hh) {
          bf16x8_t kfr[NDS];
#pragma unroll
          for (int ds = 0; ds < NDS; ++ds)
            kfr[ds] = *(const bf16x8_t*)(sK + (hh * 32 + qr) * C::KSTR + ds * 32 + hi * 16);
#pragma unroll
          for (int ds = 0; ds < NDS; ++ds)
#pragma unroll
            for (int j = 0; j < QH; ++j) sacc[j][hh] = T::mma32(kfr[ds], qf[j][ds], sacc[j][hh]);
          __builtin_amdgcn_sched_group_barrier(0x100, NDS, 0);
          __builtin_amdgcn_sched_group_barrier(0x008, NDS * QH, 0);
        }
      }
#pragma unroll
      for (int j = 0; j < QH; ++j) {
        if (kb + KT > Lk || (causal && kb + KT - 1 > P + wq0 + 32 * j)) {
#pragma unroll
          for (int hh = 0; hh < 2; ++hh)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
              const int key = kb + hh * 32 + 8 * (r >> 2) + 4 * hi + (r & 3);
              if (key >= Lk || (causal && key > P + qi[j])) sacc[j][hh][r] = -INFINITY;
            }
        }
        float mx = sacc[j][0][0];
#pragma unroll
        for (int r = 1; r < 16; ++r) mx = fmaxf(mx, sacc[j][0][r]);
#pragma unroll
        for (int r = 0; r < 16; ++r) mx = fmaxf(mx, sacc[j][1][r]);
        mx = max_xhalf(mx);
        const float m_new = fmaxf(m_run[j], mx);
        const float m_use = (m_new == -INFINITY) ? 0.f : m_new;
        if (__any(m_new > m_run[j])) {
          const float alpha = exp2f((m_run[j] - m_use) * c);
          l_part[j] *= alpha;
#pragma unroll
          for (int i = 0; i < NDB; ++i) oacc[j][i] *= alpha;
        }
        m_run[j] = m_new;
        const float mc = -m_use * c;
        float psum = 0.f;
#pragma unroll
        for (int hh = 0; hh < 2; ++hh)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const float p = __builtin_amdgcn_exp2f(fmaf(sacc[j][hh][r], c, mc));  // raw v_exp_f32
            sacc[j][hh][r] = p;
            psum += p;
          }
        l_part[j] += psum;
      }

      // O^T += V^T P^T over 4 k-steps of 16 keys: slot (hi, j) -> key 16kc + 8(j>>2) + 4hi + (j&3)
#pragma unroll
      for (int kc = 0; kc < 4; ++kc) {
        const int hh = kc >> 1, cb = (kc & 1) * 8;
        bf16x8_t pb[QH];
#pragma unroll
        for (int j = 0; j < QH; ++j) {
          const u32x4_t pw = u32x4_t{T::pack2(sacc[j][hh][cb], sacc[j][hh][cb + 1]),
                                     T::pack2(sacc[j][hh][cb + 2], sacc[j][hh][cb + 3]),
                                     T::pack2(sacc[j][hh][cb + 4], sacc[j][hh][cb + 5]),
                                     T::pack2(sacc[j][hh][cb + 6], sacc[j][hh][cb + 7])};
          pb[j] = __builtin_bit_cast(bf16x8_t, pw);
        }
        const int g = lane >> 4, li = lane & 15;
        const int row0 = kc * 16 + 4 * (g >> 1) + (li >> 2);
#pragma unroll
        for (int db = 0; db < NDB; ++db) {
          const int col = db * 32 + 16 * (g & 1) + 4 * (li & 3);
          const s16x4_t lo = lds_read_tr16(sV + row0 * C::VSTR + col * 2);
          const s16x4_t hi8 = lds_read_tr16(sV + (row0 + 8) * C::VSTR + col * 2);
          const bf16x8_t va = bf16x8_t{lo[0], lo[1], lo[2], lo[3], hi8[0], hi8[1], hi8[2], hi8[3]};
#pragma unroll
          for (int j = 0; j < QH; ++j) oacc[j][db] = T::mma32(va, pb[j], oacc[j][db]);
        }
      }
    }
    if (t + 1 < ntiles) store_tile(cur ^ 1);
    __syncthreads();
  }

#pragma unroll
  for (int j = 0; j < QH; ++j) {
    const float l_tot = sum_xhalf(l_part[j]);
    const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
    if (qvalid[j]) {
      bf16_t* orow = o + (size_t)(s0 + qi[j]) * ldo + h * D;
#pragma unroll
      for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const int d = db * 32 + 8 * g + 4 * hi;
          *(u32x2_t*)(orow + d) = u32x2_t{T::pack2(oacc[j][db][4 * g] * inv, oacc[j][db][4 * g + 1] * inv),
                                          T::pack2(oacc[j][db][4 * g + 2] * inv, oacc[j][db][4 * g + 3] * inv)};
        }
    }
  }
}

// ------------------------------------------------------------------------------------------
// flash_attn_pipe: the same math and fragment layouts as flash_attn_v2<D, 4, 1>, software-pipelined
// one tile deep (guide T15): the S MFMAs of tile t + 1 are issued before the softmax + P·V of tile t,
// so the softmax VALU work never waits on the MFMA results it follows (RAW) and the matrix pipe has
// independent work while a wave is in its exp/max/pack stretch. Three LDS tile buffers: tile t
// (P·V), t + 1 (S) and t + 2 (being written); one barrier per tile.
//
// SPEC = true: speculative softmax against a deferred running max (guide T13). The round-2 form put
// the S MFMAs of tile t + 1, the max / rescale branch and the exp / pack / P·V of tile t in separate
// basic blocks, so the compiler could not interleave the softmax VALU of t with the S MFMAs of t + 1
// (ISA: a 12-MFMA block with no VALU, then a 116-VALU + 32-exp block; the SIMD ran them back to back).
// With SPEC, an unmasked tile (every key visible to every query of the wave) is one straight-line
// block: S(t + 1) MFMAs interleaved with max(t), p = exp2(s·c - m_run·c) against the STALE running
// max, row sums and the bf16 pack. The reference max of a query moves only when its tile max
// overshoots it by SPEC_TAU (log2 units of p; the first tile always does), branch-free per lane;
// only the O rescale that such a move needs is a (rare, wave-uniform) branch before P·V. Masked
// tiles (causal diagonal, sequence end) take the exact path. p <= 2^SPEC_TAU keeps the fp32 sums
// and the bf16 P exact in relative terms; the result is normalised by the same l, so only rounding
// differs from SPEC = false.
//
// DMA = true (D = 96, shared prefix a multiple of 64 keys): K / V tiles arrive by LDS-DMA
// (buffer_load ... lds) instead of register staging, in rings that give each tile TWO steps of
// latency cover (staging gave one, and a step is ~0.5 us against 1-2 us of loaded HBM / L2
// latency): at the start of step t the wave issues K(t + 3) into the slot S(t) read in step t - 1
// and V(t + 2) into the slot P·V(t - 1) read; before the step's barrier it waits for K(t + 2) and
// V(t + 1) (vmcnt(6): the 3 + 3 pieces of step t may stay in flight). K rows are unpadded (192 B)
// with 16-B chunk c of row r at slot c ^ ((r >> 2) & 3) — applied on the DMA source side — so the
// 16 rows one ds_read_b128 lane group reads hit 16 distinct bank slots; V keeps its linear rows.
// No staging registers, no ds_write, no per-tile address VALU. Past the last tile the pieces are
// issued at an out-of-range offset (no memory traffic, zeros into a free slot): uniform counts.
constexpr float SPEC_TAU = 8.f;

// Three 1-KiB LDS-DMA pieces (buffer_load_dwordx4 ... lds) into LDS lds, lds + 1 KiB, lds + 2 KiB,
// lane l's 16 B from rsrc + v_i + soff. Inline asm on purpose: through the builtin, hipcc treats the
// transposed V reads (ds_read_b64_tr_b16) as possibly aliasing the DMA and drains vmcnt to 0 before
// them, which would cancel the prefetch; these ops are invisible to its counters, and the kernel
// waits for them with explicit vmcnt. No VGPR destination (register-safe); M0 is saved and
// restored inside the statement; s_nop 4 covers an SGPR operand fresh from v_readfirstlane.
__device__ __forceinline__ void dma3_lds(__amdgpu_buffer_rsrc_t rs, unsigned lds, unsigned v0, unsigned v1,
                                         unsigned v2, int soff) {
  unsigned keep;
  asm volatile(
      "s_nop 4\n\t"
      "s_mov_b32 %0, m0\n\t"
      "s_mov_b32 m0, %5\n\t"
      "s_nop 0\n\t"
      "buffer_load_dwordx4 %1, %4, %6 offen lds\n\t"
      "s_add_u32 m0, m0, 0x400\n\t"
      "s_nop 0\n\t"
      "buffer_load_dwordx4 %2, %4, %6 offen lds\n\t"
      "s_add_u32 m0, m0, 0x400\n\t"
      "s_nop 0\n\t"
      "buffer_load_dwordx4 %3, %4, %6 offen lds\n\t"
      "s_mov_b32 m0, %0"
      : "=&s"(keep)
      : "v"(v0), "v"(v1), "v"(v2), "s"(rs), "s"(lds), "s"(soff)
      : "memory", "scc");
}

// Two such pieces.
__device__ __forceinline__ void dma2_lds(__amdgpu_buffer_rsrc_t rs, unsigned lds, unsigned v0, unsigned v1) {
  unsigned keep;
  asm volatile(
      "s_nop 4\n\t"
      "s_mov_b32 %0, m0\n\t"
      "s_mov_b32 m0, %4\n\t"
      "s_nop 0\n\t"
      "buffer_load_dwordx4 %1, %3, 0 offen lds\n\t"
      "s_add_u32 m0, m0, 0x400\n\t"
      "s_nop 0\n\t"
      "buffer_load_dwordx4 %2, %3, 0 offen lds\n\t"
      "s_mov_b32 m0, %0"
      : "=&s"(keep)
      : "v"(v0), "v"(v1), "s"(rs), "s"(lds)
      : "memory", "scc");
}

// Bidirectional attention of the encoders (D = 64, no prefix): flash_attn_v2<64, 4, 1>'s tiles and arithmetic, with Q, K and V
// by LDS-DMA, in rings of three K and two V tiles: the first of them are on their way with the queries, a K tile has two steps
// to arrive in, and 40 KB and 128 registers let a CU have four workgroups (a third V tile, three workgroups: 92 us for 86). One
// barrier a tile. 16-B chunk c of row r is at c ^ (r >> 1) in a K (and Q, O) tile and at c ^ ((r & 2) << 1) in a V tile: both
// reads are free of bank conflicts. A wave without queries only moves its part of the tiles. Rows go out whole, through LDS.
// The maximum that weights are relative to moves when it is 2^SPEC_TAU off (rescaling O takes a quarter of a tile's vector
// instructions, and some row of 32 has a new maximum at most tiles of a short sequence). bf16: all of them 2^-SPEC_TAU times
// that, so that sums of values near the type's largest don't leave fp32 (fp16 has no range below for it, and values of 2^16 at most).
// Bound by the vector ALU (of 64 x 512 rows, 16 heads: 63 % of its cycles, the MFMAs 30 %) and by what is left of a round for
// ragged sequences. us, by registers one tile ahead with two workgroups a CU / this: 80 texts of 61 - 512 rows, 16 heads, fp16
// 85 / 70; 64 of 512 115 / 97 (710 TF); 12 heads, bf16: 80 of 61 - 512 67 / 55, 64 of 512 85 / 73; one of 400 rows 11.4 / 9.4.
template <typename T>
__global__ void __launch_bounds__(256, 4)
flash_attn_enc_kernel(const bf16_t* __restrict__ q, const bf16_t* __restrict__ k, const bf16_t* __restrict__ v, int ldq, int ldk,
                      int ldv, const int* __restrict__ cu, int H, int Hkv, float c, bf16_t* __restrict__ o, int ldo, int rev) {
  constexpr int D = 64, KT = 64, RB = D * 2, TILE = KT * RB;
  __shared__ __attribute__((aligned(16))) char smem[5 * TILE];
  typedef __attribute__((address_space(3))) char lds_char;  // LDS byte offset, not the flat address

  const FaBlock fb = fa_block(rev, 0, H / Hkv);
  const int b = fb.b, h = fb.h, q0 = fb.qb * 128;
  const int s0 = __builtin_amdgcn_readfirstlane(cu[b]), L = __builtin_amdgcn_readfirstlane(cu[b + 1]) - s0;
  if (q0 >= L) return;
  const int hk = h / (H / Hkv);
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int qr = lane & 31, hi = lane >> 5;
  const int wq0 = q0 + w * 32;
  const bool live = wq0 < L;
  const int ntiles = (L + KT - 1) / KT;
  const unsigned ring = (unsigned)(size_t)(lds_char*)smem;
  auto rows_of = [&](const bf16_t* base, int ld, int r0, int n) __attribute__((always_inline)) {  // rows past the sequence: none
    const int rows = __builtin_amdgcn_readfirstlane(max(0, min(n, L - r0)));
    return __builtin_amdgcn_make_buffer_rsrc((void*)(base + (size_t)(s0 + r0) * ld), (short)0, rows * ld * 2, 0x00020000);
  };
  // piece i of this wave: rows 16 w + 8 i + lane / 8 of a K or V tile (and of the wave's 32 queries, 8 i + lane / 8)
  unsigned kx[2], vx[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int r = w * 16 + i * 8 + (lane >> 3);
    kx[i] = (unsigned)(r * ldk * 2 + (((lane & 7) ^ ((r >> 1) & 7)) << 4));
    vx[i] = (unsigned)(r * ldv * 2 + (((lane & 7) ^ ((r & 2) << 1)) << 4));
  }
  auto issue = [&](int t, int stage) __attribute__((always_inline)) {
    dma2_lds(rows_of(k + hk * D, ldk, t * KT, KT), __builtin_amdgcn_readfirstlane(ring + stage * TILE + w * 2048), kx[0], kx[1]);
  };
  auto issue_v = [&](int t) __attribute__((always_inline)) {
    dma2_lds(rows_of(v + hk * D, ldv, t * KT, KT), __builtin_amdgcn_readfirstlane(ring + (3 + (t & 1)) * TILE + w * 2048), vx[0], vx[1]);
  };
  char* mine = smem + w * 4096;  // this wave's output
  const int qat = 2 * TILE + (w < 2 ? w : w + 2) * 4096;  // its queries: in the third K and the second V tile
  {
    const __amdgpu_buffer_rsrc_t rq = rows_of(q + h * D, ldq, wq0, 32);
    const unsigned dst = __builtin_amdgcn_readfirstlane(ring + qat);
    unsigned x[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = i * 8 + (lane >> 3);
      x[i] = (unsigned)(r * ldq * 2 + (((lane & 7) ^ ((r >> 1) & 7)) << 4));
    }
    dma2_lds(rq, dst, x[0], x[1]);
    dma2_lds(rq, dst + 2048, x[2], x[3]);
  }
  issue(0, 0);
  issue_v(0);
  issue(1, 1);
  int xo[4];  // chunk 2 ds + hi of row qr
#pragma unroll
  for (int ds = 0; ds < 4; ++ds) xo[ds] = qr * RB + (((2 * ds + hi) ^ ((qr >> 1) & 7)) << 4);
  // transposed V reads of a 16-key step: row 4 (g >> 1) + li / 4 (and 8 on), columns 32 db + 16 (g & 1) + 4 (li & 3)
  const int g = lane >> 4, li = lane & 15;
  int vo[2];
#pragma unroll
  for (int db = 0; db < 2; ++db)
    vo[db] = (4 * (g >> 1) + (li >> 2)) * RB + ((db ^ (li >> 3)) << 6) + (g & 1) * 32 + (li & 3) * 8;
  f32x16_t oacc[2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) oacc[i][r] = 0.f;
  float m_run = -INFINITY, l_part = 0.f;
  asm volatile("s_waitcnt vmcnt(6)" ::: "memory");  // the queries; the tiles may be on their way
  bf16x8_t qf[4];
#pragma unroll
  for (int ds = 0; ds < 4; ++ds) qf[ds] = *(const bf16x8_t*)(smem + qat + xo[ds]);

  int rd = 0;
  for (int t = 0; t < ntiles; ++t) {
    // this wave's part of tile t is in (K of t + 1 newer); after the barrier everyone's, and the places of t - 1 are free
    asm volatile("s_waitcnt vmcnt(2) lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    issue_v(t + 1);
    issue(t + 2, rd == 0 ? 2 : rd - 1);
    if (live) {
      const char* sK = smem + rd * TILE;
      const char* sV = smem + (3 + (t & 1)) * TILE;
      f32x16_t sacc[2];
#pragma unroll
      for (int hh = 0; hh < 2; ++hh)
#pragma unroll
        for (int r = 0; r < 16; ++r) sacc[hh][r] = 0.f;
      bf16x8_t kfr[2][4];
#pragma unroll
      for (int hh = 0; hh < 2; ++hh)
#pragma unroll
        for (int ds = 0; ds < 4; ++ds) kfr[hh][ds] = *(const bf16x8_t*)(sK + hh * 32 * RB + xo[ds]);
#pragma unroll
      for (int ds = 0; ds < 4; ++ds)
#pragma unroll
        for (int hh = 0; hh < 2; ++hh) sacc[hh] = T::mma32(kfr[hh][ds], qf[ds], sacc[hh]);
      __builtin_amdgcn_sched_group_barrier(0x100, 8, 0);  // DS reads
      __builtin_amdgcn_sched_group_barrier(0x008, 8, 0);  // MFMAs
      if (t * KT + KT > L) {
#pragma unroll
        for (int hh = 0; hh < 2; ++hh)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            if (t * KT + hh * 32 + 8 * (r >> 2) + 4 * hi + (r & 3) >= L) sacc[hh][r] = -INFINITY;
      }
      float mx = sacc[0][0];
#pragma unroll
      for (int r = 1; r < 16; ++r) mx = fmaxf(mx, sacc[0][r]);
#pragma unroll
      for (int r = 0; r < 16; ++r) mx = fmaxf(mx, sacc[1][r]);
      mx = max_xhalf(mx);
      if (__any((mx - m_run) * c > SPEC_TAU)) {  // (weights of up to 2^SPEC_TAU are as exact)
        const float m_new = fmaxf(m_run, mx);
        const float alpha = exp2f((m_run - (m_new == -INFINITY ? 0.f : m_new)) * c);  // (scores of -inf only: 0, not NaN)
        m_run = m_new;
        l_part *= alpha;
#pragma unroll
        for (int i = 0; i < 2; ++i) oacc[i] *= alpha;
      }
      const float mc = m_run == -INFINITY ? 0.f : fmaf(-m_run, c, T::kF16 ? 0.f : -SPEC_TAU);
      float psum = 0.f;
#pragma unroll
      for (int hh = 0; hh < 2; ++hh)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const float p = __builtin_amdgcn_exp2f(fmaf(sacc[hh][r], c, mc));
          sacc[hh][r] = p;
          psum += p;
        }
      l_part += psum;
      // O^T += V^T P^T over 4 steps of 16 keys: slot (hi, j) -> key 16 kc + 8 (j >> 2) + 4 hi + (j & 3)
#pragma unroll
      for (int kc = 0; kc < 4; ++kc) {
        const int hh = kc >> 1, cb = (kc & 1) * 8;
        const bf16x8_t pb = __builtin_bit_cast(
            bf16x8_t, u32x4_t{T::pack2(sacc[hh][cb], sacc[hh][cb + 1]), T::pack2(sacc[hh][cb + 2], sacc[hh][cb + 3]),
                              T::pack2(sacc[hh][cb + 4], sacc[hh][cb + 5]), T::pack2(sacc[hh][cb + 6], sacc[hh][cb + 7])});
#pragma unroll
        for (int db = 0; db < 2; ++db) {
          const s16x4_t lo = lds_read_tr16(sV + kc * 16 * RB + vo[db]);
          const s16x4_t up = lds_read_tr16(sV + (kc * 16 + 8) * RB + vo[db]);
          oacc[db] = T::mma32(bf16x8_t{lo[0], lo[1], lo[2], lo[3], up[0], up[1], up[2], up[3]}, pb, oacc[db]);
        }
      }
    }
    rd = rd == 2 ? 0 : rd + 1;
  }
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");  // (tiles past the end write zeros)
  __builtin_amdgcn_s_barrier();
  if (!live) return;
  const float l_tot = sum_xhalf(l_part);
  const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
#pragma unroll
  for (int db = 0; db < 2; ++db)
#pragma unroll
    for (int e = 0; e < 4; ++e)
      *(u32x2_t*)(mine + qr * RB + (((db * 4 + e) ^ ((qr >> 1) & 7)) << 4) + hi * 8) =
          u32x2_t{T::pack2(oacc[db][4 * e] * inv, oacc[db][4 * e + 1] * inv),
                  T::pack2(oacc[db][4 * e + 2] * inv, oacc[db][4 * e + 3] * inv)};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = i * 8 + (lane >> 3);
    const u32x4_t row = *(const u32x4_t*)(mine + r * RB + (((lane & 7) ^ ((r >> 1) & 7)) << 4));
    if (wq0 + r < L) *(u32x4_t*)(o + (size_t)(s0 + wq0 + r) * ldo + h * D + (lane & 7) * 8) = row;
  }
}

template <int D, bool SPEC, bool DMA>
__global__ void __launch_bounds__(256, 2)
flash_attn_pipe_kernel(const bf16_t* __restrict__ q, const bf16_t* __restrict__ k, const bf16_t* __restrict__ v,
                       int ldq, int ldk, int ldv, const int* __restrict__ cu, int H, int Hkv, int causal,
                       float c, bf16_t* __restrict__ o, int ldo, FaPrefix pre) {
  using C = FA2Cfg<D, 4, 1>;
  constexpr int KT = C::KT, NDS = D / 16, NDB = D / 32, CPR = C::CPR, LPT = C::LPT, NT = C::NT;
  constexpr bool EVEN = (KT * CPR) % NT == 0;
  static_assert(NDS <= 6, "pipelined flash: D <= 96");
  static_assert(!DMA || (D == 96 && C::VSTR == D * 2), "DMA tiles: D = 96 (linear V rows)");
  constexpr int KSTR = DMA ? D * 2 : C::KSTR, KBUF = KT * KSTR, TBUF = KBUF + C::VBUF;
  extern __shared__ __attribute__((aligned(16))) char smem[];

  const FaBlock fb = fa_block(pre.rev, causal, H / Hkv);  // dispatch order: see fa_block
  const int b = fb.b, h = fb.h, qb = fb.qb;
  const int s0 = cu[b], L = cu[b + 1] - s0;
  const int q0 = qb * C::QB;
  if (q0 >= L) return;
  const int hk = h / (H / Hkv);
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int qr = lane & 31, hi = lane >> 5;
  const int wq0 = q0 + wid * C::QW;
  const int qi = wq0 + qr;
  const bool qvalid = qi < L;
  bf16x8_t qf[NDS];
#pragma unroll
  for (int ds = 0; ds < NDS; ++ds)
    qf[ds] = qvalid ? *(const bf16x8_t*)(q + (size_t)(s0 + qi) * ldq + h * D + ds * 16 + hi * 8)
                    : bf16x8_t{0, 0, 0, 0, 0, 0, 0, 0};
  f32x16_t oacc[NDB];
#pragma unroll
  for (int i = 0; i < NDB; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) oacc[i][r] = 0.f;
  float m_run = -INFINITY, l_part = 0.f;

  const int P = pre.len, Lk = P + L;
  const int kv_end = causal ? min(Lk, P + q0 + C::QB) : Lk;
  const int wave_end = causal ? min(Lk, P + wq0 + C::QW) : Lk;
  const int ntiles = (kv_end + KT - 1) / KT;

  const bf16_t* kbase_p = k + (size_t)s0 * ldk + hk * D;
  const bf16_t* vbase_p = v + (size_t)s0 * ldv + hk * D;
  if (pre.kv_slot) {  // own keys in the cache (the launcher passes ldk = ldv = D)
    const size_t off = (size_t)pre.kv_slot[s0] * pre.slot_stride + (size_t)hk * pre.hstride + (size_t)pre.kv_pos[s0] * D;
    kbase_p = pre.kc + off;
    vbase_p = pre.vc + off;
  }
  const bf16_t* kpre = pre.k + hk * pre.hstride;
  const bf16_t* vpre = pre.v + hk * pre.hstride;
  auto buf_of = [&](int t) { return smem + (t % 3) * TBUF; };
  u32x4_t kst[LPT], vst[LPT];
  unsigned koff[LPT], voff[LPT];
#pragma unroll
  for (int i = 0; i < LPT; ++i) {
    const int idx = tid + NT * i, r = idx / CPR, cc = idx % CPR;
    const bool in = EVEN || idx < KT * CPR;
    koff[i] = in ? (unsigned)(r * ldk * 2 + cc * 16) : 0x80000000u;
    voff[i] = in ? (unsigned)(r * ldv * 2 + cc * 16) : 0x80000000u;
  }
  // DMA pieces: wave wid fills LDS 16-B positions (3 wid + i) * 64 + lane of a tile (768 = 64 rows x
  // 12 chunks): row r, slot sl; K slot sl holds chunk sl ^ ((r >> 2) & 3), V slot sl chunk sl
  unsigned dkr[3], dkc[3], dvc[3];
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const int pos = (wid * 3 + i) * 64 + lane, r = pos / 12, sl = pos % 12;
    dkr[i] = r;
    dkc[i] = (sl ^ ((r >> 2) & 3)) * 16;
    dvc[i] = sl * 16;
  }
  // tile t's K (KV = false) or V pieces into slot t % 3; t >= ntiles: out of range, no traffic
  auto dma_tile = [&](int t, bool is_v) {
    const int k0 = t * KT;
    const bf16_t* base = is_v ? vbase_p : kbase_p;
    const bf16_t* pbase = is_v ? vpre : kpre;
    const int ld = is_v ? ldv : ldk;
    const bool own = k0 >= P;
    const int o0 = k0 - P;
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(own ? base + (size_t)o0 * ld : pbase + (size_t)k0 * D), (short)0,
        own ? max(L - o0, 0) * ld * 2 : (P - k0) * D * 2, 0x00020000);
    const unsigned rstride = own ? ld * 2 : D * 2;
    const int soff = t < ntiles ? 0 : 0x7ffffff0;
    typedef __attribute__((address_space(3))) char lds_char;  // LDS byte offset, not the flat address
    const unsigned dst = (unsigned)(size_t)(lds_char*)(buf_of(t) + (is_v ? KBUF : 0)) + wid * 3 * 1024;
    dma3_lds(rs, __builtin_amdgcn_readfirstlane(dst), dkr[0] * rstride + (is_v ? dvc[0] : dkc[0]),
             dkr[1] * rstride + (is_v ? dvc[1] : dkc[1]), dkr[2] * rstride + (is_v ? dvc[2] : dkc[2]), soff);
  };
  auto load_tile = [&](int t) {
    const int k0 = t * KT;
    if (k0 >= P) {
      const int o0 = k0 - P;
      const __amdgpu_buffer_rsrc_t rk = __builtin_amdgcn_make_buffer_rsrc(
          (void*)(kbase_p + (size_t)o0 * ldk), (short)0, (L - o0) * ldk * 2, 0x00020000);
      const __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc(
          (void*)(vbase_p + (size_t)o0 * ldv), (short)0, (L - o0) * ldv * 2, 0x00020000);
#pragma unroll
      for (int i = 0; i < LPT; ++i) {
        kst[i] = __builtin_amdgcn_raw_buffer_load_b128(rk, koff[i], 0, 0);
        vst[i] = __builtin_amdgcn_raw_buffer_load_b128(rv, voff[i], 0, 0);
      }
      return;
    }
#pragma unroll
    for (int i = 0; i < LPT; ++i) {
      const int idx = tid + NT * i, r = idx / CPR, cc = idx % CPR, key = t * KT + r;
      if ((EVEN || idx < KT * CPR) && key < Lk) {
        if (key >= P) {
          kst[i] = *(const u32x4_t*)(kbase_p + (size_t)(key - P) * ldk + cc * 8);
          vst[i] = *(const u32x4_t*)(vbase_p + (size_t)(key - P) * ldv + cc * 8);
        } else {
          kst[i] = *(const u32x4_t*)(kpre + (size_t)key * D + cc * 8);
          vst[i] = *(const u32x4_t*)(vpre + (size_t)key * D + cc * 8);
        }
      } else {
        kst[i] = u32x4_t{0, 0, 0, 0};
        vst[i] = u32x4_t{0, 0, 0, 0};
      }
    }
  };
  auto store_tile = [&](int t) {
    char* sK = buf_of(t);
    char* sV = sK + C::KBUF;
#pragma unroll
    for (int i = 0; i < LPT; ++i) {
      const int idx = tid + NT * i, r = idx / CPR, cc = idx % CPR;
      if (EVEN || idx < KT * CPR) {
        *(u32x4_t*)(sK + r * C::KSTR + cc * 16) = kst[i];
        *(u32x4_t*)(sV + r * C::VSTR + cc * 16) = vst[i];
      }
    }
  };
  // byte offset of K fragment (32-key half hh, 16-dim step ds) of this lane in a K tile
  auto kfrag = [&](int hh, int ds) -> int {
    if constexpr (DMA) return (hh * 32 + qr) * KSTR + (((2 * ds + hi) ^ ((qr >> 2) & 3)) << 4);
    else return (hh * 32 + qr) * KSTR + ds * 32 + hi * 16;
  };
  // S^T of tile t: all K fragments, then the MFMAs (two independent accumulation chains)
  auto s_tile = [&](int t, f32x16_t (&sa)[2]) {
    const char* sK = buf_of(t);
#pragma unroll
    for (int hh = 0; hh < 2; ++hh)
#pragma unroll
      for (int r = 0; r < 16; ++r) sa[hh][r] = 0.f;
    if constexpr (SPEC) {
      // one 32-key half at a time: 6 fragments (24 VGPRs) live instead of 12 beside the softmax of t
#pragma unroll
      for (int hh = 0; hh < 2; ++hh) {
        bf16x8_t kfr[NDS];
#pragma unroll
        for (int ds = 0; ds < NDS; ++ds)
          kfr[ds] = *(const bf16x8_t*)(sK + kfrag(hh, ds));
#pragma unroll
        for (int ds = 0; ds < NDS; ++ds) sa[hh] = mfma32(kfr[ds], qf[ds], sa[hh]);
      }
    } else {
      bf16x8_t kfr[2][NDS];
#pragma unroll
      for (int hh = 0; hh < 2; ++hh)
#pragma unroll
        for (int ds = 0; ds < NDS; ++ds)
          kfr[hh][ds] = *(const bf16x8_t*)(sK + kfrag(hh, ds));
#pragma unroll
      for (int ds = 0; ds < NDS; ++ds)
#pragma unroll
        for (int hh = 0; hh < 2; ++hh) sa[hh] = mfma32(kfr[hh][ds], qf[ds], sa[hh]);
    }
  };
  // O^T += V^T P^T of tile t, P packed to bf16 (kc = 16-key step)
  auto pv_tile = [&](int t, const u32x4_t (&pw)[4]) {
    const char* sV = buf_of(t) + KBUF;
#pragma unroll
    for (int kc = 0; kc < 4; ++kc) {
      const bf16x8_t pb = __builtin_bit_cast(bf16x8_t, pw[kc]);
      const int g = lane >> 4, li = lane & 15;
      const int row0 = kc * 16 + 4 * (g >> 1) + (li >> 2);
#pragma unroll
      for (int db = 0; db < NDB; ++db) {
        const int col = db * 32 + 16 * (g & 1) + 4 * (li & 3);
        const s16x4_t lo = lds_read_tr16(sV + row0 * C::VSTR + col * 2);
        const s16x4_t hi8 = lds_read_tr16(sV + (row0 + 8) * C::VSTR + col * 2);
        const bf16x8_t va = bf16x8_t{lo[0], lo[1], lo[2], lo[3], hi8[0], hi8[1], hi8[2], hi8[3]};
        oacc[db] = mfma32(va, pb, oacc[db]);
      }
    }
  };
  // mask + online softmax + O^T += V^T P^T of tile t
  auto finish = [&](int t, f32x16_t (&sa)[2]) {
    const int kb = t * KT;
    if (kb + KT > Lk || (causal && kb + KT - 1 > P + wq0)) {
#pragma unroll
      for (int hh = 0; hh < 2; ++hh)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int key = kb + hh * 32 + 8 * (r >> 2) + 4 * hi + (r & 3);
          if (key >= Lk || (causal && key > P + qi)) sa[hh][r] = -INFINITY;
        }
    }
    float mx = sa[0][0];
#pragma unroll
    for (int r = 1; r < 16; ++r) mx = fmaxf(mx, sa[0][r]);
#pragma unroll
    for (int r = 0; r < 16; ++r) mx = fmaxf(mx, sa[1][r]);
    mx = max_xhalf(mx);
    const float m_new = fmaxf(m_run, mx);
    const float m_use = (m_new == -INFINITY) ? 0.f : m_new;
    if (__any(m_new > m_run)) {
      const float alpha = exp2f((m_run - m_use) * c);
      l_part *= alpha;
#pragma unroll
      for (int i = 0; i < NDB; ++i) oacc[i] *= alpha;
    }
    m_run = m_new;
    const float mc = -m_use * c;
    float psum = 0.f;
#pragma unroll
    for (int hh = 0; hh < 2; ++hh)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float pv = __builtin_amdgcn_exp2f(fmaf(sa[hh][r], c, mc));
        sa[hh][r] = pv;
        psum += pv;
      }
    l_part += psum;
    u32x4_t pw[4];
#pragma unroll
    for (int kc = 0; kc < 4; ++kc) {
      const int hh = kc >> 1, cb = (kc & 1) * 8;
      pw[kc] = u32x4_t{pack_bf2(sa[hh][cb], sa[hh][cb + 1]), pack_bf2(sa[hh][cb + 2], sa[hh][cb + 3]),
                       pack_bf2(sa[hh][cb + 4], sa[hh][cb + 5]), pack_bf2(sa[hh][cb + 6], sa[hh][cb + 7])};
    }
    pv_tile(t, pw);
  };
  // unmasked tile with a deferred running max (SPEC; see above the kernel). The caller issues the S
  // MFMAs of tile t + 1 just before, in the same basic block.
  const float spec_thr = SPEC_TAU / c;  // raw-score headroom above the reference max
  auto finish_spec = [&](int t, f32x16_t (&sa)[2]) {
    float mx = fmaxf(sa[0][0], sa[0][1]);
#pragma unroll
    for (int r = 2; r < 16; ++r) mx = fmaxf(mx, sa[0][r]);
#pragma unroll
    for (int r = 0; r < 16; ++r) mx = fmaxf(mx, sa[1][r]);
    mx = max_xhalf(mx);
    // the reference max moves only when the tile max overshoots it by SPEC_TAU (log2 units of p):
    // p <= 2^SPEC_TAU; first tile: m_run = -inf -> m_new = mx, alpha = 0
    const bool up = mx > m_run + spec_thr;
    const float m_new = up ? mx : m_run;
    const float alpha = exp2f((m_run - m_new) * c);
    const float mcs = -m_new * c;
    float psum = 0.f;
#pragma unroll
    for (int hh = 0; hh < 2; ++hh)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float pv = __builtin_amdgcn_exp2f(fmaf(sa[hh][r], c, mcs));
        sa[hh][r] = pv;
        psum += pv;
      }
    u32x4_t pw[4];
#pragma unroll
    for (int kc = 0; kc < 4; ++kc) {
      const int hh = kc >> 1, cb = (kc & 1) * 8;
      pw[kc] = u32x4_t{pack_bf2(sa[hh][cb], sa[hh][cb + 1]), pack_bf2(sa[hh][cb + 2], sa[hh][cb + 3]),
                       pack_bf2(sa[hh][cb + 4], sa[hh][cb + 5]), pack_bf2(sa[hh][cb + 6], sa[hh][cb + 7])};
    }
    l_part = l_part * alpha + psum;
    m_run = m_new;
    // materialise P and l here: otherwise the compiler sinks the exp / pack work past the branch
    // into the P·V block, away from the S MFMAs of t + 1 it is meant to run beside
#pragma unroll
    for (int kc = 0; kc < 4; ++kc) asm volatile("" : "+v"(pw[kc]));
    asm volatile("" : "+v"(l_part));
    if (__any(up)) {  // rare after the first tiles: O moves to the new reference
#pragma unroll
      for (int i = 0; i < NDB; ++i) oacc[i] *= alpha;
    }
    pv_tile(t, pw);
  };

  f32x16_t SA[2], SB[2];
  auto barrier = [&]() {  // LDS reads done + every wave here (no vmcnt drain: DMA stays in flight)
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
  };
  if constexpr (DMA) {
    dma_tile(0, false); dma_tile(0, true); dma_tile(1, false); dma_tile(1, true); dma_tile(2, false);
    asm volatile("s_waitcnt vmcnt(6)" ::: "memory");  // K0 V0 K1 landed (V1 K2 may fly)
    barrier();
    s_tile(0, SA);
    barrier();  // every wave's S(0) reads are done before K(3) refills slot 0
  } else {
    load_tile(0);
    store_tile(0);
    if (ntiles > 1) {
      load_tile(1);
      store_tile(1);
    }
    __syncthreads();
    if (ntiles > 2) load_tile(2);
    s_tile(0, SA);
  }
  auto step = [&](int t, f32x16_t (&cur)[2], f32x16_t (&nxt)[2]) {
    if constexpr (DMA) {
      dma_tile(t + 3, false);  // slot of K(t): read by S(t) in step t - 1
      dma_tile(t + 2, true);   // slot of V(t - 1): read by P·V(t - 1) in step t - 1
    }
    const int kb = t * KT;
    const bool nx = t + 1 < ntiles && (t + 1) * KT < wave_end;
    // unmasked for every query of this wave (the smallest query sees the tile's last key)
    const bool clean = kb + KT <= Lk && (!causal || kb + KT - 1 <= P + wq0);
    if (SPEC && nx && clean) {
      s_tile(t + 1, nxt);
      finish_spec(t, cur);
    } else if (SPEC && clean && kb < wave_end) {
      finish_spec(t, cur);
    } else {
      if (nx) s_tile(t + 1, nxt);
      if (kb < wave_end) finish(t, cur);
    }
    if constexpr (DMA) {
      asm volatile("s_waitcnt vmcnt(6)" ::: "memory");  // K(t + 2), V(t + 1) landed
      barrier();
    } else {
      if (t + 2 < ntiles) store_tile(t + 2);   // its buffer (t - 1) % 3 was last read before the previous barrier
      if (t + 3 < ntiles) load_tile(t + 3);
      __syncthreads();
    }
  };
  for (int t = 0; t < ntiles; t += 2) {
    step(t, SA, SB);
    if (t + 1 < ntiles) step(t + 1, SB, SA);
  }
  if constexpr (DMA) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // trailing no-traffic pieces

  const float l_tot = sum_xhalf(l_part);
  const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
  if (qvalid) {
    bf16_t* orow = o + (size_t)(s0 + qi) * ldo + h * D;
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int d = db * 32 + 8 * g + 4 * hi;
        *(u32x2_t*)(orow + d) = u32x2_t{pack_bf2(oacc[db][4 * g] * inv, oacc[db][4 * g + 1] * inv),
                                        pack_bf2(oacc[db][4 * g + 2] * inv, oacc[db][4 * g + 3] * inv)};
      }
  }
}

// ------------------------------------------------------------------------------------------
// Decode attention: q [B, ldq] (head h at h*D), caches [slots, Hkv, max_seq, D],
// lens[b] = tokens in cache for b (current token included), slot[b] = cache slot of b.
// Partials: po [B, H, nsplit, D] fp32 (unnormalised, relative to pm), pm/pl [B, H, nsplit].
//
// Memory-bound streaming design: for a fixed (slot, kv head) the keys of a 64-key tile are one
// contiguous [64 x D] bf16 block, so each wave loads it as a flat byte array with fully coalesced
// 16-B-per-lane loads (1 KiB per wave-instruction) — chunk c = 64*i + lane holds key c / (D/8),
// dims 8*(c % (D/8)) .. +7. Partial dot products are reduced per key with lane shuffles when a key's
// chunks sit in one wave-instruction (D = 64, 128) or through a small per-wave LDS buffer (D = 96).
// The P*V accumulation uses the same flat chunks: lane's dim-slot for chunk i is static given
// i mod NSET, so accumulators stay in registers. Each of the 4 waves streams its own tiles with its
// own online softmax (no block barriers in the loop); the waves are merged once at the end.
// Split-KV epilogue shared by the decode kernels. A split's merged (over its 4 waves) result for
// query head h: unnormalised O row `o`, running max M (log2 domain), sum ls. With one split the
// normalised bf16 output is written directly; otherwise the fp32 partial, and the LAST split of
// (b, kv head) to finish (atomic ticket in cnt[b * Hkv + hk], reset by that split so the counters
// are zero again for the next launch / graph replay) merges all splits of its G heads — the
// separate combine launch (~5 us per layer, most of a batch-1 decode attention) is gone.
// Keys per split of a row. The grid's split count is fixed at capture (sized for the cache
// capacity, max_len), but a row holds L <= max_len keys: balanced splits (the default) spread the
// row's L keys over ALL its splits (64-key multiples) instead of filling the first ceil(L / chunk)
// and leaving the rest idle — at batch 1 and 2.9k of 4k keys, 256 working workgroups instead of 192.
__device__ __forceinline__ int dec_chunk(int L, int nsplit, int chunk_arg) {
  const int c = ((L + nsplit - 1) / nsplit + 63) & ~63;
  return c < chunk_arg ? c : chunk_arg;
}

__device__ __forceinline__ void dec_store(float o, float M, float ls, int b, int h, int d, int H, int nsplit,
                                          int split, int D, float* po, float* pm, float* pl, bf16_t* out,
                                          int ldo, int act) {
  if (act == 1) {
    out[(size_t)b * ldo + h * D + d] = f2bf(ls > 0.f ? o / ls : 0.f);
    return;
  }
  const size_t pidx = ((size_t)b * H + h) * nsplit + split;
  po[pidx * D + d] = o;
  if (d == 0) { pm[pidx] = M; pl[pidx] = ls; }
}

// XC (same-XCD exchange): every split of (b, kv head) ran on ONE XCD (the launch's workgroup ->
// XCD round-robin, see decode_attn_kernel), so partials and tickets live in ordinary (cached)
// memory: the stores reach that XCD's L2, the ticket is an L2 atomic and the merging split reads
// the partials from L2 (agent-scope loads: past its L1) — L2 round trips instead of uncached ones.
template <int D, int G, bool XC = false>
__device__ __forceinline__ void dec_finish(const float* po, const float* pm, const float* pl, int H, int Hkv,
                                           int nsplit, int b, int hk, int* cnt, bf16_t* out, int ldo, int* s_last,
                                           int act) {
  if (act == 1 || cnt == nullptr) return;  // no counters: the host launches decode_combine_kernel
  const int tid = threadIdx.x;
  // Partials and tickets live in UNCACHED memory (da_malloc_uncached: MTYPE UC, L2 bypassed, L1 not), so
  // device-wide visibility needs only this workgroup's stores to have completed — no
  // __threadfence(), whose L2 write-back + invalidate of the whole cache costs more than the
  // combine launch it replaces (measured: 24.6 -> 48.4 us at batch 1).
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (tid == 0) {
    int* c = &cnt[b * Hkv + hk];
    const int old = XC ? __hip_atomic_fetch_add(c, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : atomicAdd(c, 1);
    *s_last = old == act - 1;
    if (*s_last) {
      if constexpr (XC) __hip_atomic_store(c, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      else *c = 0;
    }
  }
  __syncthreads();
  if (!*s_last) return;
  // Past this CU's L1 (agent scope), for uncached memory too: the maxima and sums of some 10 (row, head) pairs share a line, and a
  // workgroup that merged one of them here earlier in this launch has left that line, with the others' from before, in L1.
  auto ld = [](const float* p) -> float { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); };
  // One online pass over the splits, 8 splits' (m, l, o) loads issued per step: the partials sit in
  // uncached memory (~1-2 us per round trip), so a max pass + a sum pass that each walk the splits
  // one dependent load at a time cost ~2 x nsplit round trips — most of a batch-1 decode attention.
  for (int i = tid; i < G * D; i += blockDim.x) {
    const int g = i / D, d = i % D, h = hk * G + g;
    const size_t base = ((size_t)b * H + h) * nsplit;
    float M = -INFINITY, lsum = 0.f, acc = 0.f;
    for (int s0 = 0; s0 < act; s0 += 8) {
      float ms[8], ls[8], os[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int s = min(s0 + j, act - 1);
        ms[j] = ld(pm + base + s);
        ls[j] = ld(pl + base + s);
        os[j] = ld(po + (base + s) * D + d);
      }
      float mx = M;
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (s0 + j < act) mx = fmaxf(mx, ms[j]);
      const float mu = (mx == -INFINITY) ? 0.f : mx;
      const float r = (M == -INFINITY) ? 0.f : exp2f(M - mu);
      lsum *= r;
      acc *= r;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        if (s0 + j >= act) continue;
        const float f = exp2f(ms[j] - mu);
        lsum += ls[j] * f;
        acc += os[j] * f;
      }
      M = mx;
    }
    out[(size_t)b * ldo + h * D + d] = f2bf(lsum > 0.f ? acc / lsum : 0.f);
  }
}

// Fused RoPE + KV-cache write for the decode step (cs != null; MHA kernel): q is the raw qkv row
// ([q heads | k heads | v heads], row stride ldq). The kernel rotates q on its way into LDS, and
// the split holding the new token (key L-1, rope position pos[b] == L-1) takes that key's rotated
// k and v straight from the qkv row — as one extra online-softmax term, never read back from the
// cache — and writes them into the cache slot for later steps. Replaces the per-layer
// rope_cache launch of the decode step (bit-identical: the same bf16 roundings).
struct DecRope {
  bf16_t* kc;           // cache bases (writable) for the new token's k / v
  bf16_t* vc;
  const float* cs;      // [max_pos][D/2][2] (cos, sin)
  const int* pos;       // [B]
};

template <int D, int G, int VAR>
__global__ void __launch_bounds__(256)
decode_attn_kernel(const bf16_t* __restrict__ q, int ldq, const bf16_t* __restrict__ kc,
                   const bf16_t* __restrict__ vc, const int* __restrict__ lens, const int* __restrict__ slot,
                   const int* __restrict__ pre,
                   int H, int Hkv, int max_seq, int chunk_max, int nsplit, float scale_log2e,
                   float* __restrict__ po, float* __restrict__ pm, float* __restrict__ pl,
                   bf16_t* __restrict__ out, int ldo, int* __restrict__ cnt, DecRope rope) {
  constexpr int KT = 64;
  constexpr int CPR = D / 8;                       // 16-B chunks per key row
  constexpr int GCD = (CPR % 16 == 0) ? 16 : ((CPR % 8 == 0) ? 8 : ((CPR % 4 == 0) ? 4 : 2));
  constexpr int NSET = CPR / GCD;                  // distinct dim-slots per lane
  constexpr bool SHFL = (64 % CPR) == 0;           // a key's chunks live in one wave-instruction
  // 4 waves per workgroup (8, a split's tiles all in flight at once at batch 1, measured 2x slower:
  // profiles/r4/rejected_r4.txt)
  constexpr int NWV = 4, NTH = 64 * NWV;
  __shared__ float sq[G][D];
  __shared__ float sp[NWV][G][KT];
  __shared__ float spart[SHFL ? 1 : NWV][SHFL ? 1 : G * KT * CPR];
  __shared__ float so[G == 1 ? 1 : NWV][G][D];
  __shared__ float sacc[G == 1 ? NWV * NSET * 64 * 8 : 1];
  __shared__ float swm[NWV][G], swl[NWV][G];

  // VAR bit3 (XC): workgroup w of the launch runs on XCD w % 8 (round-robin dispatch; the host
  // enables XC only after a placement probe confirmed it), so (b, kv head) pair p takes the nsplit
  // workgroups w = 8 * (nsplit * (p / 8) + split) + p % 8: all of its splits on one XCD, their
  // partials exchanged through that XCD's L2 (dec_finish<XC>). Needs (B * Hkv) % 8 == 0.
  constexpr bool XC = (VAR & 8) != 0;
  int split = blockIdx.x, hk = blockIdx.y, b = blockIdx.z;
  if constexpr (XC) {
    const int wl = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
    const int s8 = wl >> 3, pair = (s8 / nsplit) * 8 + (wl & 7);
    split = s8 % nsplit;
    hk = pair % Hkv;
    b = pair / Hkv;
  }
  const int L = lens[b];
  DA_ASSERT(L >= 0 && L <= max_seq && slot[b] >= 0);
  const int chunk = dec_chunk(L, nsplit, chunk_max);
  const int kstart = split * chunk;
  const bool fr = rope.cs != nullptr;
  const bool own_new = fr && kstart <= L - 1 && L - 1 < kstart + chunk;  // this split holds key L-1
  const int kend = min(fr ? L - 1 : L, kstart + chunk);                  // fused: key L-1 comes from qkv
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const size_t cbase = ((size_t)slot[b] * Hkv + hk) * (size_t)max_seq * D;
  const int P = pre ? pre[2 * b] : 0;  // shared-prefix keys [0, P) live in slot pre[2b + 1]
  const size_t pbase = P ? ((size_t)pre[2 * b + 1] * Hkv + hk) * (size_t)max_seq * D : cbase;
  DA_ASSERT(P % 64 == 0 && P <= L);
  DA_ASSERT(!fr || rope.pos[b] == L - 1);
  __shared__ float skn[D], svn[D], ssn[G];

  // VAR bit0: non-temporal loads (the KV stream is read once per step); bit1: V issued together
  // with K (else after the scores: ~100 VGPRs live instead of ~200, so 4-5 waves per SIMD hide the
  // HBM latency instead of 2); bit2 (small batches, implies bit1): the wave's NEXT tile is loaded
  // before the current one is computed — at batch 1 a workgroup's few tiles are latency-bound, one
  // HBM round trip each, and occupancy buys nothing. Loads are branch-free (chunk index clamped
  // into the tile; keys >= nk get p = 0) so the compiler's vmcnt waits stay counted.
  constexpr bool NT = VAR & 1, PFT = (VAR & 4) != 0, VEARLY = PFT || (VAR & 2) != 0;
  auto ld16 = [&](const bf16_t* p) -> u32x4_t {
    if constexpr (NT) return __builtin_nontemporal_load((const u32x4_t*)p);
    else return *(const u32x4_t*)p;
  };
  auto tile_base = [&](const bf16_t* c, int t0) {
    return c + (t0 < P ? pbase : cbase) + (size_t)t0 * D;
  };
  // PFT loads are branch-free: a tile past kend reads key 0 of the row's own slot (one line, valid
  // memory, never used) so the prefetches can be issued unconditionally
  auto load_k = [&](u32x4_t (&kv)[CPR], int t0) {
    const int nk = kend - t0;
    const int last = min(KT, nk) * CPR - 1;
    const bf16_t* kb = tile_base(kc, t0);
#pragma unroll
    for (int i = 0; i < CPR; ++i) {
      const int c = i * 64 + lane;
      if constexpr (PFT) kv[i] = ld16(nk > 0 ? kb + min(c, last) * 8 : kc + cbase);
      else kv[i] = (c <= last) ? ld16(kb + c * 8) : u32x4_t{0, 0, 0, 0};
    }
  };
  auto load_v = [&](u32x4_t (&vv)[CPR], int t0) {
    const int nk = kend - t0;
    const int last = min(KT, nk) * CPR - 1;
    const bf16_t* vb = tile_base(vc, t0);
#pragma unroll
    for (int i = 0; i < CPR; ++i) {
      const int c = i * 64 + lane;
      if constexpr (PFT) vv[i] = ld16(nk > 0 ? vb + min(c, last) * 8 : vc + cbase);
      else vv[i] = (c <= last) ? ld16(vb + c * 8) : u32x4_t{0, 0, 0, 0};
    }
  };
  // RoPE (interleaved pairs (2i, 2i+1)) of one element of a head row, rounded to bf16 like the
  // rope_cache kernel / the QKV GEMM epilogue that this path replaces
  constexpr int HALF = D / 2;
  auto rot2 = [&](float x1, float x2, float c, float sn, int d) -> float {
    return bf2f(f2bf((d & 1) ? x2 * c + x1 * sn : x1 * c - x2 * sn));
  };
  auto rot = [&](const bf16_t* hp, int d, int p) -> float {
    const int i = d >> 1;
    return rot2(bf2f(hp[d & ~1]), bf2f(hp[d | 1]), rope.cs[((size_t)p * HALF + i) * 2],
                rope.cs[((size_t)p * HALF + i) * 2 + 1], d);
  };
  // PFT (small batches): the prologue's operands (this thread's q element, its RoPE partner and
  // cos / sin, the new token's k / v element) are loaded FIRST, then the first two K/V tiles of the
  // wave are requested, unconditionally (an empty tile reads one line), so the compiler's counted
  // wait for the prologue leaves the K/V stream in flight: its first HBM round trip overlaps the
  // prologue instead of following it (vmcnt retires loads in order).
  constexpr bool PRE = PFT && G * D <= 256;
  u32x4_t ka[PFT ? CPR : 1], va[PFT ? CPR : 1], kb2[PFT ? CPR : 1], vb2[PFT ? CPR : 1];
  if constexpr (PRE) {
    // straight-line, clamped loads of raw bits: no branch and no use before the K/V loads below, so
    // the wait for them is a counted vmcnt(48), not vmcnt(0) (a use inside a branch forces the latter)
    const int qi = min(tid, G * D - 1), d = qi % D;
    const bf16_t* hp = q + (size_t)b * ldq + (hk * G + qi / D) * D;
    const bf16_t rq1 = hp[d & ~1], rq2 = hp[d | 1];
    const float* csp = fr ? rope.cs + ((size_t)(L - 1) * HALF + (d >> 1)) * 2 : (const float*)hp;
    const f32x2_t rcs = *(const f32x2_t*)csp;
    const bf16_t* kr = fr ? q + (size_t)b * ldq + (size_t)(H + hk) * D : hp;
    const bf16_t* vr = fr ? q + (size_t)b * ldq + (size_t)(H + Hkv + hk) * D : hp;
    const bf16_t rk1 = kr[d & ~1], rk2 = kr[d | 1], nv = vr[d];
    const int t0 = kstart + w * KT, t1 = t0 + NWV * KT;
    load_k(ka, t0); load_v(va, t0);
    load_k(kb2, t1); load_v(vb2, t1);
    const float pc = fr ? rcs[0] : 1.f, ps = fr ? rcs[1] : 0.f;
    if (tid < G * D) {
      const float px1 = bf2f(rq1), px2 = bf2f(rq2);
      const float x = fr ? rot2(px1, px2, pc, ps, d) : ((d & 1) ? px2 : px1);
      sq[tid / D][d] = x * scale_log2e;
    }
    if (own_new && tid < D) {
      const size_t crow = cbase + (size_t)(L - 1) * D;
      const float kv = rot2(bf2f(rk1), bf2f(rk2), pc, ps, d);  // same position L - 1 -> same cos / sin
      skn[d] = kv;
      svn[d] = bf2f(nv);
      rope.kc[crow + d] = f2bf(kv);  // for later steps (read back only after this launch)
      rope.vc[crow + d] = nv;
    }
  } else {
    if constexpr (PFT) {
      const int t0 = kstart + w * KT, t1 = t0 + NWV * KT;
      load_k(ka, t0); load_v(va, t0);
      load_k(kb2, t1); load_v(vb2, t1);
    }
    for (int i = tid; i < G * D; i += NTH) {
      const int g = i / D, d = i % D;
      const bf16_t* hp = q + (size_t)b * ldq + (hk * G + g) * D;
      sq[g][d] = (fr ? rot(hp, d, L - 1) : bf2f(hp[d])) * scale_log2e;
    }
  }
  if (own_new && !PRE) {
    const size_t crow = cbase + (size_t)(L - 1) * D;
    const bf16_t* kr = q + (size_t)b * ldq + (size_t)(H + hk) * D;
    const bf16_t* vr = q + (size_t)b * ldq + (size_t)(H + Hkv + hk) * D;
    for (int d = tid; d < D; d += NTH) {
      const float kv = rot(kr, d, L - 1);
      skn[d] = kv;
      svn[d] = bf2f(vr[d]);
      rope.kc[crow + d] = f2bf(kv);  // for later steps (read back only after this launch)
      rope.vc[crow + d] = vr[d];
    }
  }
  if constexpr (G > 1) {
    for (int i = tid; i < NWV * G * D; i += NTH) (&so[0][0][0])[i] = 0.f;
  }
  __syncthreads();
  if (own_new && w == 0) {  // score of the new key for each query head of this kv head
#pragma unroll
    for (int g = 0; g < G; ++g) {
      float part = 0.f;
      for (int d = lane; d < D; d += 64) part += sq[g][d] * skn[d];
      part = wave_sum(part);
      if (lane == 0) ssn[g] = part;
    }
  }

  float m[G], l[G], acc[G][NSET][8];
#pragma unroll
  for (int g = 0; g < G; ++g) {
    m[g] = -INFINITY; l[g] = 0.f;
#pragma unroll
    for (int s = 0; s < NSET; ++s)
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[g][s][e] = 0.f;
  }

  auto process = [&](const u32x4_t (&kv)[CPR], u32x4_t (&vv)[CPR], int t0) {
    const int nk = min(KT, kend - t0);
    // ---- scores ----
#pragma unroll
    for (int i = 0; i < CPR; ++i) {
      const int c = i * 64 + lane;
      const int dp = c % CPR;
      float kf[8];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        kf[2 * e] = bf2f((bf16_t)(kv[i][e] & 0xffff));
        kf[2 * e + 1] = bf2f((bf16_t)(kv[i][e] >> 16));
      }
#pragma unroll
      for (int g = 0; g < G; ++g) {
        const f32x4_t q0 = *(const f32x4_t*)&sq[g][dp * 8];
        const f32x4_t q1 = *(const f32x4_t*)&sq[g][dp * 8 + 4];
        float part = kf[0] * q0[0] + kf[1] * q0[1] + kf[2] * q0[2] + kf[3] * q0[3] +
                     kf[4] * q1[0] + kf[5] * q1[1] + kf[6] * q1[2] + kf[7] * q1[3];
        if constexpr (SHFL) {
#pragma unroll
          for (int o = 1; o < CPR; o <<= 1) part += __shfl_xor(part, o, 64);
          if (dp == 0) sp[w][g][c / CPR] = part;
        } else {
          spart[w][g * KT * CPR + c] = part;
        }
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    // ---- online softmax; lane = key ----
#pragma unroll
    for (int g = 0; g < G; ++g) {
      float sc;
      if constexpr (SHFL) {
        sc = sp[w][g][lane];
      } else {
        sc = 0.f;
#pragma unroll
        for (int j = 0; j < CPR; ++j) sc += spart[w][g * KT * CPR + lane * CPR + j];
      }
      if (lane >= nk) sc = -INFINITY;
      const float tmax = wave_max(sc);
      const float m_new = fmaxf(m[g], tmax);
      const float m_use = (m_new == -INFINITY) ? 0.f : m_new;
      const float alpha = exp2f(m[g] - m_use);
      const float p = exp2f(sc - m_use);
      l[g] = l[g] * alpha + wave_sum(p);
      m[g] = m_new;
      sp[w][g][lane] = p;
#pragma unroll
      for (int st = 0; st < NSET; ++st)
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[g][st][e] *= alpha;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    // ---- P * V ----
    asm volatile("" ::: "memory");
    if constexpr (!VEARLY) load_v(vv, t0);
#pragma unroll
    for (int i = 0; i < CPR; ++i) {
      const int c = i * 64 + lane;
      const int key = c / CPR;
      float vf[8];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        vf[2 * e] = bf2f((bf16_t)(vv[i][e] & 0xffff));
        vf[2 * e + 1] = bf2f((bf16_t)(vv[i][e] >> 16));
      }
#pragma unroll
      for (int g = 0; g < G; ++g) {
        const float pk = sp[w][g][key];
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[g][i % NSET][e] += pk * vf[e];
      }
    }
    __builtin_amdgcn_wave_barrier();
  };

  if constexpr (PFT) {  // two tiles in flight per wave: ka/va and kb2/vb2 alternate
    int t0 = kstart + w * KT;
    while (t0 < kend) {
      const int t1 = t0 + NWV * KT;
      process(ka, va, t0);
      if (t1 >= kend) break;
      const int t2 = t1 + NWV * KT;
      if (t2 < kend) { load_k(ka, t2); load_v(va, t2); }
      process(kb2, vb2, t1);
      if (t2 >= kend) break;
      const int t3 = t2 + NWV * KT;
      if (t3 < kend) { load_k(kb2, t3); load_v(vb2, t3); }
      t0 = t2;
    }
  } else {
    for (int t0 = kstart + w * KT; t0 < kend; t0 += NWV * KT) {
      u32x4_t kv[CPR], vv[CPR];
      load_k(kv, t0);
      if constexpr (VEARLY) load_v(vv, t0);
      process(kv, vv, t0);
    }
  }
  // ---- merge lanes -> per-wave O, then waves -> block partial ----
  // MHA (G = 1): every lane parks its accumulators in LDS with plain 16-B stores and the output
  // threads sum the (dim-slot, lane) entries that hold their dim. LDS float atomics — 5-6 lanes per
  // address — took 7.5 us of a 20 us batch-1 launch (bench/decode_trace.py), more than the K/V stream.
  if constexpr (G == 1) {
#pragma unroll
    for (int st = 0; st < NSET; ++st) {
      float* dst = &sacc[((w * NSET + st) * 64 + lane) * 8];
      *(f32x4_t*)dst = f32x4_t{acc[0][st][0], acc[0][st][1], acc[0][st][2], acc[0][st][3]};
      *(f32x4_t*)(dst + 4) = f32x4_t{acc[0][st][4], acc[0][st][5], acc[0][st][6], acc[0][st][7]};
    }
  } else {
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
      for (int st = 0; st < NSET; ++st) {
        const int dp = (lane + 64 * st) % CPR;
#pragma unroll
        for (int e = 0; e < 8; ++e) atomicAdd(&so[w][g][dp * 8 + e], acc[g][st][e]);
      }
  }
  if (lane == 0) {
#pragma unroll
    for (int g = 0; g < G; ++g) { swm[w][g] = m[g]; swl[w][g] = l[g]; }
  }
  __syncthreads();
  for (int i = tid; i < G * D; i += NTH) {
    const int g = i / D, d = i % D;
    float M = fmaxf(fmaxf(swm[0][g], swm[1][g]), fmaxf(swm[2][g], swm[3][g]));
#pragma unroll
    for (int ww = 4; ww < NWV; ++ww) M = fmaxf(M, swm[ww][g]);
    if (own_new) M = fmaxf(M, ssn[g]);
    const float Mu = (M == -INFINITY) ? 0.f : M;
    float o = 0.f, ls = 0.f;
#pragma unroll
    for (int ww = 0; ww < NWV; ++ww) {
      const float f = exp2f(swm[ww][g] - Mu);
      float ow;
      if constexpr (G == 1) {
        // lane l's slot st holds dims 8 * ((64 st + l) % CPR) .. +7
        // fixed trip counts: all of a wave's reads are independent and issued back to back
        ow = 0.f;
        const int dp = d >> 3, e = d & 7;
#pragma unroll
        for (int st = 0; st < NSET; ++st) {
          const int l0 = ((dp - 64 * st) % CPR + CPR) % CPR;
#pragma unroll
          for (int j = 0; j < (64 + CPR - 1) / CPR; ++j) {
            const int l = l0 + j * CPR;
            if (l < 64) ow += sacc[((ww * NSET + st) * 64 + l) * 8 + e];
          }
        }
      } else {
        ow = so[ww][g][d];
      }
      o += ow * f;
      ls += swl[ww][g] * f;
    }
    if (own_new) {  // the new token's key: weight exp2(s - M), value straight from the qkv row
      const float f = exp2f(ssn[g] - Mu);
      o += svn[d] * f;
      ls += f;
    }
    dec_store(o, M, ls, b, hk * G + g, d, H, nsplit, split, D, po, pm, pl, out, ldo, nsplit);
  }
  __shared__ int s_last;
  dec_finish<D, G, XC>(po, pm, pl, H, Hkv, nsplit, b, hk, cnt, out, ldo, &s_last, nsplit);
}

// ------------------------------------------------------------------------------------------
// GQA decode attention on MFMA (G = H/Hkv query heads share one KV head: Llama-3-8B G=4,
// Llama-3-70B at TP=8 G=8). The G queries of a KV head form the N=16 side of
// v_mfma_f32_16x16x32_bf16 (zero-padded), so K and V are read once per KV head instead of being
// multiplied against each query on the VALU (the G >= 2 path of decode_attn_kernel is VALU-bound).
// Per wave and 32-key tile:
//   S^T[key][g] = K·Q^T : A = K rows from the wave's private LDS ring, B = Q^T (registers, loaded once);
//   softmax over the 32 keys of each query column: 8 values per lane + two cross-lane steps;
//   O^T[d][g] += V^T·P^T : B = P^T from the S^T registers (k index permuted), A = V^T read with ds_read_b64_tr_b16.
// K and V tiles are contiguous [32 x D] blocks of the cache, copied by LDS-DMA (1 KiB per wave instruction) with an XOR
// chunk swizzle on the source address that makes both reads conflict-free. A tile's place is filled again as soon as its
// fragments are in registers, so a wave's next K tile is on its way beside the softmax and V's beside the next scores (D = 64:
// another tile more): counted waits, no barrier; rows past the end are out of the resource's range (zeros, no traffic).
// Bound by HBM and by what a CU can have on its way (some 256 requests, whatever is asked for): K rows loaded straight into A
// registers were requests of 64 B (four lanes a row), and a workgroup got 31 GB/s of the 57 that whole rows give it. 64 rows of
// 900 - 3100 keys, 8 heads x 128: 112 -> 87 us (6.0 TB/s), all of 2000 89 -> 83, 33 rows 66 -> 52, 8 of 4000 among 56 of 300
// 70 -> 55. Two stages for D = 128 leave one workgroup per CU, whose start and end nothing covers: 89, 90, 54, 55.
// by_len: a row takes at most as many splits as hold chunk_max keys each (256: a split's merge costs what reading 100 - 200
// keys does), and splits are the slowest grid dimension: as the fastest one, the workgroups of a launch with two splits
// whose rows need one only were all on the even XCDs (64 rows of 2048 keys: 147 us against 86). A workgroup of a split
// past the row's keys ends at once.
// pair_rows: whole rows, up to 64 of them, two workgroups per CU: paired_row (91 -> 87 us in the first case above).
template <int D>
__device__ __forceinline__ int vswz(int r) {
  return D == 128 ? ((r & 7) << 1) : D == 96 ? ((r >> 2) & 1) << 1 : (((r >> 1) & 3) << 1);
}
template <int D>
__device__ __forceinline__ int kswz(int r) {
  return D == 128 ? r & 15 : D == 96 ? (r >> 2) & 3 : (r >> 1) & 7;
}

// The row that workgroup row z of B <= 64 takes, and its keys: the `round` longest first (a workgroup per CU), then from the
// shortest on, so that the second workgroup of a CU with a long row has a short one; as they come where none is 512 keys off
// the first (the ranks take 1 us).
__device__ __forceinline__ int paired_row(const int* __restrict__ lens, int B, int z, int round, int& L) {
  const int lane = threadIdx.x & 63;
  const int len = lane < B ? lens[lane] : -1;
  int row = z;
  if (__ballot(lane < B && abs(len - __builtin_amdgcn_readfirstlane(len)) > 512)) {
    int rank = 0;
    for (int j = 0; j < B; ++j) {
      const int o = __builtin_amdgcn_readlane(len, j);
      rank += o > len || (o == len && j < lane);
    }
    row = __builtin_ctzll(__ballot(lane < B && rank == (z < round ? z : B - 1 - (z - round))));
  }
  L = __builtin_amdgcn_readlane(len, row);
  return row;
}

template <int D, int G>
__global__ void __launch_bounds__(256, 2)
decode_attn_gqa_kernel(const bf16_t* __restrict__ q, int ldq, const bf16_t* __restrict__ kc,
                       const bf16_t* __restrict__ vc, const int* __restrict__ lens, const int* __restrict__ slot,
                   const int* __restrict__ pre,
                       int H, int Hkv, int max_seq, int chunk_max, int nsplit, float scale_log2e,
                       float* __restrict__ po, float* __restrict__ pm, float* __restrict__ pl,
                       bf16_t* __restrict__ out, int ldo, int* __restrict__ cnt, int by_len, int pair_rows) {
  static_assert(D == 64 || D == 128, "GQA MFMA decode supports head dims 64 and 128");
  constexpr int KT = 32, NDS = D / 32, NDT = D / 16, NS = D / 8;   // d-steps (S), d-tiles (O), 16-B chunks/row
  constexpr int TB = KT * D * 2, ND = TB / 1024, ST = D == 128 ? 1 : 2;  // bytes and DMA instructions of a tile, stages
  typedef __attribute__((address_space(3))) void* lds_ptr_t;
  __shared__ __attribute__((aligned(16))) char ring[4 * ST * 2 * TB + 2 * 4 * 16 * 4 + 16];
  float (*swm)[16] = (float (*)[16])(ring + 4 * ST * 2 * TB), (*swl)[16] = swm + 4;

  const int hk = by_len ? blockIdx.x : blockIdx.y;
  const int split = by_len ? blockIdx.z : blockIdx.x;
  int b = by_len ? blockIdx.y : blockIdx.z, L;
  if (pair_rows) b = paired_row(lens, gridDim.z, b, pair_rows, L);
  else L = __builtin_amdgcn_readfirstlane(lens[b]);  // (uniform, for the DMA's resources)
  DA_ASSERT(L >= 0 && L <= max_seq && slot[b] >= 0);
  // by_len: a row's keys evenly over as many splits as hold chunk_max of them each; the others have nothing to do
  const int act = by_len && cnt ? min(nsplit, max(1, (L + chunk_max - 1) / chunk_max)) : nsplit;
  if (split >= act) return;
  const int chunk = dec_chunk(L, act, by_len ? 0x7fffffff : chunk_max);
  const int kstart = split * chunk;
  const int kend = min(L, kstart + chunk);
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int fr = lane & 15, fg = lane >> 4;
  const size_t cbase = ((size_t)__builtin_amdgcn_readfirstlane(slot[b]) * Hkv + hk) * (size_t)max_seq * D;
  const int P = pre ? __builtin_amdgcn_readfirstlane(pre[2 * b]) : 0;  // shared-prefix keys [0, P) live in slot pre[2b + 1]
  const size_t pbase = P ? ((size_t)__builtin_amdgcn_readfirstlane(pre[2 * b + 1]) * Hkv + hk) * (size_t)max_seq * D : cbase;
  DA_ASSERT(P % 64 == 0 && P <= L);
  char* mine = ring + w * (ST * 2 * TB);

  bf16x8_t qf[NDS];
#pragma unroll
  for (int ds = 0; ds < NDS; ++ds) {
    if (fr < G) qf[ds] = *(const bf16x8_t*)(q + (size_t)b * ldq + (hk * G + fr) * D + ds * 32 + fg * 8);
    else qf[ds] = bf16x8_t{0, 0, 0, 0, 0, 0, 0, 0};
  }
  // DMA sources within a tile: 1 KiB instruction i covers rows of D elements, chunk position sl holds chunk sl ^ swizzle
  unsigned ko[8], vo[8];
#pragma unroll
  for (int i = 0; i < ND; ++i) {
    const int p = i * 64 + lane, row = p / NS, sl = p % NS;
    ko[i] = (unsigned)(row * D * 2 + ((sl ^ kswz<D>(row)) << 4));
    vo[i] = (unsigned)(row * D * 2 + ((sl ^ vswz<D>(row)) << 4));
  }
  auto issue = [&](const bf16_t* cache, const unsigned (&off)[8], int t0, char* dst) __attribute__((always_inline)) {
    // the tile from key t0 on (none past kend)
    const int n = __builtin_amdgcn_readfirstlane(max(0, min(KT, kend - t0))) * D * 2;  // (uniform: no loop over resources)
    const size_t at = (t0 < P ? pbase : cbase) + (size_t)t0 * D;
    const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc((void*)(cache + at), (short)0, n, 0x00020000);
#pragma unroll
    for (int i = 0; i < ND; ++i)  // aux 2 = nt (read once per step; see decode_attn_mfma1_kernel)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_ptr_t)(dst + i * 1024), 16, off[i & 7], 0, 0, 2);
  };
  // the oldest K or V tile of the ring is in: the 2 ST - 1 issued after it may be on their way
  auto landed = [&]() __attribute__((always_inline)) {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(ND * (2 * ST - 1)) : "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  // transposed V reads: the lane's row, its half of a 16-B chunk and the odd chunk; the row's swizzle of chunk pairs
  const int vr = 4 * fg + (fr >> 2), vx = vswz<D>(vr) >> 1;
  const unsigned vrow = vr * (D * 2) + ((fr & 3) >> 1) * 16 + (fr & 1) * 8;
  f32x4_t oacc[NDT];
#pragma unroll
  for (int i = 0; i < NDT; ++i) oacc[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  float m_run = -INFINITY, l_part = 0.f;

#pragma unroll
  for (int i = 0; i < ST; ++i) {
    issue(kc, ko, kstart + (w + 4 * i) * KT, mine + i * 2 * TB);
    issue(vc, vo, kstart + (w + 4 * i) * KT, mine + i * 2 * TB + TB);
  }
#pragma unroll
  for (int ds = 0; ds < NDS; ++ds) asm volatile("" : "+v"(qf[ds]));  // (waited for here, the tiles on their way)
  int stage = 0;
  for (int t0 = kstart + w * KT; t0 < kend; t0 += 4 * KT) {
    char* kt = mine + stage * 2 * TB;
    char* vt = kt + TB;
    // ---- S^T = K Q^T; the K tile's place is free once it is in registers ----
    landed();
    bf16x8_t kf[2][NDS];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int ds = 0; ds < NDS; ++ds)
        kf[t][ds] = *(const bf16x8_t*)(kt + (16 * t + fr) * (D * 2) + (((4 * ds + fg) ^ kswz<D>(16 * t + fr)) << 4));
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    issue(kc, ko, t0 + 4 * ST * KT, kt);
    f32x4_t sacc[2] = {f32x4_t{0.f, 0.f, 0.f, 0.f}, f32x4_t{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int ds = 0; ds < NDS; ++ds)
#pragma unroll
      for (int t = 0; t < 2; ++t) sacc[t] = mfma16(kf[t][ds], qf[ds], sacc[t]);
    float mx = -INFINITY;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float sc = t0 + 16 * t + 4 * fg + i < kend ? sacc[t][i] * scale_log2e : -INFINITY;
        sacc[t][i] = sc;
        mx = fmaxf(mx, sc);
      }
    const auto rows = __builtin_amdgcn_permlane16_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
    mx = max_xhalf(fmaxf(__uint_as_float(rows[0]), __uint_as_float(rows[1])));
    if (__ballot(mx > m_run)) {  // (a new maximum is rare after the first tiles)
      const float m_new = fmaxf(m_run, mx);
      const float alpha = exp2f(m_run - (m_new == -INFINITY ? 0.f : m_new));
      m_run = m_new;
      l_part *= alpha;
#pragma unroll
      for (int i = 0; i < NDT; ++i) oacc[i] *= alpha;
    }
    const float m_use = (m_run == -INFINITY) ? 0.f : m_run;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float p = __builtin_amdgcn_exp2f(sacc[t][i] - m_use);
        sacc[t][i] = p;
        l_part += p;
      }
    // ---- O^T += V^T P^T: slot j -> key 16(j>>2) + 4fg + (j&3) ----
    const u32x4_t pw = u32x4_t{pack_bf2(sacc[0][0], sacc[0][1]), pack_bf2(sacc[0][2], sacc[0][3]),
                               pack_bf2(sacc[1][0], sacc[1][1]), pack_bf2(sacc[1][2], sacc[1][3])};
    const bf16x8_t pb = __builtin_bit_cast(bf16x8_t, pw);
    // (row 4 fg + fr / 4 and the one 16 on, whose swizzle is the same; with the builtin hipcc drains the DMA first)
    landed();
    const unsigned va0 = (unsigned)(size_t)(lds_ptr_t)vt + vrow;
    s16x4_t v[2][8];
#pragma unroll
    for (int h = 0; h < NDT / 4; ++h) {
      const int dt = 4 * h;
      asm volatile("ds_read_b64_tr_b16 %0, %8\n\tds_read_b64_tr_b16 %1, %8 offset:%12\n\t"
                   "ds_read_b64_tr_b16 %2, %9\n\tds_read_b64_tr_b16 %3, %9 offset:%12\n\t"
                   "ds_read_b64_tr_b16 %4, %10\n\tds_read_b64_tr_b16 %5, %10 offset:%12\n\t"
                   "ds_read_b64_tr_b16 %6, %11\n\tds_read_b64_tr_b16 %7, %11 offset:%12\n\ts_waitcnt lgkmcnt(0)"
                   : "=&v"(v[h][0]), "=&v"(v[h][1]), "=&v"(v[h][2]), "=&v"(v[h][3]), "=&v"(v[h][4]), "=&v"(v[h][5]),
                     "=&v"(v[h][6]), "=&v"(v[h][7])
                   : "v"(va0 + ((dt ^ vx) << 5)), "v"(va0 + (((dt + 1) ^ vx) << 5)), "v"(va0 + (((dt + 2) ^ vx) << 5)),
                     "v"(va0 + (((dt + 3) ^ vx) << 5)), "n"(16 * D * 2)
                   : "memory");
      if (h == NDT / 4 - 1) issue(vc, vo, t0 + 4 * ST * KT, vt);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const s16x4_t lo = v[h][2 * j], hi = v[h][2 * j + 1];
        oacc[dt + j] = mfma16(bf16x8_t{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]}, pb, oacc[dt + j]);
      }
    }
    stage = stage + 1 == ST ? 0 : stage + 1;
  }
  // ---- merge the 4 waves: per-query (m, l) and O^T partials through LDS ----
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (pieces past the end write zeros)
  float l_tot = l_part + __shfl_xor(l_part, 16, 64);
  l_tot = sum_xhalf(l_tot);
  if (fg == 0) { swm[w][fr] = m_run; swl[w][fr] = l_tot; }
  __syncthreads();  // every wave is done with its ring
  float* so = (float*)ring;  // [4][16][D]
#pragma unroll
  for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
    for (int i = 0; i < 4; ++i) so[(w * 16 + fr) * D + dt * 16 + 4 * fg + i] = oacc[dt][i];
  __syncthreads();
  for (int i = tid; i < G * D; i += 256) {
    const int g = i / D, d = i % D;
    const float M = fmaxf(fmaxf(swm[0][g], swm[1][g]), fmaxf(swm[2][g], swm[3][g]));
    const float Mu = (M == -INFINITY) ? 0.f : M;
    float o = 0.f, ls = 0.f;
#pragma unroll
    for (int ww = 0; ww < 4; ++ww) {
      const float f = exp2f(swm[ww][g] - Mu);
      o += so[(ww * 16 + g) * D + d] * f;
      ls += swl[ww][g] * f;
    }
    dec_store(o, M, ls, b, hk * G + g, d, H, nsplit, split, D, po, pm, pl, out, ldo, act);
  }
  dec_finish<D, G>(po, pm, pl, H, Hkv, nsplit, b, hk, cnt, out, ldo, (int*)(swl + 4), act);
}

// MHA decode attention (G = 1) on MFMA: the GQA kernel's data path, with the one query in all 16 columns, so that every lane has
// the weights of its 8 keys. They stay fp32: column 0 of P^T holds their upper 8 bits (as bf16), column 1 the next 8, column 2
// the last, and the three columns of O^T are added at the end. (Dot products and weighted sums on the VALU, decode_attn_kernel,
// take it 2000 cycles per 64 keys: this kernel had only launches of up to 32 pairs, K rows by 64-B requests and weights of 16
// bits, the others the VALU.) us before / after, 32 heads x 96: one row of 60 / 300 / 2935 / 4000 keys 7.6 / 8.5 / 13.2 / 15.0 ->
// 5.5 / 7.3 / 11.6 / 13.5; rows of 64 - 146 keys, 4 / 12 / 30 / 40 of them, 10.6 / 18.1 / 17.9 / 23.2 -> 6.5 / 7.9 / 14.1 /
// 16.3; of 500 - 2000 19.0 / 50.8 / 86.7 / 89.1 -> 16.6 / 41.6 / 79.4 / 88.5 (5.9 TB/s). Few keys: bound by the launch, the
// chain length -> addresses -> keys and the merge, about 5 us.
// One stage of tiles: with two for D = 64 a CU has two workgroups, which short rows wait for, us two / one (the VALU before): 12
// heads, 64 rows of 40 - 146 keys 10.8 / 8.1 (8.5), 32 of 200 - 500 15.0 / 12.3 (13.1), 16 of 500 - 2000 19.5 / 16.2 (18.9); long rows
// lose some of it, 48 of 900 - 3100 51.6 / 55.8 (59.8), one of 4000 among 31 of 200 17.6 / 19.4 (31.7).
// by_len (as in the GQA kernel): even splits of 12 rows of 64 - 146 keys in a cache of 4096 take 10.9 us, of 200 - 500 15.8 (16.5
// by length).
// XC: same-XCD split exchange (see dec_finish).
// RP: fused RoPE + new-token KV write (DecRope, as decode_attn_kernel): q is the raw qkv row; q is
// rotated into LDS while the tiles fly, key L - 1 enters as one extra online-softmax term of the
// split that holds it (taken from the qkv row, written into the cache for later steps).
template <int D, bool XC, bool RP>
__global__ void __launch_bounds__(256, 2)
decode_attn_mfma1_kernel(const bf16_t* __restrict__ q, int ldq, const bf16_t* __restrict__ kc,
                         const bf16_t* __restrict__ vc, const int* __restrict__ lens, const int* __restrict__ slot,
                         const int* __restrict__ pre, int H, int Hkv, int max_seq, int chunk_max, int nsplit,
                         float scale_log2e, float* __restrict__ po, float* __restrict__ pm, float* __restrict__ pl,
                         bf16_t* __restrict__ out, int ldo, int* __restrict__ cnt, DecRope rope, int by_len) {
  static_assert(D == 64 || D == 96 || D == 128, "head dim");
  constexpr int KT = 32, NDS = D / 32, NDT = D / 16, NS = D / 8;
  constexpr int TB = KT * D * 2, ND = TB / 1024, ST = 1;
  typedef __attribute__((address_space(3))) void* lds_ptr_t;
  // (one array: with several, hipcc has every LDS read wait for the DMA)
  __shared__ __attribute__((aligned(16))) char ring[4 * ST * 2 * TB + 64 + D * 10];
  float* swm = (float*)(ring + 4 * ST * 2 * TB);
  float *swl = swm + 4, *ssn = swm + 8, *skn = swm + 16, *svn = skn + D;
  bf16_t* sqb = (bf16_t*)(svn + D);

  int split = by_len ? blockIdx.z : blockIdx.x, hk = by_len ? blockIdx.x : blockIdx.y, b = by_len ? blockIdx.y : blockIdx.z;
  if constexpr (XC) {  // the same-XCD mapping of decode_attn_kernel
    const int wl = blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z);
    const int s8 = wl >> 3, pair = (s8 / nsplit) * 8 + (wl & 7);
    split = s8 % nsplit;
    hk = pair % Hkv;
    b = pair / Hkv;
  }
  const int L = __builtin_amdgcn_readfirstlane(lens[b]);  // (uniform, for the DMA's resources)
  DA_ASSERT(L >= 0 && L <= max_seq && slot[b] >= 0);
  const int act = by_len && cnt ? min(nsplit, max(1, (L + chunk_max - 1) / chunk_max)) : nsplit;  // (see the GQA kernel)
  if (split >= act) return;
  const int chunk = dec_chunk(L, act, by_len ? 0x7fffffff : chunk_max);
  const int kstart = split * chunk;
  const bool own_new = RP && kstart <= L - 1 && L - 1 < kstart + chunk;  // this split holds key L - 1
  const int kend = min(RP ? L - 1 : L, kstart + chunk);                  // RP: key L - 1 from the qkv row
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int fr = lane & 15, fg = lane >> 4;
  const size_t cbase = ((size_t)__builtin_amdgcn_readfirstlane(slot[b]) * Hkv + hk) * (size_t)max_seq * D;
  const int P = pre ? __builtin_amdgcn_readfirstlane(pre[2 * b]) : 0;  // shared-prefix keys [0, P) live in slot pre[2b + 1]
  const size_t pbase = P ? ((size_t)__builtin_amdgcn_readfirstlane(pre[2 * b + 1]) * Hkv + hk) * (size_t)max_seq * D : cbase;
  DA_ASSERT(P % 64 == 0 && P <= L);
  DA_ASSERT(!RP || rope.pos[b] == L - 1);
  char* mine = ring + w * (ST * 2 * TB);

  // this thread's element d of the query and (RP) of the new key and value, with its partner in the pair and its angle
  const bf16_t* qrow = q + (size_t)b * ldq;
  bf16x8_t qf[NDS];
  [[maybe_unused]] unsigned rq = 0, rk = 0, rv = 0;
  [[maybe_unused]] f32x2_t rcs = f32x2_t{1.f, 0.f};
  const int d = min(tid, D - 1);
  if constexpr (RP) {
    rq = *(const unsigned*)(qrow + hk * D + (d & ~1));
    rk = *(const unsigned*)(qrow + (size_t)(H + hk) * D + (d & ~1));
    rv = *(const unsigned*)(qrow + (size_t)(H + Hkv + hk) * D + (d & ~1));
    rcs = *(const f32x2_t*)(rope.cs + ((size_t)max(L - 1, 0) * (D / 2) + (d >> 1)) * 2);
  } else {
#pragma unroll
    for (int ds = 0; ds < NDS; ++ds) qf[ds] = *(const bf16x8_t*)(qrow + hk * D + ds * 32 + fg * 8);
  }
  unsigned ko[8], vo[8];  // DMA sources within a tile
#pragma unroll
  for (int i = 0; i < ND; ++i) {
    const int p = i * 64 + lane, row = p / NS, sl = p % NS;
    ko[i] = (unsigned)(row * D * 2 + ((sl ^ kswz<D>(row)) << 4));
    vo[i] = (unsigned)(row * D * 2 + ((sl ^ vswz<D>(row)) << 4));
  }
  __builtin_amdgcn_sched_barrier(0);  // (the loads above are the oldest)
  auto issue = [&](const bf16_t* cache, const unsigned (&off)[8], int t0, char* dst) __attribute__((always_inline)) {
    // the tile from key t0 on (none past kend)
    const int n = __builtin_amdgcn_readfirstlane(max(0, min(KT, kend - t0))) * D * 2;
    const size_t at = (t0 < P ? pbase : cbase) + (size_t)t0 * D;
    const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc((void*)(cache + at), (short)0, n, 0x00020000);
#pragma unroll
    for (int i = 0; i < ND; ++i)
      // aux 2 = nt: the KV stream is read once per step; allocating it in L2 / MALL cost the GEMVs
      // that follow ~3 % (their weights lose cache residency): profiles/r5/decode_mfma1/
      __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (lds_ptr_t)(dst + i * 1024), 16, off[i & 7], 0, 0, 2);
  };
  auto landed = [&]() __attribute__((always_inline)) {  // the oldest K or V tile of the ring is in
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(ND * (2 * ST - 1)) : "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
#pragma unroll
  for (int i = 0; i < ST; ++i) {
    issue(kc, ko, kstart + (w + 4 * i) * KT, mine + i * 2 * TB);
    issue(vc, vo, kstart + (w + 4 * i) * KT, mine + i * 2 * TB + TB);
  }
  [[maybe_unused]] bf16_t kn = 0;
  if constexpr (RP) {
    asm volatile("" : "+v"(rq), "+v"(rk), "+v"(rv), "+v"(rcs));  // (waited for here, the tiles on their way)
    // rotate q (and the new key) at position L - 1, rounded to bf16 like the rope_cache kernel
    auto rot = [&](unsigned x) {
      const float x1 = bf2f((bf16_t)(x & 0xffff)), x2 = bf2f((bf16_t)(x >> 16));
      return f2bf((d & 1) ? x2 * rcs[0] + x1 * rcs[1] : x1 * rcs[0] - x2 * rcs[1]);
    };
    kn = rot(rk);
    if (tid < D) {
      sqb[d] = rot(rq);
      skn[d] = bf2f(kn);
      svn[d] = bf2f((bf16_t)((d & 1) ? rv >> 16 : rv & 0xffff));
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();  // (__syncthreads() would wait for the tiles)
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int ds = 0; ds < NDS; ++ds) qf[ds] = *(const bf16x8_t*)(sqb + ds * 32 + fg * 8);
    if (own_new && w == 0) {  // score of the new key (log2 units)
      float part = 0.f;
      for (int e = lane; e < D; e += 64) part += bf2f(sqb[e]) * skn[e];
      part = wave_sum(part);
      if (lane == 0) *ssn = part * scale_log2e;
    }
  } else {
#pragma unroll
    for (int ds = 0; ds < NDS; ++ds) asm volatile("" : "+v"(qf[ds]));
  }
  // transposed V reads (see the GQA kernel)
  const int vr = 4 * fg + (fr >> 2), vx = vswz<D>(vr) >> 1;
  const unsigned vrow = vr * (D * 2) + ((fr & 3) >> 1) * 16 + (fr & 1) * 8;
  f32x4_t oacc[NDT];
#pragma unroll
  for (int i = 0; i < NDT; ++i) oacc[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  float m_run = -INFINITY, l_part = 0.f;
  int stage = 0;
  for (int t0 = kstart + w * KT; t0 < kend; t0 += 4 * KT) {
    char* kt = mine + stage * 2 * TB;
    char* vt = kt + TB;
    landed();
    bf16x8_t kf[2][NDS];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int ds = 0; ds < NDS; ++ds)
        kf[t][ds] = *(const bf16x8_t*)(kt + (16 * t + fr) * (D * 2) + (((4 * ds + fg) ^ kswz<D>(16 * t + fr)) << 4));
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    issue(kc, ko, t0 + 4 * ST * KT, kt);
    f32x4_t sacc[2] = {f32x4_t{0.f, 0.f, 0.f, 0.f}, f32x4_t{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int ds = 0; ds < NDS; ++ds)
#pragma unroll
      for (int t = 0; t < 2; ++t) sacc[t] = mfma16(kf[t][ds], qf[ds], sacc[t]);
    float mx = -INFINITY;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float sc = t0 + 16 * t + 4 * fg + i < kend ? sacc[t][i] * scale_log2e : -INFINITY;
        sacc[t][i] = sc;
        mx = fmaxf(mx, sc);
      }
    const auto rows = __builtin_amdgcn_permlane16_swap(__float_as_uint(mx), __float_as_uint(mx), false, false);
    mx = max_xhalf(fmaxf(__uint_as_float(rows[0]), __uint_as_float(rows[1])));
    if (__ballot(mx > m_run)) {  // (a new maximum is rare after the first tiles)
      const float m_new = fmaxf(m_run, mx);
      const float alpha = exp2f(m_run - (m_new == -INFINITY ? 0.f : m_new));
      m_run = m_new;
      l_part *= alpha;
#pragma unroll
      for (int i = 0; i < NDT; ++i) oacc[i] *= alpha;
    }
    const float m_use = (m_run == -INFINITY) ? 0.f : m_run;
    unsigned pw[4];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int i = 0; i < 4; i += 2) {
        unsigned x[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {  // this column's 8 bits of the weight
          const float p = __builtin_amdgcn_exp2f(sacc[t][i + j] - m_use);
          l_part += p;
          const float r1 = p - __uint_as_float(__float_as_uint(p) & 0xffff0000u);
          const float r2 = r1 - __uint_as_float(__float_as_uint(r1) & 0xffff0000u);
          x[j] = __float_as_uint(fr == 0 ? p : fr == 1 ? r1 : r2);
        }
        pw[2 * t + i / 2] = __builtin_amdgcn_perm(x[1], x[0], 0x07060302u);
      }
    const bf16x8_t pb = __builtin_bit_cast(bf16x8_t, u32x4_t{pw[0], pw[1], pw[2], pw[3]});
    landed();
    const unsigned va0 = (unsigned)(size_t)(lds_ptr_t)vt + vrow;
    s16x4_t v[2][8];
    constexpr int HT = NDT % 4 ? 3 : 4;  // d-tiles of a block of transposed reads
#pragma unroll
    for (int h = 0; h < NDT / HT; ++h) {
      const int dt = HT * h;
      if constexpr (HT == 4)
        asm volatile("ds_read_b64_tr_b16 %0, %8\n\tds_read_b64_tr_b16 %1, %8 offset:%12\n\t"
                     "ds_read_b64_tr_b16 %2, %9\n\tds_read_b64_tr_b16 %3, %9 offset:%12\n\t"
                     "ds_read_b64_tr_b16 %4, %10\n\tds_read_b64_tr_b16 %5, %10 offset:%12\n\t"
                     "ds_read_b64_tr_b16 %6, %11\n\tds_read_b64_tr_b16 %7, %11 offset:%12\n\ts_waitcnt lgkmcnt(0)"
                     : "=&v"(v[h][0]), "=&v"(v[h][1]), "=&v"(v[h][2]), "=&v"(v[h][3]), "=&v"(v[h][4]), "=&v"(v[h][5]),
                       "=&v"(v[h][6]), "=&v"(v[h][7])
                     : "v"(va0 + ((dt ^ vx) << 5)), "v"(va0 + (((dt + 1) ^ vx) << 5)), "v"(va0 + (((dt + 2) ^ vx) << 5)),
                       "v"(va0 + (((dt + 3) ^ vx) << 5)), "n"(16 * D * 2)
                     : "memory");
      else
        asm volatile("ds_read_b64_tr_b16 %0, %6\n\tds_read_b64_tr_b16 %1, %6 offset:%9\n\t"
                     "ds_read_b64_tr_b16 %2, %7\n\tds_read_b64_tr_b16 %3, %7 offset:%9\n\t"
                     "ds_read_b64_tr_b16 %4, %8\n\tds_read_b64_tr_b16 %5, %8 offset:%9\n\ts_waitcnt lgkmcnt(0)"
                     : "=&v"(v[h][0]), "=&v"(v[h][1]), "=&v"(v[h][2]), "=&v"(v[h][3]), "=&v"(v[h][4]), "=&v"(v[h][5])
                     : "v"(va0 + ((dt ^ vx) << 5)), "v"(va0 + (((dt + 1) ^ vx) << 5)), "v"(va0 + (((dt + 2) ^ vx) << 5)),
                       "n"(16 * D * 2)
                     : "memory");
      if (h == NDT / HT - 1) issue(vc, vo, t0 + 4 * ST * KT, vt);
#pragma unroll
      for (int j = 0; j < HT; ++j) {
        const s16x4_t lo = v[h][2 * j], hi = v[h][2 * j + 1];
        oacc[dt + j] = mfma16(bf16x8_t{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]}, pb, oacc[dt + j]);
      }
    }
    stage = stage + 1 == ST ? 0 : stage + 1;
  }
  // ---- merge the 4 waves (columns 0 - 2: lanes fr < 3) through LDS ----
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (pieces past the end write zeros)
  if (RP && own_new && tid < D) {  // for later steps (read back only after this launch)
    const size_t crow = cbase + (size_t)(L - 1) * D;
    rope.kc[crow + d] = kn;
    rope.vc[crow + d] = (bf16_t)((d & 1) ? rv >> 16 : rv & 0xffff);
  }
  float l_tot = l_part + __shfl_xor(l_part, 16, 64);
  l_tot = sum_xhalf(l_tot);
  if (lane == 0) { swm[w] = m_run; swl[w] = l_tot; }
  __syncthreads();  // every wave is done with its ring
  float* so = (float*)ring;  // [4][3][D]
  if (fr < 3) {
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
      for (int i = 0; i < 4; ++i) so[(w * 3 + fr) * D + dt * 16 + 4 * fg + i] = oacc[dt][i];
  }
  __syncthreads();
  if (tid < D) {
    float M = fmaxf(fmaxf(swm[0], swm[1]), fmaxf(swm[2], swm[3]));
    if (own_new) M = fmaxf(M, *ssn);
    const float Mu = (M == -INFINITY) ? 0.f : M;
    float o = 0.f, ls = 0.f;
#pragma unroll
    for (int ww = 0; ww < 4; ++ww) {
      const float f = exp2f(swm[ww] - Mu);
      // (an infinite value: the upper bits' sum has it, the others' may be 0 times it, NaN)
      const float up = so[(ww * 3) * D + d], low = so[(ww * 3 + 1) * D + d] + so[(ww * 3 + 2) * D + d];
      o += (fabsf(up) < INFINITY ? up + low : up) * f;
      ls += swl[ww] * f;
    }
    if (own_new) {  // the new token's key: weight exp2(s - M), value straight from the qkv row
      const float f = exp2f(*ssn - Mu);
      o += svn[d] * f;
      ls += f;
    }
    dec_store(o, M, ls, b, hk, d, H, nsplit, split, D, po, pm, pl, out, ldo, act);
  }
  dec_finish<D, 1, XC>(po, pm, pl, H, Hkv, nsplit, b, hk, cnt, out, ldo, (int*)(ssn + 1), act);
}

template <int D>
__global__ void decode_combine_kernel(const float* __restrict__ po, const float* __restrict__ pm,
                                      const float* __restrict__ pl, int H, int nsplit, bf16_t* __restrict__ o,
                                      int ldo) {
  const int b = blockIdx.y, h = blockIdx.x;
  const size_t base = ((size_t)b * H + h) * nsplit;
  float M = -INFINITY;
  for (int s = 0; s < nsplit; ++s) M = fmaxf(M, pm[base + s]);
  const float Mu = (M == -INFINITY) ? 0.f : M;
  float lsum = 0.f;
  for (int s = 0; s < nsplit; ++s) lsum += pl[base + s] * exp2f(pm[base + s] - Mu);
  const float inv = lsum > 0.f ? 1.f / lsum : 0.f;
  for (int d = threadIdx.x; d < D; d += blockDim.x) {
    float acc = 0.f;
    for (int s = 0; s < nsplit; ++s) acc += po[(base + s) * D + d] * exp2f(pm[base + s] - Mu);
    o[(size_t)b * ldo + h * D + d] = f2bf(acc * inv);
  }
}

template <int D, int VAR>
static int launch_decode_v(int G, dim3 grid, hipStream_t s, const bf16_t* q, int ldq, const bf16_t* kc,
                           const bf16_t* vc, const int* lens, const int* slot, const int* pre, int H, int Hkv, int max_seq, int chunk,
                           int nsplit, float sl2e, float* po, float* pm, float* pl, bf16_t* out, int ldo,
                           int* cnt, DecRope rope) {
#define DEC(GG) decode_attn_kernel<D, GG, VAR><<<grid, 256, 0, s>>>(q, ldq, kc, vc, lens, slot, pre, H, Hkv, max_seq, \
                                                                     chunk, nsplit, sl2e, po, pm, pl, out, ldo, cnt, rope)
  switch (G) {
    case 1: DEC(1); break;
    case 2: DEC(2); break;
    case 4: DEC(4); break;
    case 8: DEC(8); break;
    default: return (int)hipErrorInvalidValue;
  }
#undef DEC
  return (int)hipGetLastError();
}

// GQA groups (G >= 2) take the MFMA kernel: 1.8x (Llama-3-8B, G=4) to 5x (Llama-3-70B TP=8, G=8)
// over the VALU path (profiles/decode_attn_gqa_mfma_r1.json); the VALU kernel covers the other
// head dims. So does MHA (G = 1), with decode_attn_mfma1_kernel; DA_DECODE_MFMA1=0 gives it the VALU kernel, which
// prefetches each wave's next tile (VAR bit 2) when the launch has few (row, kv head) pairs (B * Hkv <= 32), else streams
// with V issued with K. With G >= 2 the extra V registers cost more occupancy than they buy
// (profiles/decode_attn_variants_r1.json), so those keep V after the scores (nt loads only).
constexpr int kDecPrefetchPairs = 32;

template <int D>
static int launch_decode(int G, dim3 grid, hipStream_t s, const bf16_t* q, int ldq, const bf16_t* kc,
                         const bf16_t* vc, const int* lens, const int* slot, const int* pre, int H, int Hkv, int max_seq, int chunk,
                         int nsplit, float sl2e, float* po, float* pm, float* pl, bf16_t* out, int ldo,
                         int* cnt, DecRope rope, int xc) {
  const int by_len = xc >> 1;  // on MFMA: splits by the row's length (bit 1)
  xc &= 1;
  static int mfma1 = -1;
  if (mfma1 < 0) {
    const char* e = getenv("DA_DECODE_MFMA1");
    mfma1 = (e && e[0] == '0') ? 0 : 1;
  }
  if (mfma1 && G == 1) {
    if (xc && ((grid.y * grid.z) % 8 || !cnt || nsplit < 2)) return (int)hipErrorInvalidValue;
    const dim3 grid_g = by_len && !xc ? dim3(Hkv, grid.z, nsplit) : grid;
#define M1(XCV, RPV) decode_attn_mfma1_kernel<D, XCV, RPV><<<grid_g, 256, 0, s>>>(q, ldq, kc, vc, lens, slot, pre, H, Hkv, \
                         max_seq, chunk, nsplit, sl2e, po, pm, pl, out, ldo, cnt, rope, by_len)
    if (xc) { if (rope.cs) M1(true, true); else M1(true, false); }
    else { if (rope.cs) M1(false, true); else M1(false, false); }
#undef M1
    return (int)hipGetLastError();
  }
  if (by_len && G == 1) chunk = 0x7fffffc0;  // (even splits of any length)
  if (xc) {  // same-XCD split exchange (cached ws / counters): the prefetching MHA form only
    if (G != 1 || (int)(grid.y * grid.z) > kDecPrefetchPairs || (grid.y * grid.z) % 8 || !cnt || nsplit < 2)
      return (int)hipErrorInvalidValue;
    return launch_decode_v<D, 15>(G, grid, s, q, ldq, kc, vc, lens, slot, pre, H, Hkv, max_seq, chunk, nsplit, sl2e, po, pm, pl, out, ldo, cnt, rope);
  }
  if (G == 1) {
    if ((int)(grid.y * grid.z) <= kDecPrefetchPairs)
      return launch_decode_v<D, 7>(G, grid, s, q, ldq, kc, vc, lens, slot, pre, H, Hkv, max_seq, chunk, nsplit, sl2e, po, pm, pl, out, ldo, cnt, rope);
    return launch_decode_v<D, 3>(G, grid, s, q, ldq, kc, vc, lens, slot, pre, H, Hkv, max_seq, chunk, nsplit, sl2e, po, pm, pl, out, ldo, cnt, rope);
  }
  if (rope.cs) return (int)hipErrorInvalidValue;  // fused RoPE: MHA kernel only
  if constexpr (D == 64 || D == 128) {
    const dim3 grid_g = by_len ? dim3(Hkv, grid.z, nsplit) : grid;
    const int pair_rows = nsplit == 1 && !by_len && grid.z <= 64 && Hkv * grid.z > 256 ? 256 / Hkv : 0;
    switch (G) {
      case 2: decode_attn_gqa_kernel<D, 2><<<grid_g, 256, 0, s>>>(q, ldq, kc, vc, lens, slot, pre, H, Hkv, max_seq, chunk, nsplit, sl2e, po, pm, pl, out, ldo, cnt, by_len, pair_rows); break;
      case 4: decode_attn_gqa_kernel<D, 4><<<grid_g, 256, 0, s>>>(q, ldq, kc, vc, lens, slot, pre, H, Hkv, max_seq, chunk, nsplit, sl2e, po, pm, pl, out, ldo, cnt, by_len, pair_rows); break;
      case 8: decode_attn_gqa_kernel<D, 8><<<grid_g, 256, 0, s>>>(q, ldq, kc, vc, lens, slot, pre, H, Hkv, max_seq, chunk, nsplit, sl2e, po, pm, pl, out, ldo, cnt, by_len, pair_rows); break;
      default: return (int)hipErrorInvalidValue;
    }
    return (int)hipGetLastError();
  }
  return launch_decode_v<D, 1>(G, grid, s, q, ldq, kc, vc, lens, slot, pre, H, Hkv, max_seq, chunk, nsplit, sl2e, po, pm, pl, out, ldo, cnt, rope);
}

// ws must hold B*H*nsplit*(D+2) floats. chunk = keys per split (multiple of 64).
// pre (nullable): int32 [B][2] = (P, prefix slot) per row — keys [0, P) of row b are read from the
// prefix slot (a prompt head shared by the whole batch, stored once; P % 64 == 0 so no 64-key tile
// straddles the two sources). Every row of the batch reads the same prefix lines, so they are served
// from L2 / MALL instead of HBM.
// counters (nullable): int32 [B * Hkv], all zero, left zero by every launch -> the splits are merged
// inside the attention kernel (last split per (b, kv head)); null -> separate combine launch. With
// counters, ws and counters must be uncached allocations (da_malloc_uncached).
DA_EXPORT int da_malloc_uncached(long long bytes, void** out) {
  hipError_t e = hipExtMallocWithFlags(out, (size_t)bytes, hipDeviceMallocUncached);
  if (e != hipSuccess) return (int)e;
  e = hipMemset(*out, 0, (size_t)bytes);
  if (e != hipSuccess) return (int)e;
  return (int)hipDeviceSynchronize();
}

// cos_sin / pos (both null, or both set): fused RoPE + new-token KV-cache write (MHA only; q is
// then the raw qkv row, see DecRope).
static int decode_attn_impl(const void* q, int ldq, const void* k_cache, const void* v_cache, const void* lens,
                            const void* slot, const void* pre, int B, int H, int Hkv, int D, int max_seq, int chunk,
                            int nsplit, float scale, void* ws, void* o, int ldo, void* counters, const void* cos_sin,
                            const void* pos, int xc, void* stream) {
  bf16_t* out = (bf16_t*)o;
  int* cnt = (int*)counters;
  if (H % Hkv || chunk % 64 || nsplit < 1 || (long)chunk * nsplit < 1) return (int)hipErrorInvalidValue;
  if ((cos_sin == nullptr) != (pos == nullptr) || (cos_sin && (H != Hkv || ldq < (H + 2 * Hkv) * D)))
    return (int)hipErrorInvalidValue;
  DecRope rope{(bf16_t*)k_cache, (bf16_t*)v_cache, (const float*)cos_sin, (const int*)pos};
  if (B == 0) return 0;
  const int G = H / Hkv;
  float* po = (float*)ws;
  float* pm = po + (size_t)B * H * nsplit * D;
  float* pl = pm + (size_t)B * H * nsplit;
  dim3 grid(nsplit, Hkv, B);
  const float sl2e = scale * 1.4426950408889634f;
  hipStream_t s = (hipStream_t)stream;
  int err;
  switch (D) {
    case 64: err = launch_decode<64>(G, grid, s, (const bf16_t*)q, ldq, (const bf16_t*)k_cache, (const bf16_t*)v_cache,
                                     (const int*)lens, (const int*)slot, (const int*)pre, H, Hkv, max_seq, chunk, nsplit, sl2e, po, pm, pl, out, ldo, cnt, rope, xc);
      break;
    case 96: err = launch_decode<96>(G, grid, s, (const bf16_t*)q, ldq, (const bf16_t*)k_cache, (const bf16_t*)v_cache,
                                     (const int*)lens, (const int*)slot, (const int*)pre, H, Hkv, max_seq, chunk, nsplit, sl2e, po, pm, pl, out, ldo, cnt, rope, xc);
      break;
    case 128: err = launch_decode<128>(G, grid, s, (const bf16_t*)q, ldq, (const bf16_t*)k_cache, (const bf16_t*)v_cache,
                                       (const int*)lens, (const int*)slot, (const int*)pre, H, Hkv, max_seq, chunk, nsplit, sl2e, po, pm, pl, out, ldo, cnt, rope, xc);
      break;
    default: return (int)hipErrorInvalidValue;
  }
  if (err) return err;
  if (nsplit == 1 || cnt) return 0;
  dim3 cgrid(H, B);
  switch (D) {
    case 64: decode_combine_kernel<64><<<cgrid, 64, 0, s>>>(po, pm, pl, H, nsplit, (bf16_t*)o, ldo); break;
    case 96: decode_combine_kernel<96><<<cgrid, 128, 0, s>>>(po, pm, pl, H, nsplit, (bf16_t*)o, ldo); break;
    case 128: decode_combine_kernel<128><<<cgrid, 128, 0, s>>>(po, pm, pl, H, nsplit, (bf16_t*)o, ldo); break;
  }
  DA_LAUNCH_CHECK();
}

// xc = 1: same-XCD split exchange (ws / counters in ordinary device memory; the caller has checked
// the launch's workgroup -> XCD round-robin with the placement probe). 0: uncached ws / counters.
DA_EXPORT int da_decode_attn(const void* q, int ldq, const void* k_cache, const void* v_cache, const void* lens,
                             const void* slot, const void* pre, int B, int H, int Hkv, int D, int max_seq, int chunk,
                             int nsplit, float scale, void* ws, void* o, int ldo, void* counters, const void* cos_sin,
                             const void* pos, int xc, void* stream) {
  return decode_attn_impl(q, ldq, k_cache, v_cache, lens, slot, pre, B, H, Hkv, D, max_seq, chunk, nsplit, scale, ws,
                          o, ldo, counters, cos_sin, pos, xc, stream);
}

// Dispatch order of the flash kernels (FaPrefix::rev, fa_block): causal longest query blocks first
// and the query blocks of one (sequence, kv head) pair on one XCD (737 -> 778 TF/s on the Phi-3 QA
// chunk, profiles/r4/flash_order/).
constexpr int kFaDispatch = 3;

// The encoders' kernel takes bidirectional attention over own keys, D = 64, rows that 16-B accesses can reach and a tile's rows
// within 2 GiB.
template <typename T>
static bool launch_fa_enc(const void* q, const void* k, const void* v, int ldq, int ldk, int ldv, const void* cu, int B,
                          int max_seqlen, int H, int Hkv, float sl2e, void* o, int ldo, hipStream_t s) {
  if (ldo % 8 || ((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)o) % 16 || max(max(ldq, ldk), ldv) > 1 << 22) return false;
  flash_attn_enc_kernel<T><<<dim3((max_seqlen + 127) / 128, H, B), 256, 0, s>>>((const bf16_t*)q, (const bf16_t*)k,
      (const bf16_t*)v, ldq, ldk, ldv, (const int*)cu, H, Hkv, sl2e, (bf16_t*)o, ldo, kFaDispatch);
  return true;
}

// fp16 (the encoder's DTYPE=fp16): bidirectional or causal, no shared prefix, 4 waves x 32 queries
DA_EXPORT int da_flash_attn_f16(const void* q, const void* k, const void* v, int ldq, int ldk, int ldv,
                                const void* cu_seqlens, int B, int max_seqlen, int H, int Hkv, int D, int causal,
                                float scale, void* o, int ldo, void* stream) {
  if (H % Hkv || ldq % 8 || ldk % 8 || ldv % 8 || ldo % 4) return (int)hipErrorInvalidValue;
  if (B == 0 || max_seqlen == 0) return 0;
  const FaPrefix pre{nullptr, nullptr, 0, 0, kFaDispatch};
  dim3 grid((max_seqlen + 127) / 128, H, B);
  hipStream_t s = (hipStream_t)stream;
  if (D == 64 && !causal && launch_fa_enc<F16T>(q, k, v, ldq, ldk, ldv, cu_seqlens, B, max_seqlen, H, Hkv,
                                                scale * 1.4426950408889634f, o, ldo, s))
    return (int)hipGetLastError();
#define FA_ARGS16 (const bf16_t*)q, (const bf16_t*)k, (const bf16_t*)v, ldq, ldk, ldv, (const int*)cu_seqlens, H, Hkv, \
                  causal, scale * 1.4426950408889634f, (bf16_t*)o, ldo, pre
  switch (D) {
    case 64: flash_attn_v2_kernel<64, 4, 1, F16T><<<grid, 256, FA2Cfg<64, 4, 1>::SMEM, s>>>(FA_ARGS16); break;
    case 96: flash_attn_v2_kernel<96, 4, 1, F16T><<<grid, 256, FA2Cfg<96, 4, 1>::SMEM, s>>>(FA_ARGS16); break;
    default: return (int)hipErrorInvalidValue;
  }
#undef FA_ARGS16
  return (int)hipGetLastError();
}

template <int NW, int QH>
static int launch_fa2(const void* q, const void* k, const void* v, int ldq, int ldk, int ldv, const void* cu_seqlens,
                      int B, int max_seqlen, int H, int Hkv, int D, int causal, float sl2e, void* o, int ldo,
                      FaPrefix pre, hipStream_t s) {
  static bool attr_set = false;
  if constexpr (NW * QH <= 8) {
    if (!attr_set) {
      (void)hipFuncSetAttribute((const void*)flash_attn_v2_kernel<128, NW, QH>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                FA2Cfg<128, NW, QH>::SMEM);
      attr_set = true;
    }
  }
  dim3 grid((max_seqlen + 32 * QH * NW - 1) / (32 * QH * NW), H, B);
#define FA_ARGS (const bf16_t*)q, (const bf16_t*)k, (const bf16_t*)v, ldq, ldk, ldv, (const int*)cu_seqlens, H, Hkv, \
                causal, sl2e, (bf16_t*)o, ldo, pre
  switch (D) {
    case 32: flash_attn_v2_kernel<32, NW, QH><<<grid, 64 * NW, FA2Cfg<32, NW, QH>::SMEM, s>>>(FA_ARGS); break;
    case 64: flash_attn_v2_kernel<64, NW, QH><<<grid, 64 * NW, FA2Cfg<64, NW, QH>::SMEM, s>>>(FA_ARGS); break;
    // 8 waves x 64 queries exceed 256 VGPRs (spills) above D = 64: not instantiated
    case 96:
      if constexpr (NW * QH <= 8) flash_attn_v2_kernel<96, NW, QH><<<grid, 64 * NW, FA2Cfg<96, NW, QH>::SMEM, s>>>(FA_ARGS);
      else return (int)hipErrorInvalidValue;
      break;
    case 128:
      if constexpr (NW * QH <= 8) flash_attn_v2_kernel<128, NW, QH><<<grid, 64 * NW, FA2Cfg<128, NW, QH>::SMEM, s>>>(FA_ARGS);
      else return (int)hipErrorInvalidValue;
      break;
    default: return (int)hipErrorInvalidValue;
  }
#undef FA_ARGS
  return (int)hipGetLastError();
}

// Causal D = 96 (the Phi-3 prefill) runs the software-pipelined kernel (flash_attn_pipe: 576 -> 656
// TF/s; the short bidirectional BGE sequences, 8 tiles, lose to its longer pipeline fill, 617 -> 531
// at D = 64, profiles/r2/attn_bench_v5.txt) with the speculative softmax (654 -> 689 TF/s,
// profiles/r3/attn_bench_spec.txt) and LDS-DMA K / V tiles when the prefix is whole 64-key tiles and
// the operands 16-B aligned (711 TF/s); every other shape the 4-wave flash_attn_v2_kernel (8 waves
// at D = 128 where fa_eight_waves).
template <int D, bool DMA>
static constexpr int fa_pipe_smem() {
  return 3 * ((DMA ? 64 * D * 2 : FA2Cfg<D, 4, 1>::KBUF) + FA2Cfg<D, 4, 1>::VBUF);
}

template <bool DMA>
static int launch_fa_pipe(const void* q, const void* k, const void* v, int ldq, int ldk, int ldv, const void* cu_seqlens,
                          int B, int max_seqlen, int H, int Hkv, int causal, float sl2e, void* o, int ldo,
                          FaPrefix pre, hipStream_t s) {
  static bool attr_set = false;
  if (!attr_set) {
    (void)hipFuncSetAttribute((const void*)flash_attn_pipe_kernel<96, true, DMA>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, fa_pipe_smem<96, DMA>());
    attr_set = true;
  }
  dim3 grid((max_seqlen + 127) / 128, H, B);
  flash_attn_pipe_kernel<96, true, DMA><<<grid, 256, fa_pipe_smem<96, DMA>(), s>>>(
      (const bf16_t*)q, (const bf16_t*)k, (const bf16_t*)v, ldq, ldk, ldv, (const int*)cu_seqlens, H, Hkv, causal, sl2e,
      (bf16_t*)o, ldo, pre);
  return (int)hipGetLastError();
}

// D = 128: 256 queries a workgroup, two waves a SIMD that share the staged tiles, or 128 and one. A tile's chain (scores, exponentials,
// sums) is what a workgroup takes its time for, so one wave a SIMD is nearly twice as fast where the chip has workgroups to spare,
// and shorter blocks leave less behind the causal diagonal and the texts' ends; with many blocks the tiles' second reading costs more, the more
// the longer the shared head (pre) that all of them walk and the less the diagonal is of that. Both give the same bits.
// us, 8 waves / 4, 32 heads over 8: 139 + 138 queries behind 320 keys 21.9 / 18.6, 277 16.2 / 12.5, 820 31.1 / 25.0, 1750 62.2 / 52.0, 1900 + 2000 +
// 1700 behind 256 171 / 161, 64 x 100 behind 256 129 / 80, 2048 65 / 57, behind 1024 100 / 93, 2560 82 / 73, 2816 91 / 83; 3072 99 / 100,
// 3600 135 / 146, 8192 560 / 590, 2 x 2560 136 / 139, 6 x 3000 620 / 630.
// Blocks that have a CU each: 700 behind 4096 151 / 127, behind 16384 533 / 487. One round of both, a long head: 1500 behind 4096 181 / 177, behind 16384
// 556 / 597, 2048 behind 4096 202 / 208; 64 heads over 8, 507 + 350 behind 3000 126 / 137; 40 heads, 481 + 360 + 250 behind 3000 122 / 133. More of
// them: 2 x 2048 behind 1024 and 4096 157 / 174 and 370 / 402, 16 x 1500 864 / 904 and 2111 / 2269, 2560 behind 1024 122 / 142; of shorter texts by
// their lengths, 8 to 882 behind 3000 480 / 402, 16 to 484 875 / 792, 16 x 700 behind 4096 950 / 1032.
static bool fa_eight_waves(int max_seqlen, int H, int B, int pre_len) {
  const auto blocks = [&](int n, int rows) { return (long)((n + rows - 1) / rows) * H * B; };
  if (max_seqlen > 2816 || (max_seqlen > 2048 && blocks(max_seqlen, 256) > 400)) return true;
  const int some = B > 1 ? (max_seqlen * 3 + 3) / 4 : max_seqlen;  // (the others' lengths are not known here)
  if (blocks(some, 128) <= 256) return false;
  if (blocks(some, 256) <= 256) return pre_len > max_seqlen / 2 * 3;
  return max_seqlen > 1408 && pre_len >= 512;
}

// pre_k / pre_v: shared-prefix K/V of KV head 0 in a cache slot (nullptr / pre_len 0: none),
// pre_hstride: elements between KV heads there (max_seq * D).
// kv_slot / kv_pos (nullable; per token, int32): the sequences' own keys are read from the KV cache
// k_cache / v_cache [slots, Hkv, max_seq, D] (pre_hstride = max_seq * D) instead of k / v — causal
// D = 96 only.
DA_EXPORT int da_flash_attn_v2(const void* q, const void* k, const void* v, int ldq, int ldk, int ldv,
                               const void* cu_seqlens, int B, int max_seqlen, int H, int Hkv, int D, int causal,
                               float scale, void* o, int ldo, const void* pre_k, const void* pre_v,
                               long long pre_hstride, int pre_len, const void* kv_slot, const void* kv_pos,
                               const void* k_cache, const void* v_cache, void* stream) {
  const bool from_cache = kv_slot != nullptr;
  if (from_cache) {
    if (!causal || D != 96 || !kv_pos || !k_cache || !v_cache || pre_hstride < (long long)D ||
        pre_hstride % D || ((uintptr_t)k_cache | (uintptr_t)v_cache) % 16)
      return (int)hipErrorInvalidValue;
    k = k_cache; v = v_cache; ldk = ldv = D;  // rows D apart inside a (slot, head) block
  }
  if (H % Hkv || ldq % 8 || ldk % 8 || ldv % 8 || ldo % 4) return (int)hipErrorInvalidValue;
  if (pre_len < 0 || (pre_len > 0 && (!pre_k || !pre_v || pre_hstride < (long long)pre_len * D)))
    return (int)hipErrorInvalidValue;
  if (B == 0 || max_seqlen == 0) return 0;
  const float sl2e = scale * 1.4426950408889634f;
  hipStream_t s = (hipStream_t)stream;
  const FaPrefix pre{(const bf16_t*)pre_k, (const bf16_t*)pre_v, pre_hstride, pre_len, kFaDispatch,
                     (const int*)kv_slot, (const int*)kv_pos, (const bf16_t*)k_cache, (const bf16_t*)v_cache,
                     from_cache ? (long long)Hkv * pre_hstride : 0LL};
  if (causal && D == 96) {
    const bool dma = pre_len % 64 == 0 && ((uintptr_t)k | (uintptr_t)v | (uintptr_t)pre_k | (uintptr_t)pre_v) % 16 == 0;
    if (dma) return launch_fa_pipe<true>(q, k, v, ldq, ldk, ldv, cu_seqlens, B, max_seqlen, H, Hkv, causal, sl2e, o, ldo, pre, s);
    return launch_fa_pipe<false>(q, k, v, ldq, ldk, ldv, cu_seqlens, B, max_seqlen, H, Hkv, causal, sl2e, o, ldo, pre, s);
  }
  if (D == 64 && !causal && pre_len == 0 &&
      launch_fa_enc<BF16T>(q, k, v, ldq, ldk, ldv, cu_seqlens, B, max_seqlen, H, Hkv, sl2e, o, ldo, s))
    return (int)hipGetLastError();
  if (D == 128 && fa_eight_waves(max_seqlen, H, B, pre_len))
    return launch_fa2<8, 1>(q, k, v, ldq, ldk, ldv, cu_seqlens, B, max_seqlen, H, Hkv, D, causal, sl2e, o, ldo, pre, s);
  return launch_fa2<4, 1>(q, k, v, ldq, ldk, ldv, cu_seqlens, B, max_seqlen, H, Hkv, D, causal, sl2e, o, ldo, pre, s);
}
