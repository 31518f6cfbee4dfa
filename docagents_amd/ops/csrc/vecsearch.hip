// In-HBM vector index kernels: cosine similarity (dot product of L2-normalised bf16 rows) fused
// with the document filter, the similarity floor and a per-workgroup top-k select, then a
// second-pass merge. Replaces pgvector's `1 - (v <=> q) >= 0.7 ... ORDER BY ... LIMIT k` with
// `WHERE document_id = ANY(...)` (internal/store/postgres.go:218-285).
//
//  * topk_dense:  batched queries x all rows as MFMA tiles (16 rows x 16 queries per wave-MFMA),
//                 doc filter as a per-query bitmap over the shard's local doc slots. Also used for
//                 IVF coarse probing (rows = centroids) and k-means assignment (k = 1).
//  * topk_ranges: per-query row ranges (rows of a document are contiguous in the shard, and IVF
//                 lists are contiguous runs) — only the rows a query can match are read.
//  * topk_merge:  per query, select the global top-k over all workgroups' candidates (sorted desc,
//                 ties -> smaller row id first).
//  * kmeans_accum: centroid sums / counts for IVFFlat training (fp32 atomics, 256-B rows).
#include <cstring>
#include <type_traits>

#include "common.h"

#define TK_MAX 32

__device__ __forceinline__ bool better(float a, int ia, float b, int ib) {
  return a > b || (a == b && ia >= 0 && (ib < 0 || ia < ib));
}

// Merge 64 new candidates (one per lane: a/ia) into a running sorted top-K list held in LDS
// (best/bidx, K entries) — executed by one full wave.
__device__ __forceinline__ void wave_merge_topk(float a, int ia, float* best, int* bidx, int K, int lane) {
  const float kth = best[K - 1];
  const int kthi = bidx[K - 1];
  // early exit: nothing beats the current k-th
  const bool cand = better(a, ia, kth, kthi) && a != -INFINITY;
  if (__ballot(cand) == 0ull) return;
  float b = lane < K ? best[lane] : -INFINITY;
  int ib = lane < K ? bidx[lane] : -1;
  float outv = -INFINITY;
  int outi = -1;
  for (int r = 0; r < K; ++r) {
    // local best of (a, b)
    float v; int vi; int which;
    if (better(a, ia, b, ib)) { v = a; vi = ia; which = 0; } else { v = b; vi = ib; which = 1; }
    if (v == -INFINITY) { vi = -1; }
    float wv = v; int wi = vi; int wl = lane;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      const float ov = __shfl_xor(wv, o, 64);
      const int oi = __shfl_xor(wi, o, 64);
      const int ol = __shfl_xor(wl, o, 64);
      if (better(ov, oi, wv, wi) || (ov == wv && oi == wi && ol < wl)) { wv = ov; wi = oi; wl = ol; }
    }
    if (lane == r) { outv = wv; outi = (wv == -INFINITY) ? -1 : wi; }
    if (lane == wl) {
      if (which == 0) { a = -INFINITY; ia = -1; } else { b = -INFINITY; ib = -1; }
    }
  }
  if (lane < K) { best[lane] = outv; bidx[lane] = outi; }
}

// X [N, d] bf16 rows, slots [N] local doc slot per row (or null), Qv [Q, d] bf16, bitmap [Q, W] (or null)
// out_s / out_i : [gridDim.x, Q, K]
__global__ void __launch_bounds__(256)
topk_dense_kernel(const bf16_t* __restrict__ X, int N, int d, const int* __restrict__ slots,
                  const bf16_t* __restrict__ Qv, int Q, const unsigned* __restrict__ bitmap, int W, float thr,
                  int K, int rows_per_block, float* __restrict__ out_s, int* __restrict__ out_i) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int qstr = d * 2 + 16;
  char* sQ = smem;                                   // [16][d] bf16 padded
  float* sc = (float*)(smem + 16 * qstr);            // [16][64 + 1]
  float* best = sc + 16 * 65;                        // [16][TK_MAX]
  int* bidx = (int*)(best + 16 * TK_MAX);            // [16][TK_MAX]

  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int fr = lane & 15, fg = lane >> 4;
  const int qbase = blockIdx.y * 16;
  const int nq = min(16, Q - qbase);
  for (int i = tid; i < 16 * (d / 8); i += 256) {
    const int r = i / (d / 8), c = i % (d / 8);
    u32x4_t v = u32x4_t{0, 0, 0, 0};
    if (r < nq) v = *(const u32x4_t*)(Qv + (size_t)(qbase + r) * d + c * 8);
    *(u32x4_t*)(sQ + r * qstr + c * 16) = v;
  }
  for (int i = tid; i < 16 * TK_MAX; i += 256) { best[i] = -INFINITY; bidx[i] = -1; }
  __syncthreads();

  const int rbeg = blockIdx.x * rows_per_block;
  const int rend = min(N, rbeg + rows_per_block);
  const int nkk = d / 32;
  for (int r0 = rbeg; r0 < rend; r0 += 64) {
    // ---- S[row][q] for this wave's 16 rows ----
    const int row_a = r0 + wid * 16 + fr;
    f32x4_t acc = f32x4_t{0.f, 0.f, 0.f, 0.f};
    const bf16_t* xr = X + (size_t)(row_a < N ? row_a : 0) * d + fg * 8;
    for (int kk = 0; kk < nkk; ++kk) {
      bf16x8_t a = *(const bf16x8_t*)(xr + kk * 32);
      if (row_a >= rend) a = bf16x8_t{0, 0, 0, 0, 0, 0, 0, 0};
      const bf16x8_t bq = *(const bf16x8_t*)(sQ + fr * qstr + kk * 64 + fg * 16);
      acc = mfma16(a, bq, acc);
    }
    const int q = fr;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int rl = wid * 16 + fg * 4 + i;
      const int row = r0 + rl;
      float s = acc[i];
      bool ok = row < rend && q < nq && s >= thr;
      if (ok && slots) {  // removed rows (slot -1) never match; the bitmap (if any) filters documents
        const int sl = slots[row];
        ok = sl >= 0 && (!bitmap || ((sl >> 5) < W && ((bitmap[(size_t)(qbase + q) * W + (sl >> 5)] >> (sl & 31)) & 1u)));
      }
      sc[q * 65 + rl] = ok ? s : -INFINITY;
    }
    __syncthreads();
    // ---- merge into running per-query top-K: wave w owns queries w, w+4, w+8, w+12 ----
    for (int qq = wid; qq < nq; qq += 4) {
      const float a = sc[qq * 65 + lane];
      wave_merge_topk(a, r0 + lane, best + qq * TK_MAX, bidx + qq * TK_MAX, K, lane);
    }
    __syncthreads();
  }
  for (int i = tid; i < nq * K; i += 256) {
    const int qq = i / K, j = i % K;
    const size_t o = ((size_t)blockIdx.x * Q + qbase + qq) * K + j;
    out_s[o] = best[qq * TK_MAX + j];
    out_i[o] = bidx[qq * TK_MAX + j];
  }
}

// ------------------------------------------------------------------------------------------------
// Streaming dense scan (d = 384, 768, 1024): the whole-shard pass of flat search and IVF coarse probing, built to run at HBM
// speed. In two launches:
//  1. a scan that leaves, per query, the best score of every group of 16 rows (a power of two of them from 65536 groups on)
//     that the filter and the floor let pass: four selects, two cross-lane steps and a store of 4 B per group and query;
//  2. topk_pick_kernel: the K best groups of a query hold its K best rows (whoever is in another group has K groups before
//     it, each with a better row, or an equal one of a smaller id); it scores those groups again, with the scan's own
//     instructions, and orders the rows.
// A top-K list kept beside the scan starts empty in every workgroup, so with a few hundred to a few thousand rows each nearly
// every tile held a row that beat the list so far: appending, cutting and merging took 20 - 85 % of a pass. Whole searches, us,
// lists / groups (few rows: scores, see scan_plan): 1.25 M x 1024, K = 5, 1 query 506 / 395, 16 600 / 417, 64 708 / 443, 128
// 795 / 496; 411812 x 768, 113 queries, K = 5 309 / 148, K = 20 518 / 161; 75595 x 384, 36 queries, K = 19 159 / 33; 30000 x
// 1024, 20 queries 69 / 29; 512 x 768 (centroids), 24 queries 27 / 12.
__device__ __forceinline__ unsigned td_key(float v, int id) {  // larger = better; empty (id < 0) = 0
  const unsigned u = __float_as_uint(v + 0.f);  // (-0 as 0)
  return id < 0 ? 0u : ((u & 0x80000000u) ? ~u : (u | 0x80000000u));
}
__device__ __forceinline__ float td_unkey(unsigned k) {
  return k == 0u ? -INFINITY : __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}
__device__ __forceinline__ void wave_sync_lds() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The top K of the wave's 64 (v, id) (one per lane; id < 0 = empty) into cs/ci[0, K) of a list, unsorted, empty
// places behind them. Returns a bound that the K-th best reaches and the next one does not (-inf while fewer than K
// are real). Every lane must have read what it passes before the call (the list slots are overwritten).
// The masks are uniform (scalar unit), and the rounds end at the bit that tells the K-th best from the next: about
// 16 of 32 rounds for scores of one magnitude.
__device__ __forceinline__ float td_cut(float v, int id, int K, int lane, float* cs, int* ci) {
  const unsigned key = td_key(v, id);
  unsigned long long act = __ballot(key != 0u), sel = 0ull;
  unsigned T = 0;  // prefix of the K-th largest key
  int need = K;
  if (__popcll(act) <= K) {
    sel = act;
    need = 0;
  }
  for (int bt = 31; bt >= 0 && need > 0; --bt) {
    const unsigned long long one = __ballot((key >> bt) & 1u) & act;
    const int c = __popcll(one);
    if (c >= need) T |= 1u << bt;
    if (c > need) {
      act = one;
    } else {
      sel |= one;
      need -= c;
      act &= ~one;
    }
  }
  for (; need > 0; --need) {  // exact ties at the threshold (rare): smallest row ids first
    int m = ((act >> lane) & 1ull) ? id : 0x7fffffff;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) m = min(m, __shfl_xor(m, o, 64));
    unsigned long long w = __ballot(((act >> lane) & 1ull) && id == m);
    w &= ~w + 1;
    sel |= w;
    act &= ~w;
  }
  const int pos = __builtin_amdgcn_mbcnt_hi((unsigned)(sel >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)sel, 0u));
  const int real = __popcll(sel);
  wave_sync_lds();
  if ((sel >> lane) & 1ull) { cs[pos] = v; ci[pos] = id; }
  if (lane >= real && lane < K) { cs[lane] = -INFINITY; ci[lane] = -1; }
  wave_sync_lds();
  const float t = td_unkey(T);
  return t != t ? -INFINITY : t;  // (a prefix below -FLT_MAX)
}


// What a scan leaves of a run of 16-row tiles for a wave's 16 queries: lane (fr, fg) of query fr keeps groups 4 fg .. 4 fg + 3
// of every 16 and stores them together. A run's groups are padded to a multiple of 4 with -inf. lg < 0: its rows' scores
// instead, padded to whole tiles.
struct GroupMax {
  float* line;  // this lane's query's groups of this run; null: no such query
  int slots, lg, g;  // groups of a run (padded), log2 of a group's tiles, groups so far
  f32x4_t keep;
  float best;

  __device__ __forceinline__ void init(float* l, int n, int log_tiles) {
    line = l; slots = n; lg = log_tiles; g = 0;
    best = -INFINITY;
    keep = f32x4_t{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
  }
  __device__ __forceinline__ void flush(int at, int fg) {
    if (line && at + 4 * fg < slots) *(f32x4_t*)(line + at + 4 * fg) = keep;
    keep = f32x4_t{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
  }
  __device__ __forceinline__ void close(int fg) {  // the group ends
    const int own = (g >> 2) & 3;
#pragma unroll
    for (int i = 0; i < 4; ++i) keep[i] = fg == own && (g & 3) == i ? best : keep[i];
    best = -INFINITY;
    if ((++g & 15) == 0) flush(g - 16, fg);
  }
  // tile t of the run: lane (fr, fg) holds the scores of rows row0 .. row0 + 3 (row0 = its first row + 4 fg) whose doc slots
  // are sl (removed rows: -1); rows from `end` on are padding
  __device__ __forceinline__ void tile(const f32x4_t& acc, int t, int row0, int end, float thr, const int (&sl)[4],
                                       const unsigned* __restrict__ bits, int W, int fg) {
    f32x4_t s;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      bool ok = row0 + i < end && sl[i] >= 0 && acc[i] >= thr;
      if (bits && ok) ok = (sl[i] >> 5) < W && ((bits[sl[i] >> 5] >> (sl[i] & 31)) & 1u);
      s[i] = ok ? acc[i] : -INFINITY;
    }
    if (lg < 0) {  // every row's score
      if (line) *(f32x4_t*)(line + t * 16 + 4 * fg) = s;
      return;
    }
    const float m = fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3]));
    const auto rows = __builtin_amdgcn_permlane16_swap(__float_as_uint(m), __float_as_uint(m), false, false);
    best = fmaxf(best, max_xhalf(fmaxf(__uint_as_float(rows[0]), __uint_as_float(rows[1]))));
    if (((t + 1) & ((1 << lg) - 1)) == 0) close(fg);
  }
  __device__ __forceinline__ void finish(int tiles, int fg) {
    if (lg < 0) {
      for (int t = tiles; t * 16 < slots; ++t)
        if (line) *(f32x4_t*)(line + t * 16 + 4 * fg) = keep;
      return;
    }
    if (tiles & ((1 << lg) - 1)) close(fg);
    for (int at = g & ~15; at < slots; at += 16) flush(at, fg);
  }
};

typedef __attribute__((address_space(3))) void* vs_lds_t;

// Up to 16 queries: a wave has a run of rows to itself. A tile is 16 rows x d in LDS, by LDS-DMA in column groups of 128 (256 B
// of a row: 16-B chunk c of row r at c ^ r), and a group's place is filled with the next tile's as soon as its fragments are
// in registers: no barrier, counted waits; the queries' fragments stay in registers.
// (Rows loaded straight into the MFMA's A registers are requests of 64 B, of which a CU has no more on their way than of
// whole lines.)
// Bound by HBM: 1.25 M x 1024 at 6.5 TB/s with one query, 6.1 with 16 (5.1 and 4.3 by registers, with lists).
template <int NG>
__global__ void __launch_bounds__(256, 1)
topk_dense_stream_kernel(const bf16_t* __restrict__ X, int N, const int* __restrict__ slots,
                         const bf16_t* __restrict__ Qv, int Q, const unsigned* __restrict__ bitmap, int W, float thr,
                         int rows_per_wave, float* __restrict__ gm, int GT, int run_slots, int lg) {
  constexpr int d = NG * 128, RB = d * 2, NK = d / 32, TB = 16 * RB;
  __shared__ __attribute__((aligned(16))) char sX[4 * TB];
  __shared__ __attribute__((aligned(16))) int sS[4][2][64];  // doc slots of this tile and the next
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int fr = lane & 15, fg = lane >> 4;
  const int run = blockIdx.x * 4 + w;
  const int beg = (int)min((long)N, (long)run * rows_per_wave), end = (int)min((long)N, (long)beg + rows_per_wave);
  const int ntile = (end - beg + 15) / 16;
  if (!ntile) return;  // (no barrier below)
  bf16x8_t bq[NK];
#pragma unroll
  for (int kk = 0; kk < NK; ++kk) bq[kk] = *(const bf16x8_t*)(Qv + (size_t)min(fr, Q - 1) * d + kk * 32 + fg * 8);
  const __amdgpu_buffer_rsrc_t rx =
      __builtin_amdgcn_make_buffer_rsrc((void*)(X + (size_t)beg * d), (short)0, (end - beg) * RB, 0x00020000);
  const __amdgpu_buffer_rsrc_t rs =
      __builtin_amdgcn_make_buffer_rsrc((void*)(slots ? slots + beg : (const int*)X), (short)0, slots ? (end - beg) * 4 : 0, 0x00020000);
  unsigned off[4];  // 1 KiB instruction i: rows 4 i .. 4 i + 3 of the group
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = 4 * i + (lane >> 4);
    off[i] = (unsigned)(r * RB + (((lane & 15) ^ r) << 4));
  }
  char* mine = sX + w * TB;
  auto issue = [&](int t, int g) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (vs_lds_t)(mine + g * 4096 + i * 1024), 16, off[i], t * TB + g * 256, 0, 2);
  };
  auto issue_slots = [&](int t) __attribute__((always_inline)) {  // (rows behind the tile's: out of range or unused)
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (vs_lds_t)(&sS[w][t & 1][0]), 4, lane * 4, t * 64, 0, 0);
  };
  issue_slots(0);
#pragma unroll
  for (int g = 0; g < NG; ++g) issue(0, g);
#pragma unroll
  for (int kk = 0; kk < NK; ++kk) asm volatile("" : "+v"(bq[kk]));  // (waited for here, the tile on its way)
  GroupMax gx;
  gx.init(fr < Q ? gm + (size_t)fr * GT + (size_t)run * run_slots : nullptr, run_slots, lg);
  const unsigned* bits = bitmap ? bitmap + (size_t)min(fr, Q - 1) * W : nullptr;
  for (int t = 0; t < ntile; ++t) {
    f32x4_t acc = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"(4 * (NG - 1)) : "memory");  // this group is in; NG - 1 newer ones at least
      __builtin_amdgcn_sched_barrier(0);
      bf16x8_t a[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) a[j] = *(const bf16x8_t*)(mine + g * 4096 + fr * 256 + (((4 * j + fg) ^ fr) << 4));
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      if (g == 0) issue_slots(t + 1);
      issue(t + 1, g);
#pragma unroll
      for (int j = 0; j < 4; ++j) acc = mfma16(a[j], bq[4 * g + j], acc);
    }
    int sl[4] = {0, 0, 0, 0};
    if (slots) {
#pragma unroll
      for (int i = 0; i < 4; ++i) sl[i] = sS[w][t & 1][4 * fg + i];
    }
    gx.tile(acc, t, beg + t * 16 + fg * 4, end, thr, sl, bits, W, fg);
  }
  gx.finish(ntile, fg);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // pieces past the end write zeros: in before the workgroup's LDS goes
}

// 17 and more queries: NW waves of 16 queries each per workgroup (8 from 65 queries on, so that a shard is read once
// for up to 128) over the SAME rows. rows_per_block rows per workgroup (multiple of 16), grid = row blocks (padded to 8) x
// query groups: the nqg groups of one row block are dispatched to one XCD back to back. A stage: 16 rows (d = 384: 32) and
// their doc slots by LDS-DMA (16-B chunk c of row r at c ^ (r & 15): the 16 rows one ds_read_b128 lane group reads hit 16
// distinct slots; the slots to each wave's own words), a ring of 2 - 5 stages, one barrier a stage. The queries' fragments
// stay in registers (d / 8 of them). 1.25 M x 1024: 6.0 TB/s with 17 queries, 5.8 with 64, 5.4 with 128, where a CU's LDS reads
// (each wave reads the whole stage) and its MFMAs take about as long as its stages; the DMA instructions spread between the
// MFMAs, two chains of them, or four waves of 32 queries each were slower (594 - 657 us for 496). A stage's transfers are asked for
// behind its products: in front of them all waves wait for one another's requests before their first read (us, in front / behind,
// whole searches: 1.25 M x 1024, 128 queries 497 / 478, 96 492 / 467, 64 435 / 433; 600000 x 768, 128 218 / 197, 40 175 / 172; 600000 x 384,
// 128 140 / 134; 100000 x 1024, 100 58.6 / 55.4; 30000 x 384, 90 21.9 / 22.0).
template <int NG, int NW>
__global__ void __launch_bounds__(64 * NW, 2)
topk_dense_mq_kernel(const bf16_t* __restrict__ X, int N, const int* __restrict__ slots,
                     const bf16_t* __restrict__ Qv, int Q, const unsigned* __restrict__ bitmap, int W, float thr,
                     int rows_per_block, int nqg, float* __restrict__ gm, int GT, int run_slots, int lg) {
  constexpr int d = NG * 128, NK = d / 32, CPR = d / 8, RB = d * 2;
  constexpr int TR = NG == 3 ? 2 : 1, STAGE = TR * 16 * RB, P1 = STAGE / 1024 / NW, P = P1 + 1;
  constexpr int LDS = NW == 8 ? 160 * 1024 : 80 * 1024, SL = NW * 256;
  constexpr int ST = LDS / (STAGE + SL) < 5 ? LDS / (STAGE + SL) : 5;
  static_assert(STAGE % (1024 * NW) == 0 && ST >= 2 && P1 <= 8, "stage");
  __shared__ __attribute__((aligned(16))) char sX[ST * (STAGE + SL)];

  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int fr = lane & 15, fg = lane >> 4;
  const int b = blockIdx.x, per = 8 * nqg;
  const int grp = b / per, rem = b % per;
  const int qg = rem / 8, rb = grp * 8 + rem % 8;
  const int q = (qg * NW + w) * 16 + fr;
  const int beg = (int)min((long)N, (long)rb * rows_per_block), end = (int)min((long)N, (long)beg + rows_per_block);
  const int ntile = (end - beg + 15) / 16, nst = (ntile + TR - 1) / TR;
  if (!nst) return;  // whole workgroup
  // this wave's B fragments: query q, columns 32 kk + 8 fg .. + 8
  bf16x8_t bq[NK];
#pragma unroll
  for (int kk = 0; kk < NK; ++kk) bq[kk] = *(const bf16x8_t*)(Qv + (size_t)min(q, Q - 1) * d + kk * 32 + fg * 8);
  // rows past the workgroup's last are zeros (masked in GroupMax::tile); no slots: an empty resource
  const __amdgpu_buffer_rsrc_t rx =
      __builtin_amdgcn_make_buffer_rsrc((void*)(X + (size_t)beg * d), (short)0, (end - beg) * RB, 0x00020000);
  const __amdgpu_buffer_rsrc_t rs =
      __builtin_amdgcn_make_buffer_rsrc((void*)(slots ? slots + beg : (const int*)X), (short)0, slots ? (end - beg) * 4 : 0, 0x00020000);
  unsigned off[8];
#pragma unroll
  for (int j = 0; j < P1; ++j) {
    const int idx = (w * P1 + j) * 64 + lane, r = idx / CPR, c = idx % CPR;
    off[j] = (unsigned)(r * RB + ((c ^ (r & 15)) << 4));
  }
  auto issue = [&](int t, int stage) __attribute__((always_inline)) {
    char* dst = sX + stage * (STAGE + SL);
#pragma unroll
    for (int j = 0; j < P1; ++j)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (vs_lds_t)(dst + (w * P1 + j) * 1024), 16, off[j & 7], t * STAGE, 0, 2);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (vs_lds_t)(dst + STAGE + w * 256), 4, lane * 4, t * (64 * TR), 0, 0);
  };
#pragma unroll
  for (int i = 0; i < ST - 1; ++i) issue(i, i);
#pragma unroll
  for (int kk = 0; kk < NK; ++kk) asm volatile("" : "+v"(bq[kk]));  // (waited for here, the stages on their way)
  int xo[4];  // where chunk 4 kk + fg of row fr is: the swizzle only touches the chunk's low four bits
#pragma unroll
  for (int j = 0; j < 4; ++j) xo[j] = fr * RB + (((j * 4 + fg) ^ fr) << 4);
  GroupMax gx;
  gx.init(q < Q ? gm + (size_t)q * GT + (size_t)rb * run_slots : nullptr, run_slots, lg);
  const unsigned* bits = bitmap ? bitmap + (size_t)min(q, Q - 1) * W : nullptr;
  int rd = 0, wr = ST - 1;
  for (int t = 0; t < nst; ++t) {
    // this wave's pieces of stage t are in (ST - 2 newer stages); after the barrier everyone's, and stage t - 1 has been read
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(P * (ST - 2)) : "memory");
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    const char* src = sX + rd * (STAGE + SL);
#pragma unroll
    for (int u = 0; u < TR; ++u) {
      f32x4_t acc = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kk = 0; kk < NK; ++kk)
        acc = mfma16(*(const bf16x8_t*)(src + u * 16 * RB + xo[kk & 3] + (kk >> 2) * 256), bq[kk], acc);
      if (u == TR - 1) issue(t + ST - 1, wr);  // (behind the LDS reads, which its writes would hold up, and beside the maxima)
      int sl[4] = {0, 0, 0, 0};
      if (slots) {
        const u32x4_t v = *(const u32x4_t*)(src + STAGE + w * 256 + u * 64 + fg * 16);
#pragma unroll
        for (int i = 0; i < 4; ++i) sl[i] = (int)v[i];
      }
      gx.tile(acc, t * TR + u, beg + (t * TR + u) * 16 + fg * 4, end, thr, sl, bits, W, fg);
    }
    rd = rd + 1 == ST ? 0 : rd + 1;
    wr = wr + 1 == ST ? 0 : wr + 1;
  }
  gx.finish(nst * TR, fg);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // pieces past the end write zeros: in before the workgroup's LDS goes
}

// A wave's unsorted top-K list in LDS: cs / ci hold TL_SL slots, [0, K) the list, the rest room for what is
// being added. kth: the K-th best score (-inf while fewer than K rows are in).
constexpr int TL_SL = 64 + TK_MAX;

struct TopList {
  float* cs; int* ci;
  int K, lane;
  float kth;

  __device__ __forceinline__ void init(float* s, int* i, int k) {
    cs = s; ci = i; K = k; lane = threadIdx.x & 63; kth = -INFINITY;
    if (lane < K) { cs[lane] = -INFINITY; ci[lane] = -1; }
    wave_sync_lds();
  }
  // one candidate per lane (id < 0: none); ties at the threshold go to the smaller row id
  __device__ __forceinline__ void add(float v, int id) {
    const bool cand = id >= 0 && v >= kth;
    const unsigned long long m = __ballot(cand);
    if (!m) return;
    const int n = __popcll(m);
    if (n + K > 64) {  // only the best K of the new ones can stay
      td_cut(cand ? v : -INFINITY, cand ? id : -1, K, lane, cs + 64, ci + 64);
      const float* s = lane < K ? cs + lane : cs + 64 + (lane - K);
      const int* i = lane < K ? ci + lane : ci + 64 + (lane - K);
      v = lane < 2 * K ? *s : -INFINITY;
      id = lane < 2 * K ? *i : -1;
    } else {
      const int pos = K + __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
      wave_sync_lds();
      if (cand) { cs[pos] = v; ci[pos] = id; }
      wave_sync_lds();
      v = lane < K + n ? cs[lane] : -INFINITY;
      id = lane < K + n ? ci[lane] : -1;
    }
    kth = td_cut(v, id, K, lane, cs, ci);
  }
};

// Wave 0 (every wave's list is in): the lists of waves 1 .. n - 1 into its own.
__device__ __forceinline__ void top_join(TopList& top, float (*cs)[TL_SL], int (*ci)[TL_SL], int n) {
  const int rest = (n - 1) * top.K;
  for (int e0 = 0; e0 < rest; e0 += 64) {
    const int e = e0 + top.lane, w = 1 + min(e, max(rest - 1, 0)) / top.K;
    top.add(cs[w][e % top.K], e < rest ? ci[w][e % top.K] : -1);
  }
  wave_sync_lds();
}

// Where a search's result goes, [Q, K] each: scores, and the rows (oi) or, with the table of external ids [N] (og, oi null),
// the rows' ids. The last kernel of a search looks them up itself: as a launch of its own that was 2 us on the device and 10
// on the host, for K numbers a query.
struct TopOut {
  float* os;
  int* oi;
  const long* ids;
  long* og;
  int N;
  __device__ __forceinline__ void put(size_t o, float v, int row) const {
    os[o] = v;
    if (og) og[o] = row >= 0 && row < N ? ids[row] : -1;  // (a bad row index never reads outside the table)
    else oi[o] = row;
  }
};

// A wave's list, best first (ties: smaller row id), empty places behind: each row's place by counting the better ones.
__device__ __forceinline__ void top_order(const TopList& top, const TopOut& out, int q) {
  const int K = top.K, lane = top.lane;
  const size_t o = (size_t)q * K;
  const float v = lane < K ? top.cs[lane] : -INFINITY;
  const int id = lane < K ? top.ci[lane] : -1;
  int rank = 0;
  for (int j = 0; j < K; ++j) {
    const float vj = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(v), j));
    const int ij = __builtin_amdgcn_readlane(id, j);
    rank += ij >= 0 && (better(vj, ij, v, id) || (vj == v && ij == id && j < lane));  // (a row named twice)
  }
  const int real = __popcll(__ballot(id >= 0));
  if (id >= 0) out.put(o + rank, v, id);
  if (lane >= real && lane < K) out.put(o + lane, -INFINITY, -1);
}

// The lists [P, Q, K] of query q put together by a workgroup of n waves, each with a list in cs / ci: each wave cuts its share
// to K, wave 0 joins what is left and orders it. Ends with the query's result written.
template <typename S, typename I>
__device__ __forceinline__ void top_collect(float (*cs)[TL_SL], int (*ci)[TL_SL], int n, int K, int P, int Q, int q,
                                            const TopOut& out, S score, I row) {
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6, nt = n * 64, all = P * K;
  TopList top;
  top.init(cs[wid], ci[wid], K);
  for (int j0 = wid * 64; j0 < all; j0 += nt * 4) {
    float v[4];
    int id[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {  // issued together: the lists come from all over the chip's caches
      const int j = j0 + lane + nt * u, jc = min(j, all - 1);
      const size_t o = ((size_t)(jc / K) * Q + q) * K + jc % K;
      v[u] = score(o);
      id[u] = row(o);
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) top.add(v[u], j0 + lane + nt * u < all ? id[u] : -1);
  }
  __syncthreads();
  if (wid) return;
  top_join(top, cs, ci, n);
  top_order(top, out, q);
}

// Per-query row ranges: ranges [R, 2] (start, end) and range_off [Q + 1], or (lists [Q, probes] != null) rows
// ranges[l] .. ranges[l + 1] of each list l that the query names (l < 0: none). rows_per_split rows of the query's concatenated ranges per
// workgroup (grid = (splits, Q)). out_s / out_i [splits, Q, K], unsorted lists (topk_merge_kernel orders them, or with counters cnt [Q], zero
// between launches, the query's last workgroup: out).
//
// A half-wave owns a row (16 B per lane and load, NCH loads), four rows of it are on their way together; 64 rows
// are scored per step and handed to wave 0, which keeps the list while the others score the next 64 (two buffers,
// one barrier a step). Bound by the latency of a step for few rows, by HBM for many: the caller splits a query's
// rows over as many workgroups as fill the chip (388 rows of 8 documents: one workgroup took 105 us, with one load
// in flight and a shuffle merge of K rounds per 64 rows; 7 workgroups take 15 us. 24 queries over 8 lists of about
// 780 rows x 768: 162 -> 41 us).
//
// Few rows are a chain of latencies, so a step of up to 32 rows is one round of loads, the query and the doc slots arrive with the
// rows and not before or behind them, and (cnt) the lists meet in the query's last workgroup instead of a launch of their own,
// which costs the host 2 us. us on the device and in all: 384 rows of 768 12.6 and 17.9 -> 10.5 and 15.8, 10 queries of 192
// 13.9 and 17.2 -> 12.1 and 15.7, 20 rows 8.2 and 17.1 -> 5.3 and 16.0.
//
// A filter's ranges come from the host. Up to TR_TABLE numbers of them ride in the launch's arguments (range_off, then the
// ranges; a workgroup takes them to LDS in one step); as two copies they took 3.3 us each on the device and about 15 on the
// host. With the ids looked up by the last kernel and one pair of events a search, one query over 8 of 100000 x 768 rows'
// documents takes 33 us, 94 before. Lists, and ranges that are on the device, have a kernel without the table (scores and merge,
// us with it -> without: 24 queries over 8 of 512 lists of 400000 x 768 rows 68.7 -> 58.2, 8 over 16 of 256 of 200000 x 384 53 -> 45,
// 8 ranges of 50 rows a query for 64 queries 21.9 -> 19.7).
constexpr int TR_TABLE = 512;  // 2 of the 4 KB that a launch's arguments may have
struct RangeTable { int v[TR_TABLE]; };
struct NoTable { int v[1]; };

template <int NCH, typename Table>
__global__ void __launch_bounds__(256)
topk_ranges_kernel(const bf16_t* __restrict__ X, int d, const int* __restrict__ slots,
                   const bf16_t* __restrict__ Qv, int Q, const int* __restrict__ ranges,
                   const int* __restrict__ range_off, const int* __restrict__ lists, int probes,
                   const unsigned* __restrict__ bitmap, int W, float thr,
                   int K, int rows_per_split, float* __restrict__ out_s, int* __restrict__ out_i, const TopOut out,
                   int* __restrict__ cnt, int n_table, const Table table) {
  constexpr bool TABLE = std::is_same_v<Table, RangeTable>;
  extern __shared__ __attribute__((aligned(16))) char joined[];  // (cnt: a list of each wave, and a flag)
  __shared__ int st[TABLE ? TR_TABLE : 1];
  __shared__ float sc[2][64];
  __shared__ int sr[2][64];
  __shared__ float cs[TL_SL];
  __shared__ int ci[TL_SL];
  const int split = blockIdx.x, q = blockIdx.y;
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int half = lane >> 5, l32 = lane & 31;
  TopList top;
  top.init(cs, ci, K);  // (every wave writes the same empty list; wave 0 keeps it)
  if constexpr (TABLE) {
    for (int i = tid; i < n_table; i += 256) st[i] = table.v[i];
    __syncthreads();
    lists = nullptr;
  }
  const auto range = [&](int i) { return TABLE ? st[Q + 1 + i] : ranges[i]; };
  const int nch = d / 8;  // 16-B chunks of a row; this lane has chunks l32 + 32 i
  const auto half_f = [](const u32x4_t& u, int e) { return bf2f((bf16_t)((e & 1) ? (u[e >> 1] >> 16) : (u[e >> 1] & 0xffff))); };
  u32x4_t qu[NCH];  // (as it is: converted here, the first rows would wait for it)
#pragma unroll
  for (int i = 0; i < NCH; ++i) qu[i] = *(const u32x4_t*)(Qv + (size_t)q * d + min(l32 + 32 * i, nch - 1) * 8);
  const int rb = TABLE ? st[q] : lists ? q * probes : range_off[q], re = TABLE ? st[q + 1] : lists ? rb + probes : range_off[q + 1];
  DA_ASSERT(rb >= 0 && re >= rb);
  const int pbeg = split * rows_per_split, pend = pbeg + rows_per_split;
  __syncthreads();
  // walk the concatenated ranges; position p counts rows across this query's ranges
  int pos = 0, buf = 0, r0 = rb;
  if (pbeg > 0 && re - rb > 16) {
    // to the range that this split begins in: 64 lengths a step and their sums (one range after another, each a load of its
    // own that the next waits for, the last of 250 splits took 0.3 us for each of 2000 ranges)
    for (; r0 < re; r0 += 64) {
      const int r = min(r0 + lane, re - 1), l = lists ? lists[r] : 0;
      const bool in = r0 + lane < re && l >= 0;
      const int at = !in ? 0 : lists ? l : 2 * r;
      const int len = range(at + 1) - range(at);
      int sum = in ? len : 0;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const int below = __shfl_up(sum, o, 64);
        sum += lane >= o ? below : 0;
      }
      const unsigned long long past = __ballot(pos + sum > pbeg);
      if (past) {
        const int first = __builtin_ctzll(past);
        pos += first ? __shfl(sum, first - 1, 64) : 0;
        r0 += first;
        break;
      }
      pos += __shfl(sum, 63, 64);
    }
    r0 = __builtin_amdgcn_readfirstlane(r0);
    pos = __builtin_amdgcn_readfirstlane(pos);
  }
  for (int r = r0; r < re; ++r) {
    const int l = lists ? lists[r] : 0;
    if (l < 0) continue;
    const int s0 = range(lists ? l : 2 * r), s1 = range(lists ? l + 1 : 2 * r + 1);
    const int len = s1 - s0;
    const int lo = max(pbeg, pos), hi = min(pend, pos + len);
    for (int p0 = lo; p0 < hi; p0 += 64) {
      // 64 rows per step: 8 half-waves x 8 rows, 4 at a time (up to 32 rows: 4 each, and the others none)
      const int each = hi - p0 > 32 ? 8 : 4;
      for (int j0 = 0; j0 < each; j0 += 4) {
        const int rl = (wid * 2 + half) * each + j0;
        u32x4_t u[4][NCH];
#pragma unroll
        for (int j = 0; j < 4; ++j) {  // rows and chunks past the end: the last one's
          const bf16_t* xr = X + (size_t)(s0 + (min(p0 + rl + j, hi - 1) - pos)) * d;
#pragma unroll
          for (int i = 0; i < NCH; ++i) u[j][i] = *(const u32x4_t*)(xr + min(l32 + 32 * i, nch - 1) * 8);
        }
        // lane j of a half-wave hands in row j
        const int p = p0 + rl + (l32 & 3), row = s0 + (min(p, hi - 1) - pos);
        const int sl = slots ? slots[row] : 0;
        float dot[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < NCH; ++i) {
          const bool in = l32 + 32 * i < nch;
          float qv[8];
#pragma unroll
          for (int e = 0; e < 8; ++e) qv[e] = half_f(qu[i], e);
#pragma unroll
          for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int e = 0; e < 8; ++e) {
              const float t = dot[j] + qv[e] * half_f(u[j][i], e);
              dot[j] = in ? t : dot[j];
            }
        }
#pragma unroll
        for (int o = 16; o > 0; o >>= 1)
#pragma unroll
          for (int j = 0; j < 4; ++j) dot[j] += __shfl_xor(dot[j], o, 64);
        const float s = (l32 == 0 ? dot[0] : l32 == 1 ? dot[1] : l32 == 2 ? dot[2] : dot[3]);
        if (l32 < 4) {
          bool ok = p < hi && s >= thr && s != -INFINITY && sl >= 0;
          if (ok && bitmap) ok = (sl >> 5) < W && ((bitmap[(size_t)q * W + (sl >> 5)] >> (sl & 31)) & 1u);
          sc[buf][rl + l32] = s;
          sr[buf][rl + l32] = ok ? row : -1;
        }
      }
      if (each == 4 && tid < 32) sr[buf][32 + tid] = -1;
      __syncthreads();  // this step's scores are in, and the list has taken the last step's
      if (wid == 0) top.add(sc[buf][lane], sr[buf][lane]);
      buf ^= 1;
    }
    pos += len;
    if (pos >= pend) break;
  }
  const size_t o = ((size_t)split * Q + q) * K + lane;
  if (!cnt) {
    if (wid == 0) {
      wave_sync_lds();
      if (lane < K) {
        out_s[o] = cs[lane];
        out_i[o] = ci[lane];
      }
    }
    return;
  }
  // ---- the query's last workgroup puts the lists together ----
  if (gridDim.x == 1) {
    if (wid == 0) {
      wave_sync_lds();
      top_order(top, out, q);
    }
    return;
  }
  int* last = (int*)joined;
  float (*js)[TL_SL] = (float (*)[TL_SL])(joined + 16);
  int (*ji)[TL_SL] = (int (*)[TL_SL])(joined + 16 + 4 * TL_SL * sizeof(float));
  if (wid == 0) {
    wave_sync_lds();
    if (lane < K) {  // past the XCDs' L2s, to where all of them see it
      __hip_atomic_store(out_s + o, cs[lane], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_store(out_i + o, ci[lane], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (lane == 0) {
      const bool all = __hip_atomic_fetch_add(cnt + q, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (int)gridDim.x - 1;
      if (all) __hip_atomic_store(cnt + q, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // for the next launch
      *last = all;
    }
  }
  __syncthreads();
  if (!*last) return;
  const auto ld = [](const auto* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); };
  top_collect(js, ji, 4, K, (int)gridDim.x, Q, q, out, [&](size_t at) { return ld(out_s + at); }, [&](size_t at) { return ld(out_i + at); });
}

// cand [P, Q, K] -> out [Q, K] sorted desc (ties: smaller row id). One workgroup per query, a wave per 64 candidates
// up to 16 (TM_WAVES): each wave cuts its share to K, wave 0 joins the lists and orders them by counting the better
// ones of each. Bound by the chain of cuts (about 1 us each), hence many waves: K rounds of a workgroup-wide argmax
// with two barriers each took 18 us for 256 parts of K = 5, cuts by 4 waves 23 us, by 16 16.5 us.
constexpr int TM_WAVES = 16;

__global__ void __launch_bounds__(64 * TM_WAVES)
topk_merge_kernel(const float* __restrict__ cand_s, const int* __restrict__ cand_i, int P, int Q, int K,
                  const TopOut out) {
  __shared__ float cs[TM_WAVES][TL_SL];
  __shared__ int ci[TM_WAVES][TL_SL];
  top_collect(cs, ci, (int)blockDim.x / 64, K, P, Q, blockIdx.x, out, [&](size_t o) { return cand_s[o]; },
              [&](size_t o) { return cand_i[o]; });
}

// The second half of a scan (see there): per query the K best of its GT groups, their rows scored again (16 rows a wave and
// step, the query in all of the MFMA's columns), the K best of those in order. Group g is tiles (g % run_slots) << lg .. of
// run g / run_slots, run_rows rows each.
// Bound by latency. A cut of a list of 64 takes about 1 us, and 80000 values in any order improve on one many times (lists
// kept by every wave, as topk_merge_kernel does: 100 us for 80000 groups, K = 5; 49 for 8000, K = 19), so a bound comes first:
// the K-th best of the threads' own best values, to its upper 20 bits. What reaches it (little more than K values) is
// collected and cut once, and the same again with the rows that reach the K-th best group. Where more than 256 reach it
// (equal scores), the K-th best is found to its last bit by counting, a pass over the groups for each bit that is open, and its first
// equals are taken in order. us, lists of every scan / lists of the pick's waves / this: 20000 equal rows x 384, one query, K = 20
// 155 / 811 / 65, 600000 of 20 kinds, K = 5 181 / 488 / 163, 600000 equal, 64 queries, K = 5 187 / 792 / 187; rows that overflow are done over by the waves' lists.
// A thread keeps its best four of groups and the largest behind it, so that nearly always one four is read again and not the
// whole line (5 us of 34 at 40000 groups). Rows of more tiles than waves come through LDS in whole lines: as MFMA operands they are
// requests of 64 B, 512 a tile, of which a CU has 256 on their way (24 tiles 13.6 -> 8.3 us; of up to 8 tiles the ring is 1 us
// slower). Whole searches, us: 102624 x 768, 10 queries, K = 20 50.8 -> 45.1, 110468 x 1024, 42, K = 14 64.3 -> 60.0, 52331 x 1024,
// one, K = 14 41.3 -> 36.3, 10000 x 768, 24, K = 5 17.1 -> 15.2, 958291 x 1024, 18, K = 12 340 -> 335; 20000 x 768, 128, K = 5 26.9 -> 27.3.
// Groups that are none (few rows reach the least similarity) are no tiles: 100000 x 1024, 17 queries, K = 32, rows of 0.95 and more 47.2 us
// with the ring's steps left out for them, 60.0 without.
constexpr int TP_WAVES = 8, TP_CAP = 1024, TP_FOLD = 256, TP_RING = 3;

// The largest bound, to its upper 20 bits, that at least `need` of the 8 keys of each lane reach (0: there are not as many).
__device__ __forceinline__ unsigned reached_by(const unsigned (&key)[8], int need) {
  unsigned T = 0;
  for (int bt = 31; bt >= 12; --bt) {
    const unsigned t = T | (1u << bt);
    int c = 0;
#pragma unroll
    for (int u = 0; u < 8; ++u) c += __popcll(__ballot(key[u] >= t));
    if (c >= need) T = t;
    if (c == need) break;
  }
  return T;
}

template <int NG>
__global__ void __launch_bounds__(64 * TP_WAVES, 2)
topk_pick_kernel(const float* __restrict__ gm, int GT, int run_slots, int run_rows, int lg, const bf16_t* __restrict__ X, int N,
                 const int* __restrict__ slots, const bf16_t* __restrict__ Qv, const unsigned* __restrict__ bitmap, int W,
                 float thr, int K, const TopOut out) {
  constexpr int d = NG * 128, NK = d / 32, nt = 64 * TP_WAVES;
  static_assert(TP_WAVES == 8, "a key of each thread: 8 per lane of a wave");
  __shared__ float cs[TP_WAVES][TL_SL], cand_s[TP_CAP];
  __shared__ int ci[TP_WAVES][TL_SL], cand_i[TP_CAP];
  __shared__ int groups[TK_MAX], n_groups, count, reach[32], equal[TP_WAVES];
  __shared__ float bound;
  __shared__ unsigned keys[nt], bkey;
  __shared__ __attribute__((aligned(16))) bf16_t sq[d];
  extern __shared__ __attribute__((aligned(16))) char tp_tiles[];  // (groups of more than TP_WAVES tiles) [TP_WAVES][TP_RING] pieces of 16 rows x 128 columns
  const int q = blockIdx.x, tid = threadIdx.x, lane = tid & 63, fr = lane & 15, fg = lane >> 4;
  const int wid = __builtin_amdgcn_readfirstlane(tid >> 6);
  for (int i = tid; i < d / 8; i += nt) *(u32x4_t*)(sq + i * 8) = *(const u32x4_t*)(Qv + (size_t)q * d + i * 8);
  const f32x4_t* line = (const f32x4_t*)(gm + (size_t)q * GT);
  TopList top;
  top.init(cs[wid], ci[wid], K);
  // the best rows or groups so far collected: through wave 0's list, best K of them; overflowed: every wave's own
  auto collect = [&](float v, int id, bool in) __attribute__((always_inline)) {
    if (!in) return;
    const int at = atomicAdd(&count, 1);
    if (at < TP_CAP) { cand_s[at] = v; cand_i[at] = id; }
  };
  auto fold = [&](int n) __attribute__((always_inline)) {  // wave 0
    for (int j = 0; j < n; j += 64) {
      const int e = min(j + lane, n - 1);
      top.add(cand_s[e], j + lane < n ? cand_i[e] : -1);
    }
    wave_sync_lds();
  };

  // ---- groups ----
  const int nv = GT / 4;
  float best = -INFINITY, next = -INFINITY;  // of this thread's fours, by their largest: the best, and the one behind it
  int at4 = 0;
  auto see = [&](const f32x4_t& v, int j) __attribute__((always_inline)) {  // (a value counts for one thread only)
    const float m = j < nv ? fmaxf(fmaxf(v[0], v[1]), fmaxf(v[2], v[3])) : -INFINITY;
    next = fmaxf(next, fminf(m, best));
    at4 = m > best ? j : at4;
    best = fmaxf(best, m);
  };
  auto look = [&](auto ahead) __attribute__((always_inline)) {
    constexpr int U = decltype(ahead)::value;
    for (int j0 = tid; j0 < nv; j0 += nt * U) {
      f32x4_t v[U];
#pragma unroll
      for (int u = 0; u < U; ++u) v[u] = line[min(j0 + nt * u, nv - 1)];
#pragma unroll
      for (int u = 0; u < U; ++u) see(v[u], j0 + nt * u);
    }
  };
  if (nv <= 4 * nt) look(std::integral_constant<int, 4>{});
  else look(std::integral_constant<int, 8>{});
  keys[tid] = td_key(best, best > -INFINITY ? 0 : -1);
  if (tid == 0) count = 0;
  if (tid < 32) reach[tid] = 0;
  __syncthreads();
  if (wid == 0) {
    unsigned key[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) key[u] = keys[u * 64 + lane];
    const unsigned by = reached_by(key, K);
    const float b = td_unkey(by);
    if (lane == 0) { bound = b != b ? -INFINITY : b; bkey = b != b ? 0 : by; }
  }
  __syncthreads();
  const float T = bound;
  if (best >= T && best > -INFINITY) {
    const bool more = next >= T && next > -INFINITY;  // (then all of them: rarely more than the one)
    for (int j0 = more ? tid : at4; j0 < nv; j0 += more ? nt : nv) {
      const f32x4_t v = line[j0];
#pragma unroll
      for (int e = 0; e < 4; ++e) collect(v[e], 4 * j0 + e, v[e] >= T && v[e] > -INFINITY);
    }
  }
  __syncthreads();
  int found = count;
  __syncthreads();  // (count is written below)
  if (found > TP_FOLD) {
    // the K-th best to its last bit (from bkey to the best), then what is better than it, and as many of its equals as are
    // missing, first rows first
    unsigned Tk = 0, kmax = 0;
    for (int u = 0; u < 8; ++u) kmax = max(kmax, keys[u * 64 + lane]);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) kmax = max(kmax, (unsigned)__shfl_xor((int)kmax, o, 64));
    for (int bt = 31; bt >= 0; --bt) {
      const unsigned t = Tk | (1u << bt);
      if (t <= bkey) Tk = t;
      if (t <= bkey || t > kmax) continue;
      int c = 0;  // (whole in lane 0, which takes part in every step of its wave)
      for (int j0 = tid; j0 < nv; j0 += nt) {
        const f32x4_t v = line[j0];
#pragma unroll
        for (int e = 0; e < 4; ++e) c += __popcll(__ballot(v[e] > -INFINITY && td_key(v[e], 0) >= t));
      }
      if (lane == 0) atomicAdd(&reach[bt], c);
      __syncthreads();
      if (reach[bt] >= K) Tk = t;
    }
    if (tid == 0) count = 0;
    __syncthreads();
    for (int j0 = tid; j0 < nv; j0 += nt) {
      const f32x4_t v = line[j0];
#pragma unroll
      for (int e = 0; e < 4; ++e) collect(v[e], 4 * j0 + e, v[e] > -INFINITY && td_key(v[e], 0) > Tk);
    }
    __syncthreads();
    found = count;  // (less than K)
    for (int j0 = 0; j0 < nv && found < K; j0 += nt) {
      const f32x4_t v = line[min(j0 + tid, nv - 1)];
      unsigned m = 0;
#pragma unroll
      for (int e = 0; e < 4; ++e) m |= (unsigned)(j0 + tid < nv && v[e] > -INFINITY && td_key(v[e], 0) == Tk) << e;
      int at = __popc(m);  // equals up to this lane's last
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const int x = __shfl_up(at, o, 64);
        if (lane >= o) at += x;
      }
      if (lane == 63) equal[wid] = at;
      __syncthreads();
      int all = found;
      at += found - __popc(m);
      for (int w = 0; w < TP_WAVES; ++w) {
        if (w < wid) at += equal[w];
        all += equal[w];
      }
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if ((m >> e) & 1) {
          if (at < K) { cand_s[at] = v[e]; cand_i[at] = 4 * (j0 + tid) + e; }
          ++at;
        }
      found = min(all, K);
      __syncthreads();  // (equal is written again)
    }
  }
  if (wid == 0) {
    fold(found);
    if (lg < 0) {  // these are the rows
      if (lane < K && ci[0][lane] >= 0) ci[0][lane] = ci[0][lane] / run_slots * run_rows + ci[0][lane] % run_slots;
      wave_sync_lds();
      top_order(top, out, q);
      return;
    }
    const unsigned long long real = __ballot(lane < K && ci[0][min(lane, K - 1)] >= 0);  // (fewer than K where few rows reach thr)
    if ((real >> lane) & 1) groups[__popcll(real & ((1ull << lane) - 1))] = ci[0][lane];
    if (lane == 0) n_groups = __popcll(real);
    float low = lane < K && ci[0][lane] >= 0 ? cs[0][lane] : lane < K ? -INFINITY : INFINITY;  // the K-th best group
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) low = fminf(low, __shfl_xor(low, o, 64));
    if (lane == 0) { bound = low; count = 0; }
  }
  if (lg < 0) return;
  __syncthreads();

  // ---- their rows ----
  const float R = bound;
  top.init(cs[wid], ci[wid], K);
  char* mine = tp_tiles + wid * TP_RING * 4096;
  unsigned off[4];  // 1 KiB instruction i: rows 4 i .. 4 i + 3, 256 B of each: chunk c of row r at c ^ r
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = 4 * i + (lane >> 4);
    off[i] = (unsigned)(r * d * 2 + (((lane & 15) ^ r) << 4));
  }
  const int all = n_groups << lg;
  // the wave's i-th tile: its first row, and the end of the run (0: none)
  auto tile = [&](int i, int& row0, int& end) __attribute__((always_inline)) {
    const int it = wid + i * TP_WAVES, g = it < all ? groups[it >> lg] : -1;
    const long first = (long)(g / run_slots) * run_rows;
    row0 = g < 0 ? 0 : (int)first + ((((g % run_slots) << lg) + (it & ((1 << lg) - 1))) * 16);
    end = g < 0 ? 0 : (int)min((long)N, first + run_rows);
    row0 = __builtin_amdgcn_readfirstlane(row0);
    end = __builtin_amdgcn_readfirstlane(end);
  };
  auto issue = [&](int row0, int end, int g, int slot) __attribute__((always_inline)) {  // 128 columns of a tile (rows past the end: zeros)
    const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc((void*)(X + (size_t)row0 * d), (short)0,
                                                                        max(0, min(end - row0, 16)) * d * 2, 0x00020000);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (vs_lds_t)(mine + slot * 4096 + i * 1024), 16, off[i], g * 256, 0, 0);
  };
  const int tiles = (all - wid + TP_WAVES - 1) / TP_WAVES;
  const bool one = all <= TP_WAVES;
  for (int again = 0; again < 2; ++again) {
    int row0, end, row1 = 0, end1 = 0, slot = 0;
    tile(0, row0, end);
    if (!one && tiles > 0)
#pragma unroll 1
      for (int g = 0; g < TP_RING; ++g) issue(row0, end, g, g);
    for (int i = 0; i < tiles; ++i) {
      tile(i + 1, row1, end1);  // (past the last: no rows)
      // lane (fr, fg), fr < 4: row 4 fg + fr of the tile
      const int row = row0 + 4 * fg + (fr & 3);
      const int sl = slots && row < end ? slots[row] : 0;
      f32x4_t acc = f32x4_t{0.f, 0.f, 0.f, 0.f};
      if (one) {
        const bf16_t* xr = X + (size_t)max(0, min(row0 + fr, end - 1)) * d + fg * 8;
        bf16x8_t a[NK];
#pragma unroll
        for (int kk = 0; kk < NK; ++kk) a[kk] = *(const bf16x8_t*)(xr + kk * 32);
#pragma unroll
        for (int kk = 0; kk < NK; ++kk) acc = mfma16(a[kk], *(const bf16x8_t*)(sq + kk * 32 + fg * 8), acc);
      } else {
#pragma unroll 1
        for (int g = 0; g < NG; ++g) {
          asm volatile("s_waitcnt vmcnt(%0)" ::"n"(4 * (TP_RING - 1)) : "memory");  // this group is in, newer ones on their way
          __builtin_amdgcn_sched_barrier(0);
          bf16x8_t a[4];
#pragma unroll
          for (int j = 0; j < 4; ++j) a[j] = *(const bf16x8_t*)(mine + slot * 4096 + fr * 256 + (((4 * j + fg) ^ fr) << 4));
          asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
          __builtin_amdgcn_sched_barrier(0);
          const bool on = g + TP_RING >= NG;  // the next tile's
          issue(on ? row1 : row0, on ? end1 : end, on ? g + TP_RING - NG : g + TP_RING, slot);
          slot = slot + 1 == TP_RING ? 0 : slot + 1;
#pragma unroll
          for (int j = 0; j < 4; ++j) acc = mfma16(a[j], *(const bf16x8_t*)(sq + (4 * g + j) * 32 + fg * 8), acc);
        }
      }
      const float s = fr == 0 ? acc[0] : fr == 1 ? acc[1] : fr == 2 ? acc[2] : acc[3];
      bool ok = fr < 4 && row < end && sl >= 0 && s >= thr && s > -INFINITY && s >= R;
      if (ok && bitmap) ok = (sl >> 5) < W && ((bitmap[(size_t)q * W + (sl >> 5)] >> (sl & 31)) & 1u);
      if (again) top.add(s, ok ? row : -1);
      else collect(s, row, ok);
      row0 = row1;
      end = end1;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (pieces past the last tile write zeros)
    __syncthreads();
    if (again || count <= TP_CAP) {  // (no more writes to count)
      if (wid) return;
      if (again) top_join(top, cs, ci, TP_WAVES);
      else fold(count);
      top_order(top, out, q);
      return;
    }
  }
}

// out[i] = ids[rows[i]], -1 where rows[i] names no row of [0, N) (a bad row index must never read outside the table).
// One launch where nine elementwise ones of 2 to 5 us each did it.
__global__ void __launch_bounds__(256)
gather_ids_kernel(const int* __restrict__ rows, int n, const long* __restrict__ ids, int N, long* __restrict__ out) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const int r = rows[i];
  out[i] = r >= 0 && r < N ? ids[r] : -1;
}

// k-means accumulation: sums[assign[i]] += X[i] (fp32), counts[assign[i]] += 1
__global__ void kmeans_accum_kernel(const bf16_t* __restrict__ X, int N, int d, const int* __restrict__ assign,
                                    float* __restrict__ sums, float* __restrict__ counts) {
  const int row = blockIdx.x;
  if (row >= N) return;
  const int c = assign[row];
  if (c < 0) return;
  for (int j = threadIdx.x; j < d; j += blockDim.x) atomicAdd(&sums[(size_t)c * d + j], bf2f(X[(size_t)row * d + j]));
  if (threadIdx.x == 0) atomicAdd(&counts[c], 1.f);
}

// (out: rows, int; with ids [N]: their ids, long)
static TopOut top_out(void* out_s, void* out, const void* ids, int N) {
  return ids ? TopOut{(float*)out_s, nullptr, (const long*)ids, (long*)out, N} : TopOut{(float*)out_s, (int*)out, nullptr, nullptr, 0};
}

static int topk_merge(const void* cs, const void* ci, int P, int Q, int K, const TopOut& out, hipStream_t s) {
  const long waves = min((long)TM_WAVES, max(1L, ((long)P * K + 63) / 64));
  topk_merge_kernel<<<Q, 64 * (int)waves, 0, s>>>((const float*)cs, (const int*)ci, P, Q, K, out);
  DA_LAUNCH_CHECK();
}

DA_EXPORT size_t da_topk_dense_ws(int N, int Q, int K, int rows_per_block) {
  const int nblk = (N + rows_per_block - 1) / rows_per_block;
  return (size_t)nblk * Q * K * 8;
}

DA_EXPORT int da_topk_dense(const void* X, int N, int d, const void* slots, const void* Qv, int Q, const void* bitmap,
                            int W, float thr, int K, int rows_per_block, void* ws, void* out_s, void* out,
                            const void* ids, int n_ids, void* stream) {
  if (d % 32 || K < 1 || K > TK_MAX || rows_per_block % 64 || rows_per_block <= 0) return (int)hipErrorInvalidValue;
  if (Q == 0) return 0;
  hipStream_t s = (hipStream_t)stream;
  const int nblk = N > 0 ? (N + rows_per_block - 1) / rows_per_block : 1;
  float* cs = (float*)ws;
  int* ci = (int*)(cs + (size_t)nblk * Q * K);
  const size_t lds = 16 * (d * 2 + 16) + 16 * 65 * 4 + 16 * TK_MAX * 8;
  if (lds > 160 * 1024) return (int)hipErrorInvalidValue;
  dim3 grid(nblk, (Q + 15) / 16);
  topk_dense_kernel<<<grid, 256, lds, s>>>((const bf16_t*)X, N, d, (const int*)slots, (const bf16_t*)Qv, Q,
                                           (const unsigned*)bitmap, W, thr, K, rows_per_block, cs, ci);
  int err = (int)hipGetLastError();
  if (err) return err;
  return topk_merge(cs, ci, nblk, Q, K, top_out(out_s, out, ids, n_ids), s);
}

// The streaming scan (d = 384, 768 or 1024). hipErrorInvalidValue for shapes it does not take (the caller then uses
// da_topk_dense). Its runs of rows, and their groups in ws: Q lines of `groups` floats.
struct ScanPlan {
  int runs, run_rows, run_slots, lg;  // run_slots: a run's groups, padded to 4; lg < 0: its rows, padded to 16
  long groups() const { return (long)runs * run_slots; }
};

// A run is a wave's (up to 16 queries; rows_per_wave at least) or a workgroup's (17 and more), 16 to 524288 rows (32-bit
// offsets), and as many as one round of resident workgroups needs: a second round starts its pipelines anew, us with 1024
// waves / 4096: 100000 x 1024, 16 queries, 48.7 / 56.3; 411812 x 768 113.6 / 121.0; 1250000 x 1024 417 / 419.
// A group is a tile up to 65536 of them, and 2, 4, .. tiles from there on; with the padding of the runs' ends the pick reads 290 KB
// a query at most (1.05 and 2.1 M rows 279, scores of 57925 rows with K = 32 290).
// Up to 10000 + 1500 K rows each row's score is left, and nothing is scored again: more to write and to read for fewer steps of
// the pick, a wave's tile of a group each. us, groups / scores: 464 x 1024, K = 24, 2 queries 36 / 14; 512 x 768, K = 8, 24
// queries 19 / 12; 10000 x 1024, 24 queries, K = 5 25 / 21, K = 20 39 / 22; 20000 x 768, 128 queries 29 / 33 and 41 / 34;
// 30000 x 1024, 20 queries 29 / 31 and 45 / 32; 60000 x 384, 128 queries 32 / 47 and 40 / 48.
static ScanPlan scan_plan(long N, int Q, int K, int rows_per_wave) {
  const long runs = Q <= 16 ? 1024 : Q <= 64 ? 512 : 256;
  ScanPlan p;
  p.run_rows = (int)min(524288L, max(Q <= 16 ? (rows_per_wave + 15L) / 16 * 16 : 16L, (N + runs * 16 - 1) / (runs * 16) * 16));
  p.runs = (int)((N + p.run_rows - 1) / p.run_rows);
  p.lg = N <= 10000 + 1500L * K ? -1 : 0;
  while (p.lg >= 0 && (N >> (4 + p.lg)) > 65536) ++p.lg;
  const int tiles = p.run_rows / 16 + 1;  // (32-row stages: one tile past the end)
  p.run_slots = p.lg < 0 ? tiles * 16 : ((tiles + (1 << p.lg) - 1 >> p.lg) + 3) & ~3;
  return p;
}

DA_EXPORT size_t da_topk_stream_ws(int N, int Q, int K, int rows_per_wave) {
  return (size_t)scan_plan(N, Q, K, rows_per_wave).groups() * Q * 4;
}

DA_EXPORT int da_topk_dense_stream(const void* X, int N, int d, const void* slots, const void* Qv, int Q,
                                   const void* bitmap, int W, float thr, int K, int rows_per_wave, void* ws, void* out_s,
                                   void* out, const void* ids, int n_ids, void* stream) {
  if ((d != 384 && d != 768 && d != 1024) || K < 1 || K > TK_MAX || N < 1 || rows_per_wave < 16)
    return (int)hipErrorInvalidValue;
  if (Q == 0) return 0;
  hipStream_t s = (hipStream_t)stream;
  const ScanPlan p = scan_plan(N, Q, K, rows_per_wave);
  const int nw = Q > 64 ? 8 : 4, nqg = (Q + 16 * nw - 1) / (16 * nw);
  const long blocks = Q <= 16 ? (p.runs + 3) / 4 : (long)(p.runs + 7) / 8 * 8 * nqg;
  if (p.groups() > 0x7fffffffL || blocks > 0x7fffffffL) return (int)hipErrorInvalidValue;
  float* gm = (float*)ws;
  const int GT = (int)p.groups();
#define TDQ(NG, NW)                                                                                                  \
  topk_dense_mq_kernel<NG, NW><<<(int)blocks, 64 * NW, 0, s>>>((const bf16_t*)X, N, (const int*)slots, (const bf16_t*)Qv, Q, \
      (const unsigned*)bitmap, W, thr, p.run_rows, nqg, gm, GT, p.run_slots, p.lg)
#define TDS(NG)                                                                                                      \
  do {                                                                                                               \
    if (Q <= 16)                                                                                                     \
      topk_dense_stream_kernel<NG><<<(int)blocks, 256, 0, s>>>((const bf16_t*)X, N, (const int*)slots,               \
          (const bf16_t*)Qv, Q, (const unsigned*)bitmap, W, thr, p.run_rows, gm, GT, p.run_slots, p.lg);             \
    else if (Q <= 64)                                                                                                \
      TDQ(NG, 4);                                                                                                    \
    else                                                                                                             \
      TDQ(NG, 8);                                                                                                    \
    const int err = (int)hipGetLastError();                                                                          \
    if (err) return err;                                                                                             \
    topk_pick_kernel<NG><<<Q, 64 * TP_WAVES, p.lg < 0 || K << p.lg <= TP_WAVES ? 0 : TP_WAVES * TP_RING * 4096, s>>>(gm, GT, p.run_slots, p.run_rows, p.lg, (const bf16_t*)X, N,      \
        (const int*)slots, (const bf16_t*)Qv, (const unsigned*)bitmap, W, thr, K, top_out(out_s, out, ids, n_ids));   \
  } while (0)
  switch (d) {
    case 384: TDS(3); break;
    case 768: TDS(6); break;
    default: TDS(8); break;
  }
#undef TDS
#undef TDQ
  DA_LAUNCH_CHECK();
}

DA_EXPORT int da_topk_ranges(const void* X, int d, const void* slots, const void* Qv, int Q, const void* ranges,
                             const void* range_off, const void* lists, int probes, const void* bitmap, int W,
                             float thr, int K, int splits, int rows_per_split, void* ws, void* out_s, void* out,
                             const void* ids, int n_ids, const void* host_table, int n_table, void* cnt, void* stream) {
  if (d % 8 || d < 8 || d > 4096 || K < 1 || K > TK_MAX || splits < 1 || rows_per_split < 1 ||
      (!range_off && !n_table && (!lists || probes < 0)) || n_table < 0 || n_table > TR_TABLE ||
      (n_table && (lists || !host_table || n_table < Q + 1)))
    return (int)hipErrorInvalidValue;
  if (Q == 0) return 0;
  hipStream_t s = (hipStream_t)stream;
  float* cs = (float*)ws;
  int* ci = (int*)(cs + (size_t)splits * Q * K);
  dim3 grid(splits, Q);
  const TopOut result = top_out(out_s, out, ids, n_ids);
  const size_t lds = cnt && splits > 1 ? 16 + 4 * TL_SL * 8 : 0;
  auto launch = [&](const auto& table) {
    using Table = std::decay_t<decltype(table)>;
#define TRG(NCH)                                                                                                    \
  topk_ranges_kernel<NCH, Table><<<grid, 256, lds, s>>>((const bf16_t*)X, d, (const int*)slots, (const bf16_t*)Qv, Q,  \
                                                        (const int*)ranges, (const int*)range_off, (const int*)lists, \
                                                        probes, (const unsigned*)bitmap, W, thr, K, rows_per_split, cs, ci, \
                                                        result, (int*)cnt, n_table, table)
    if (d <= 256) TRG(1);
    else if (d <= 512) TRG(2);
    else if (d <= 768) TRG(3);
    else if (d <= 1024) TRG(4);
    else if (d <= 2048) TRG(8);
    else TRG(16);
#undef TRG
  };
  if (n_table) {
    RangeTable table;
    memcpy(table.v, host_table, (size_t)n_table * sizeof(int));
    launch(table);
  } else {
    launch(NoTable{});
  }
  int err = (int)hipGetLastError();
  if (err || cnt) return err;
  return topk_merge(cs, ci, splits, Q, K, result, s);
}

DA_EXPORT int da_topk_merge(void* cand_s, void* cand_i, int P, int Q, int K, void* out_s, void* out, const void* ids, int n_ids,
                            void* stream) {
  if (K < 1 || K > TK_MAX) return (int)hipErrorInvalidValue;
  if (Q == 0) return 0;
  return topk_merge(cand_s, cand_i, P, Q, K, top_out(out_s, out, ids, n_ids), (hipStream_t)stream);
}

DA_EXPORT int da_gather_ids(const void* rows, int n, const void* ids, int N, void* out, void* stream) {
  if (n < 0 || N < 0) return (int)hipErrorInvalidValue;
  if (n == 0) return 0;
  gather_ids_kernel<<<(n + 255) / 256, 256, 0, (hipStream_t)stream>>>((const int*)rows, n, (const long*)ids, N,
                                                                      (long*)out);
  DA_LAUNCH_CHECK();
}

DA_EXPORT int da_kmeans_accum(const void* X, int N, int d, const void* assign, void* sums, void* counts, void* stream) {
  if (N == 0) return 0;
  kmeans_accum_kernel<<<N, 256, 0, (hipStream_t)stream>>>((const bf16_t*)X, N, d, (const int*)assign, (float*)sums,
                                                           (float*)counts);
  DA_LAUNCH_CHECK();
}
