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
// Streaming dense scan (d % 128 == 0): the whole-shard pass of flat search, IVF coarse probing and
// k-means assignment, built to run at HBM speed.
//
//  * Every wave is an independent worker over its own contiguous run of rows, 16 rows per MFMA
//    tile, against the workgroup's 16 queries (B fragments from LDS, one copy per workgroup).
//  * The rows stream from HBM through a ring of R groups (4 MFMA k-steps = 64 B per lane each)
//    that runs across tile boundaries: group s + R is requested as soon as group s is consumed,
//    so ~R * 4 KB per wave stay in flight (the old kernel issued one row load, waited, issued the
//    next: 3.5 TB/s on a 10M x 1024 shard).
//  * A tile's 16 x 16 scores are tested against each query's running k-th best; only rows that beat
//    it do any top-K work (TdWave below).
//  * Up to 16 queries (one query block): topk_dense_stream_kernel, every wave its own rows, the
//    rows loaded non-temporally straight into the MFMA A registers.
//  * 17 and more: topk_dense_mq_kernel, the workgroup's 4 waves = 4 (or 8) query blocks over the SAME
//    rows: each 16-row tile is read from HBM once into LDS and feeds all four waves (B fragments of
//    a wave's queries live in its registers). Query blocks as separate workgroups over the same
//    rows, even dispatched back to back to one XCD, missed in L2 and read the shard once per block
//    (batch 64: 12.1 ms vs 3.6 ms for batch 1, profiles/r5/index/).
// out [row blocks (padded to 8), Q, K]: one unsorted top-K list per (workgroup, query), ordered and
// merged by topk_merge_kernel.
constexpr int TD_G = 4;    // MFMA k-steps (of 32) per load group: 64 B per lane

// One wave's top-K state for its 16 queries over a run of 16-row tiles. Per query, 64 LDS slots:
// [0, K) the current top-K (unsorted), then one candidate sub-buffer of SB slots for each of the
// query's 4 lanes; the k-th best score sits in a register of those lanes.
//  * tile(): a lane's rows that beat the k-th best pass the doc filter / floor and go to ITS
//    sub-buffer at a lane-local count: no cross-lane traffic on the append path.
//  * cut(): once a sub-buffer could overflow on the next tile, the query's list + buffered rows (one
//    per lane, <= 64) are cut to the top K by a radix select on the ballot unit: 32 rounds of ballot
//    + popcount on an order-preserving integer image of the score find the K-th largest (ties at
//    the threshold go to the smaller row id), the winners are compacted into [0, K) by mbcnt. The
//    sorted-list merge it replaces (K rounds of a 6-level shuffle argmax per (tile, query), then
//    per 48 candidates) stalled the workgroup's load pipeline: 64 queries took 10.5 ms against
//    3.7 ms with no candidate work (bench/scan_probe.py, profiles/r5/index/).
// Lists leave unsorted; topk_merge_kernel orders them.
constexpr int TD_SL = 64;  // LDS slots per (wave, query)

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

struct TdWave {
  float* cs; int* ci;  // [16][TD_SL] scores / rows
  int K, SB, lane, fr, fg;
  float kth;  // this lane's query (fr): its current k-th best score
  int cnt;    // entries in this lane's sub-buffer

  __device__ __forceinline__ void init(float* s, int* i, int k) {
    cs = s; ci = i; K = k; SB = (TD_SL - k) / 4;  // K <= 32: SB >= 8
    lane = threadIdx.x & 63; fr = lane & 15; fg = lane >> 4;
    kth = -INFINITY; cnt = 0;
    for (int j = lane; j < 16 * TD_SL; j += 64) { cs[j] = -INFINITY; ci[j] = -1; }
  }
  // cut the lists of the queries set in `full` (bit q) back to their top K
  __device__ __forceinline__ void flush(const unsigned long long full) {
    wave_sync_lds();
    float kq = -INFINITY;  // lane q < 16: query q's new k-th best
    for (unsigned long long left = full; left; left &= left - 1) {
      const int q = __builtin_ctzll(left);
      // lane j: list slot j (< K) or sub-buffer b = (j - K) / SB entry (j - K) % SB, live below the
      // count of lane q + 16 b
      const int b = lane < K ? 0 : min((lane - K) / SB, 3), e = lane < K ? 0 : lane - K - b * SB;
      const int nb = __shfl(cnt, q + 16 * b, 64);
      const bool live = lane < K || (lane < K + 4 * SB && e < nb);
      const float v = live ? cs[q * TD_SL + lane] : -INFINITY;
      const int id = live ? ci[q * TD_SL + lane] : -1;
      const float t = td_cut(v, id, K, lane, cs + q * TD_SL, ci + q * TD_SL);
      if (lane == q) kq = t;
    }
    const float kn = __shfl(kq, fr, 64);
    if ((full >> fr) & 1ull) { kth = kn; cnt = 0; }
  }
  // a finished 16 x 16 tile: lane (fr, fg) holds rows row0 + i (row0 = tile base + 4 fg) of query fr
  // (global query index qrow); rows from `end` on are padding. slot: the doc slot of row fr of the tile, loaded with
  // its rows (0 without slots): most tiles of a whole-shard pass have a candidate somewhere, and a load of its slot
  // here had every wave of the workgroup wait for memory once a tile.
  __device__ __forceinline__ void tile(const f32x4_t& acc, int row0, int end, bool qok, float thr, int slot,
                                       const unsigned* __restrict__ bitmap, int W, int qrow) {
    bool cand = false;
#pragma unroll
    for (int i = 0; i < 4; ++i) cand |= qok && row0 + i < end && acc[i] >= thr && acc[i] > kth;
    if (!__ballot(cand)) return;  // the common case after the first tiles
    float* bs = cs + fr * TD_SL + K + fg * SB;
    int* bi = ci + fr * TD_SL + K + fg * SB;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = row0 + i;
      const int sl = __shfl(slot, 4 * fg + i, 64);
      bool ok = qok && row < end && acc[i] >= thr && acc[i] > kth && sl >= 0;  // removed rows (slot -1) never match
      if (ok && bitmap) ok = (sl >> 5) < W && ((bitmap[(size_t)qrow * W + (sl >> 5)] >> (sl & 31)) & 1u);
      if (ok) { bs[cnt] = acc[i]; bi[cnt] = row; ++cnt; }
    }
    // a lane's next tile adds <= 4: cut the queries with a sub-buffer past SB - 4
    const unsigned long long over = __ballot(cnt > SB - 4);
    if (over) flush((over | (over >> 16) | (over >> 32) | (over >> 48)) & 0xffffull);
  }
  // every list cut to its top K (unsorted) in slots [0, K)
  __device__ __forceinline__ void finish() {
    const unsigned long long rest = __ballot(cnt > 0);
    if (rest) flush((rest | (rest >> 16) | (rest >> 32) | (rest >> 48)) & 0xffffull);
  }
  // merge another wave's finished lists (same 16 queries) into this wave's
  __device__ __forceinline__ void absorb(const float* os, const int* oi, int nq) {
    wave_sync_lds();
    for (int q = 0; q < nq; ++q) {
      const float v = lane < K ? cs[q * TD_SL + lane] : lane < 2 * K ? os[q * TD_SL + lane - K] : -INFINITY;
      const int id = lane < K ? ci[q * TD_SL + lane] : lane < 2 * K ? oi[q * TD_SL + lane - K] : -1;
      td_cut(v, id, K, lane, cs + q * TD_SL, ci + q * TD_SL);
    }
  }
  // lists of queries [0, nq) -> out[o0 + q * K + j] (o0: this list's (part, first query) offset)
  __device__ __forceinline__ void store(int nq, size_t o0, float* __restrict__ os, int* __restrict__ oi) {
    wave_sync_lds();
    for (int i = lane; i < nq * K; i += 64) {
      const int q = i / K, j = i % K;
      os[o0 + i] = cs[q * TD_SL + j];
      oi[o0 + i] = ci[q * TD_SL + j];
    }
  }
};

// NG = d / 128 load groups per 16-row tile (3, 6, 8: d = 384, 768, 1024): the ring holds one whole
// tile ahead (NG * 4 KB per wave in flight), every load of the loop body unconditional (clamped),
// so the compiler's vmcnt waits stay counted.
template <int NG>
__global__ void __launch_bounds__(256)
topk_dense_stream_kernel(const bf16_t* __restrict__ X, int N, const int* __restrict__ slots,
                         const bf16_t* __restrict__ Qv, int Q, const unsigned* __restrict__ bitmap, int W, float thr,
                         int K, int rows_per_wave, int nqb, float* __restrict__ out_s, int* __restrict__ out_i) {
  constexpr int d = NG * 32 * TD_G;
  constexpr int qstr = d * 2 + 16;
  __shared__ __attribute__((aligned(16))) char sQ[16 * qstr];   // [16][d] bf16, rows padded by 16 B
  __shared__ float cs_all[4][16 * TD_SL];  // per wave: top-K lists + candidate buffers (TdWave)
  __shared__ int ci_all[4][16 * TD_SL];

  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int fr = lane & 15, fg = lane >> 4;
  // XCD-grouped block order: blocks b and b + 8 i share an XCD; the nqb query blocks of row block rb
  // are b = (rb / 8) * 8 nqb + j * 8 + rb % 8
  const int b = blockIdx.x, per = 8 * nqb;
  const int grp = b / per, rem = b % per;
  const int qb = rem / 8, rb = grp * 8 + rem % 8;
  const int qbase = qb * 16, nq = min(16, Q - qbase);
  for (int i = tid; i < 16 * (d / 8); i += 256) {
    const int r = i / (d / 8), c = i % (d / 8);
    u32x4_t v = u32x4_t{0, 0, 0, 0};
    if (r < nq) v = *(const u32x4_t*)(Qv + (size_t)(qbase + r) * d + c * 8);
    *(u32x4_t*)(sQ + r * qstr + c * 16) = v;
  }
  TdWave st;
  st.init(cs_all[wid], ci_all[wid], K);
  __syncthreads();

  const int wbeg = (int)min((long)N, ((long)rb * 4 + wid) * rows_per_wave);
  const int wend = (int)min((long)N, (long)wbeg + rows_per_wave);
  const int ntile = (wend - wbeg + 15) / 16;
  const int lrow = N - 1;
  const int* sp = slots ? slots : (const int*)X;  // (without slots some word of X: loaded all the same, not used)
  auto gload = [&](u32x4_t (&v)[NG][TD_G], int t) {  // tile t's fragments (rows clamped)
    const int row = min(wbeg + t * 16 + fr, lrow);
    const bf16_t* p = X + (size_t)row * d + fg * 8;
#pragma unroll
    for (int g = 0; g < NG; ++g)
#pragma unroll
      for (int j = 0; j < TD_G; ++j) v[g][j] = __builtin_nontemporal_load((const u32x4_t*)(p + (g * TD_G + j) * 32));
  };
  u32x4_t ring[NG][TD_G];
  gload(ring, 0);
  int sl_next = sp[min(wbeg + fr, lrow)];
  const bool qok = fr < nq;
  for (int t = 0; t < ntile; ++t) {
    f32x4_t acc = f32x4_t{0.f, 0.f, 0.f, 0.f};
    const int row_next = min(wbeg + (t + 1) * 16 + fr, lrow);
    const int sl = slots ? sl_next : 0;
    sl_next = sp[row_next];
    const bf16_t* pn = X + (size_t)row_next * d + fg * 8;
#pragma unroll
    for (int g = 0; g < NG; ++g) {
#pragma unroll
      for (int j = 0; j < TD_G; ++j) {
        const int kk = g * TD_G + j;
        const bf16x8_t bq = *(const bf16x8_t*)(sQ + fr * qstr + kk * 64 + fg * 16);
        acc = mfma16(__builtin_bit_cast(bf16x8_t, ring[g][j]), bq, acc);
      }
      // group g of the NEXT tile into the slot just consumed (one tile of loads stays in flight)
#pragma unroll
      for (int j = 0; j < TD_G; ++j)
        ring[g][j] = __builtin_nontemporal_load((const u32x4_t*)(pn + (g * TD_G + j) * 32));
    }
    st.tile(acc, wbeg + t * 16 + fg * 4, wend, qok, thr, sl, bitmap, W, qbase + fr);
  }
  st.finish();
  // the 4 waves' lists -> one per workgroup (wave 0 absorbs the others'), out [rb, Q, K]
  __syncthreads();
  if (wid == 0) {
    for (int w = 1; w < 4; ++w) st.absorb(cs_all[w], ci_all[w], nq);
    st.store(nq, ((size_t)rb * Q + qbase) * K, out_s, out_i);
  }
}

// 17 and more queries: NW waves of 16 queries each per workgroup (8 from 65 queries on, so that a shard is read once
// for up to 128). rows_per_block rows per workgroup (multiple of 16), grid = row blocks (padded to 8) x query groups:
// the nqg groups of one row block are dispatched to one XCD back to back. A tile: 16 rows x d, 16 B per thread per load
// (NL loads) and the rows' doc slots, TD_PF tiles in flight in registers, written to one of two LDS buffers (16-B
// chunk c of row r at c ^ (r & 15): the 16 rows one ds_read_b128 lane group reads hit 16 distinct slots), one barrier
// per tile. The queries' fragments stay in registers (d / 8 of them).
// Bound by HBM, and by what a SIMD does between tiles when it has one wave only: a pass of 128 queries x 1.25 M rows x
// 1024 took 2304 us with 64 queries per workgroup, slots loaded where a candidate turned up and cuts of always 32
// rounds, 1087 us with 4 waves of 32 queries each, and 808 us (3.2 TB/s) with two waves per SIMD, whose waits overlap.
constexpr int TD_PF = 3;

template <int NG, int NW>
__global__ void __launch_bounds__(64 * NW, 1)
topk_dense_mq_kernel(const bf16_t* __restrict__ X, int N, const int* __restrict__ slots,
                     const bf16_t* __restrict__ Qv, int Q, const unsigned* __restrict__ bitmap, int W, float thr,
                     int K, int rows_per_block, int nqg, float* __restrict__ out_s, int* __restrict__ out_i) {
  constexpr int d = NG * 128, NK = d / 32, CPR = d / 8, RB = d * 2, TB = 16 * RB, NT = 64 * NW;
  constexpr int NL = (16 * CPR + NT - 1) / NT;  // 16-B loads of a thread per tile
  __shared__ __attribute__((aligned(16))) char sX[2][TB];
  __shared__ float cs_all[NW][16 * TD_SL];
  __shared__ int ci_all[NW][16 * TD_SL];

  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int fr = lane & 15, fg = lane >> 4;
  const int b = blockIdx.x, per = 8 * nqg;
  const int grp = b / per, rem = b % per;
  const int qg = rem / 8, rb = grp * 8 + rem % 8;
  const int qbase = (qg * NW + wid) * 16, nq = max(0, min(16, Q - qbase));
  const bool qok = fr < nq;
  // this wave's B fragments: query qbase + fr, columns 32 kk + 8 fg .. + 8
  bf16x8_t bq[NK];
#pragma unroll
  for (int kk = 0; kk < NK; ++kk)
    bq[kk] = *(const bf16x8_t*)(Qv + (size_t)min(qbase + fr, Q - 1) * d + kk * 32 + fg * 8);
  TdWave st;
  st.init(cs_all[wid], ci_all[wid], K);

  const int rbeg = (int)min((long)N, (long)rb * rows_per_block);
  const int rend = (int)min((long)N, (long)rbeg + rows_per_block);
  const int ntile = (rend - rbeg + 15) / 16;
  const int tl = max(ntile - 1, 0);
  // buffer loads: one scalar offset per tile, rows past the workgroup's last return zeros (masked in tile()).
  // Without slots some words of X are loaded in their place, and not used.
  const __amdgpu_buffer_rsrc_t rsx = __builtin_amdgcn_make_buffer_rsrc((void*)(X + (size_t)rbeg * d), (short)0,
                                                                       (rend - rbeg) * RB, 0x00020000);
  const __amdgpu_buffer_rsrc_t rss = __builtin_amdgcn_make_buffer_rsrc(
      slots ? (void*)(slots + rbeg) : (void*)(X + (size_t)rbeg * d), (short)0, (rend - rbeg) * 4, 0x00020000);
  unsigned voff[NL];   // chunk tid + NT i of a tile (one past its end: out of range, loads nothing)
  int loff[NL];
#pragma unroll
  for (int i = 0; i < NL; ++i) {
    const int idx = tid + NT * i, r = idx / CPR, c = idx % CPR;
    voff[i] = idx < 16 * CPR ? idx * 16u : 0x7ffffff0u;
    loff[i] = r * RB + ((c ^ (r & 15)) << 4);
  }
  auto gload = [&](u32x4_t (&v)[NL], int& sl, int t) {  // tile t <= tl
#pragma unroll
    for (int i = 0; i < NL; ++i)
      v[i] = __builtin_amdgcn_raw_buffer_load_b128(rsx, voff[i], t * TB, 2);  // non-temporal
    sl = __builtin_amdgcn_raw_buffer_load_b32(rss, fr * 4, t * 64, 0);
  };
  auto lstore = [&](const u32x4_t (&v)[NL], int buf) {
#pragma unroll
    for (int i = 0; i < NL; ++i)
      if ((i + 1) * NT <= 16 * CPR || tid + NT * i < 16 * CPR) *(u32x4_t*)(&sX[buf][loff[i]]) = v[i];
  };
  int xo[4];  // where chunk 4 kk + fg of row fr is: the swizzle only touches the chunk's low four bits
#pragma unroll
  for (int j = 0; j < 4; ++j) xo[j] = fr * RB + (((j * 4 + fg) ^ fr) << 4);
  __syncthreads();  // the lists' initial values (before any load is in flight: this drains them)
  u32x4_t ring[TD_PF][NL];
  int slot[TD_PF];
#pragma unroll
  for (int u = 0; u < TD_PF; ++u) {
    gload(ring[u], slot[u], min(u, tl));
    asm volatile("" ::: "memory");  // issue order = tile order (counted waits)
  }
  // whole groups of TD_PF tiles (no exit inside the unrolled group: the ring keeps fixed registers);
  // tiles past the end re-read the last one and mask every row
  for (int t0 = 0; t0 < ntile; t0 += TD_PF) {
#pragma unroll
    for (int u = 0; u < TD_PF; ++u) {
      const int t = t0 + u;
      const int buf = t & 1, sl = slots ? slot[u] : 0;
      lstore(ring[u], buf);
      gload(ring[u], slot[u], min(t + TD_PF, tl));  // clamped past the end: uniform counts
      // tile t visible to every wave, and every wave is done with tile t - 2 (same buffer): a raw
      // barrier (__syncthreads() would drain the loads in flight)
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      f32x4_t acc = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kk = 0; kk < NK; ++kk)
        acc = mfma16(*(const bf16x8_t*)(&sX[buf][xo[kk & 3] + (kk >> 2) * 256]), bq[kk], acc);
      st.tile(acc, rbeg + t * 16 + fg * 4, rend, qok, thr, sl, bitmap, W, qbase + fr);
    }
  }
  st.finish();
  st.store(nq, ((size_t)rb * Q + qbase) * K, out_s, out_i);
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

// Per-query row ranges: ranges [R, 2] (start, end) and range_off [Q + 1], or (lists [Q, probes] != null) rows
// ranges[l] .. ranges[l + 1] of each list l that the query names (l < 0: none). rows_per_split rows of the query's concatenated ranges per
// workgroup (grid = (splits, Q)). out [splits, Q, K], unsorted lists (topk_merge_kernel orders them).
//
// A half-wave owns a row (16 B per lane and load, NCH loads), four rows of it are on their way together; 64 rows
// are scored per step and handed to wave 0, which keeps the list while the others score the next 64 (two buffers,
// one barrier a step). Bound by the latency of a step for few rows, by HBM for many: the caller splits a query's
// rows over as many workgroups as fill the chip (388 rows of 8 documents: one workgroup took 105 us, with one load
// in flight and a shuffle merge of K rounds per 64 rows; 7 workgroups take 15 us. 24 queries over 8 lists of about
// 780 rows x 768: 162 -> 41 us).
template <int NCH>
__global__ void __launch_bounds__(256)
topk_ranges_kernel(const bf16_t* __restrict__ X, int d, const int* __restrict__ slots,
                   const bf16_t* __restrict__ Qv, int Q, const int* __restrict__ ranges,
                   const int* __restrict__ range_off, const int* __restrict__ lists, int probes,
                   const unsigned* __restrict__ bitmap, int W, float thr,
                   int K, int rows_per_split, float* __restrict__ out_s, int* __restrict__ out_i) {
  __shared__ float sc[2][64];
  __shared__ int sr[2][64];
  __shared__ float cs[TL_SL];
  __shared__ int ci[TL_SL];
  const int split = blockIdx.x, q = blockIdx.y;
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const int half = lane >> 5, l32 = lane & 31;
  TopList top;
  top.init(cs, ci, K);  // (every wave writes the same empty list; wave 0 keeps it)
  const int nch = d / 8;  // 16-B chunks of a row; this lane has chunks l32 + 32 i
  float qv[NCH][8];
#pragma unroll
  for (int i = 0; i < NCH; ++i) {
    const int c = l32 + 32 * i;
    u32x4_t u = *(const u32x4_t*)(Qv + (size_t)q * d + min(c, nch - 1) * 8);
#pragma unroll
    for (int e = 0; e < 8; ++e) qv[i][e] = bf2f((bf16_t)((e & 1) ? (u[e >> 1] >> 16) : (u[e >> 1] & 0xffff)));
  }
  const int rb = lists ? q * probes : range_off[q], re = lists ? rb + probes : range_off[q + 1];
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
      const int len = ranges[at + 1] - ranges[at];
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
    const int s0 = ranges[lists ? l : 2 * r], s1 = ranges[lists ? l + 1 : 2 * r + 1];
    const int len = s1 - s0;
    const int lo = max(pbeg, pos), hi = min(pend, pos + len);
    for (int p0 = lo; p0 < hi; p0 += 64) {
      // 64 rows per step: 8 half-waves x 8 rows, 4 at a time
#pragma unroll
      for (int j0 = 0; j0 < 8; j0 += 4) {
        const int rl = (wid * 2 + half) * 8 + j0;
        u32x4_t u[4][NCH];
#pragma unroll
        for (int j = 0; j < 4; ++j) {  // rows and chunks past the end: the last one's
          const bf16_t* xr = X + (size_t)(s0 + (min(p0 + rl + j, hi - 1) - pos)) * d;
#pragma unroll
          for (int i = 0; i < NCH; ++i) u[j][i] = *(const u32x4_t*)(xr + min(l32 + 32 * i, nch - 1) * 8);
        }
        float dot[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < NCH; ++i) {
          const bool in = l32 + 32 * i < nch;
#pragma unroll
          for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int e = 0; e < 8; ++e) {
              const float x = bf2f((bf16_t)((e & 1) ? (u[j][i][e >> 1] >> 16) : (u[j][i][e >> 1] & 0xffff)));
              const float t = dot[j] + qv[i][e] * x;
              dot[j] = in ? t : dot[j];
            }
        }
#pragma unroll
        for (int o = 16; o > 0; o >>= 1)
#pragma unroll
          for (int j = 0; j < 4; ++j) dot[j] += __shfl_xor(dot[j], o, 64);
        // lane j of a half-wave hands in row j
        const float s = (l32 == 0 ? dot[0] : l32 == 1 ? dot[1] : l32 == 2 ? dot[2] : dot[3]);
        if (l32 < 4) {
          const int p = p0 + rl + l32, row = s0 + (p - pos);
          bool ok = p < hi && s >= thr && s != -INFINITY;
          if (ok && slots) {
            const int sl = slots[row];
            ok = sl >= 0 && (!bitmap || ((sl >> 5) < W && ((bitmap[(size_t)q * W + (sl >> 5)] >> (sl & 31)) & 1u)));
          }
          sc[buf][rl + l32] = s;
          sr[buf][rl + l32] = ok ? row : -1;
        }
      }
      __syncthreads();  // this step's scores are in, and the list has taken the last step's
      if (wid == 0) top.add(sc[buf][lane], sr[buf][lane]);
      buf ^= 1;
    }
    pos += len;
    if (pos >= pend) break;
  }
  if (wid == 0) {
    wave_sync_lds();
    if (lane < K) {
      const size_t o = ((size_t)split * Q + q) * K + lane;
      out_s[o] = cs[lane];
      out_i[o] = ci[lane];
    }
  }
}

// cand [P, Q, K] -> out [Q, K] sorted desc (ties: smaller row id). One workgroup per query, a wave per 64 candidates
// up to 16 (TM_WAVES): each wave cuts its share to K, wave 0 joins the lists and orders them by counting the better
// ones of each. Bound by the chain of cuts (about 1 us each), hence many waves: K rounds of a workgroup-wide argmax
// with two barriers each took 18 us for 256 parts of K = 5, cuts by 4 waves 23 us, by 16 16.5 us.
constexpr int TM_WAVES = 16;

__global__ void __launch_bounds__(64 * TM_WAVES)
topk_merge_kernel(const float* __restrict__ cand_s, const int* __restrict__ cand_i, int P, int Q, int K,
                  float* __restrict__ os, int* __restrict__ oi) {
  __shared__ float cs[TM_WAVES][TL_SL];
  __shared__ int ci[TM_WAVES][TL_SL];
  const int q = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wid = tid >> 6, nt = blockDim.x;
  const int n = P * K;
  TopList top;
  top.init(cs[wid], ci[wid], K);
  for (int j0 = wid * 64; j0 < n; j0 += nt * 4) {
    float v[4];
    int id[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {  // issued together: the lists come from all over the chip's caches
      const int j = j0 + lane + nt * u, jc = min(j, n - 1);
      const size_t o = ((size_t)(jc / K) * Q + q) * K + jc % K;
      v[u] = cand_s[o];
      id[u] = j < n ? cand_i[o] : -1;
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) top.add(v[u], id[u]);
  }
  __syncthreads();
  if (wid) return;
  const int rest = (nt / 64 - 1) * K;  // the other waves' lists, one after another
  for (int e0 = 0; e0 < rest; e0 += 64) {
    const int e = e0 + lane, w = 1 + min(e, max(rest - 1, 0)) / K;
    top.add(cs[w][e % K], e < rest ? ci[w][e % K] : -1);
  }
  wave_sync_lds();
  const float v = lane < K ? cs[0][lane] : -INFINITY;
  const int id = lane < K ? ci[0][lane] : -1;
  int rank = 0;
  for (int j = 0; j < K; ++j) {
    const float vj = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(v), j));
    const int ij = __builtin_amdgcn_readlane(id, j);
    rank += ij >= 0 && (better(vj, ij, v, id) || (vj == v && ij == id && j < lane));  // (a row named twice)
  }
  const int real = __popcll(__ballot(id >= 0));
  if (id >= 0) {
    os[(size_t)q * K + rank] = v;
    oi[(size_t)q * K + rank] = id;
  }
  if (lane >= real && lane < K) {
    os[(size_t)q * K + lane] = -INFINITY;
    oi[(size_t)q * K + lane] = -1;
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

static int topk_merge(const void* cs, const void* ci, int P, int Q, int K, void* out_s, void* out_i, hipStream_t s) {
  const long waves = min((long)TM_WAVES, max(1L, ((long)P * K + 63) / 64));
  topk_merge_kernel<<<Q, 64 * (int)waves, 0, s>>>((const float*)cs, (const int*)ci, P, Q, K, (float*)out_s, (int*)out_i);
  DA_LAUNCH_CHECK();
}

DA_EXPORT size_t da_topk_dense_ws(int N, int Q, int K, int rows_per_block) {
  const int nblk = (N + rows_per_block - 1) / rows_per_block;
  return (size_t)nblk * Q * K * 8;
}

DA_EXPORT int da_topk_dense(const void* X, int N, int d, const void* slots, const void* Qv, int Q, const void* bitmap,
                            int W, float thr, int K, int rows_per_block, void* ws, void* out_s, void* out_i,
                            void* stream) {
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
  return topk_merge(cs, ci, nblk, Q, K, out_s, out_i, s);
}

// The streaming scan (d = 384, 768 or 1024): ws holds (row blocks padded to 8) * 4 * Q * K candidate
// pairs; rows_per_wave % 16 == 0. hipErrorInvalidValue for shapes it does not take (the caller
// then uses da_topk_dense).
static long blocks8(long N, long rows) { return ((N + rows - 1) / rows + 7) / 8 * 8; }
// rows per workgroup of the shared-tile kernel: one workgroup per CU over the whole shard (each pays the early top-K
// fill once), one tile at least, 1 GB at most (its 32-bit offsets)
static int mq_rows(long N) { return (int)min(524288L, max(16L, (N + 256 * 16 - 1) / (256 * 16) * 16)); }

DA_EXPORT size_t da_topk_stream_ws(int N, int Q, int K, int rows_per_wave) {
  const long parts = Q <= 16 ? blocks8(N, 4L * rows_per_wave) : blocks8(N, mq_rows(N));
  return (size_t)parts * Q * K * 8;
}

DA_EXPORT int da_topk_dense_stream(const void* X, int N, int d, const void* slots, const void* Qv, int Q,
                                   const void* bitmap, int W, float thr, int K, int rows_per_wave, void* ws,
                                   void* out_s, void* out_i, void* stream) {
  if ((d != 384 && d != 768 && d != 1024) || K < 1 || K > TK_MAX || rows_per_wave % 16 || rows_per_wave <= 0 ||
      N < 1)
    return (int)hipErrorInvalidValue;
  if (Q == 0) return 0;
  hipStream_t s = (hipStream_t)stream;
  const int rpb = mq_rows(N), qper = Q > 64 ? 128 : 64, nqg = (Q + qper - 1) / qper;
  const long parts = Q <= 16 ? blocks8(N, 4L * rows_per_wave) : blocks8(N, rpb);
  if (parts * nqg > 0x7fffffffL) return (int)hipErrorInvalidValue;
  float* cs = (float*)ws;
  int* ci = (int*)(cs + (size_t)parts * Q * K);
#define TDQ(NG, NW)                                                                                     \
  topk_dense_mq_kernel<NG, NW><<<(int)parts * nqg, 64 * NW, 0, s>>>((const bf16_t*)X, N,                \
      (const int*)slots, (const bf16_t*)Qv, Q, (const unsigned*)bitmap, W, thr, K, rpb, nqg, cs, ci)
#define TDS(NG)                                                                                         \
  do {                                                                                                  \
    if (Q <= 16)                                                                                        \
      topk_dense_stream_kernel<NG><<<(int)parts, 256, 0, s>>>((const bf16_t*)X, N, (const int*)slots,   \
          (const bf16_t*)Qv, Q, (const unsigned*)bitmap, W, thr, K, rows_per_wave, 1, cs, ci);           \
    else if (Q <= 64)                                                                                   \
      TDQ(NG, 4);                                                                                       \
    else                                                                                                \
      TDQ(NG, 8);                                                                                       \
  } while (0)
  switch (d) {
    case 384: TDS(3); break;
    case 768: TDS(6); break;
    default: TDS(8); break;
  }
#undef TDS
#undef TDQ
  int err = (int)hipGetLastError();
  if (err) return err;
  return topk_merge(cs, ci, (int)parts, Q, K, out_s, out_i, s);
}

DA_EXPORT int da_topk_ranges(const void* X, int d, const void* slots, const void* Qv, int Q, const void* ranges,
                             const void* range_off, const void* lists, int probes, const void* bitmap, int W,
                             float thr, int K, int splits, int rows_per_split, void* ws, void* out_s, void* out_i,
                             void* stream) {
  if (d % 8 || d < 8 || d > 4096 || K < 1 || K > TK_MAX || splits < 1 || rows_per_split < 1 ||
      (!range_off && (!lists || probes < 0)))
    return (int)hipErrorInvalidValue;
  if (Q == 0) return 0;
  hipStream_t s = (hipStream_t)stream;
  float* cs = (float*)ws;
  int* ci = (int*)(cs + (size_t)splits * Q * K);
  dim3 grid(splits, Q);
#define TRG(NCH)                                                                                                    \
  topk_ranges_kernel<NCH><<<grid, 256, 0, s>>>((const bf16_t*)X, d, (const int*)slots, (const bf16_t*)Qv, Q,        \
                                               (const int*)ranges, (const int*)range_off, (const int*)lists,        \
                                               probes, (const unsigned*)bitmap, W, thr, K, rows_per_split, cs, ci)
  if (d <= 256) TRG(1);
  else if (d <= 512) TRG(2);
  else if (d <= 768) TRG(3);
  else if (d <= 1024) TRG(4);
  else if (d <= 2048) TRG(8);
  else TRG(16);
#undef TRG
  int err = (int)hipGetLastError();
  if (err) return err;
  return topk_merge(cs, ci, splits, Q, K, out_s, out_i, s);
}

DA_EXPORT int da_topk_merge(void* cand_s, void* cand_i, int P, int Q, int K, void* out_s, void* out_i, void* stream) {
  if (K < 1 || K > TK_MAX) return (int)hipErrorInvalidValue;
  if (Q == 0) return 0;
  return topk_merge(cand_s, cand_i, P, Q, K, out_s, out_i, (hipStream_t)stream);
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
