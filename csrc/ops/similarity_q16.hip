// Two-stage EXACT filtered top-k over a 16-bit fixed-point semantic index: half the bytes
// a pass of the bf16 one (reference semantics pilott/memory/enhanced_memory.py:
// 93-116 semantic_search, filters as csrc/ops/similarity.hip).
//
// Storage (memory/semantic_index.py storage="q16"): every L2-normalised row x is kept as
// v = round(x / s_r), |v| <= 32512 (s_r = max|x| / 32512 per row), split into two int8 planes
//     hi = floor((v + 128) / 256)  in [-127, 127],   lo = v - 256 hi  in [-128, 127],
// each plane fragment-major in 16-row tiles for v_mfma_i32_16x16x64_i8:
//     plane[t][s][16 g + c][j] = plane_row(16 t + c)[64 s + 16 g + j]       (16 B per lane)
// plus per row (s_r, b_r = s_r ||lo||_2). Queries are quantised the same way (v_q = 256 qh +
// ql, scale s_q, c_q = s_q ||v_q||_2). The EXACT score of (row, query) is
//     S = s_r s_q (v_q . v_r) = s_r s_q (65536 qh.hi + 256 (qh.lo + ql.hi) + ql.lo)
// from four exact int32 dot products (exact_score below; the CPU reference in
// ops/reference.py q16_topk evaluates the same int64 sum and the same float64 -> float32 step,
// so GPU and reference agree bit for bit). 16-bit fixed point resolves each coordinate to
// ~3e-6 -- finer than the bf16 index's 2^-9 relative.
//
// Stage 1 (one pass, hi plane ONLY: 1 byte per dimension instead of the bf16 index's 2):
//     S^ = s_r s_q (65536 qh.hi + 256 ql.hi),     |S - S^| = s_r s_q |v_q . lo| <= c_q b_r = E
// (Cauchy-Schwarz), so L = S^ - E <= S <= U = S^ + E. Each workgroup (a slice of rows, 16
// waves, every wave a 16-row group x every query tile, two MFMAs per 64-dim k-step) keeps
// per query the rows with the C best upper bounds U, admitting a row only if U beats both the
// C-th best U so far (capacity) and the K-th best LOWER bound so far (tau_slice: k rows already
// score at least that, so a row whose U is below it cannot be in the top-k). A row refused
// for capacity marks the slice: its drop level (the C-th best U) is reported.
// Stage 2 (one workgroup per query): tau = the K-th best L over every slice's list (the global
// top-k by L is inside the union: a row missing from it was refused for capacity, and the
// drop check below catches that); every listed row with U >= tau is re-ranked EXACTLY (one
// wave per row gathers its hi and lo fragments and runs the four integer dot products), and
// the K best exact scores are the answer. If some slice's drop level reaches tau, a dropped
// row might belong to the top-k: the query is flagged and the host re-runs the batch with the
// exact scan (EXACT = true: both planes, exact scores in stage 1), so the result is always
// exact. On random unit vectors at 100M rows the band [tau - 2E, tau] holds a few hundred rows
// (E ~ 0.008 against a score spread of 1/sqrt(D) = 0.031), far below the lists' 16K entries.
#include "topk_select.h"

namespace pa {
namespace q16 {

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef signed char i8x16 __attribute__((ext_vector_type(16)));

constexpr int CAND = 512;     // candidate buffer per (slice, query), power of two
constexpr int C = 64;         // list entries kept per (slice, query): the best C upper bounds
constexpr int MAXK = 64;
constexpr int QT = 16;        // queries per MFMA tile
constexpr int MAXQ = 64;
constexpr int MAXD = 1024;
constexpr int THREADS = 1024; // 16 waves
constexpr int NW = THREADS / 64;
// One round of the bound scan (8 waves x 32 rows) a slice at least: 20,000 rows give 79 slices. With 2,048 rows a slice,
// which the sorting compactions needed, they gave 10 and the pass took 0.5 ms.
constexpr int MIN_ROWS_PER_WG = 256;
constexpr int MAX_WG = 256;   // one resident workgroup per CU

__host__ __device__ inline int num_wg(int N) {
  int nwg = (N + MIN_ROWS_PER_WG - 1) / MIN_ROWS_PER_WG;
  if (nwg > MAX_WG) nwg = MAX_WG;
  if (nwg < 1) nwg = 1;
  return nwg;
}

// the exact score (see the header); the ONLY place the integer sums become a float
__device__ __forceinline__ float exact_score(int hh, int hl, int lh, int ll, float sr, float sq) {
  const long long I = (long long)hh * 65536 + ((long long)hl + (long long)lh) * 256 + (long long)ll;
  return (float)((double)I * ((double)sr * (double)sq));
}

struct QState {  // per-query admission state of one slice (LDS)
  int cnt[MAXQ];
  float theta[MAXQ];    // admission threshold = max(cap, tauL)
  float cap[MAXQ];      // C-th best U kept (-inf until C entries)
  float tauL[MAXQ];     // K-th best L among the kept entries (-inf until K)
  int dropped[MAXQ];    // a row was refused (or truncated) for capacity
  uint32_t top[MAXQ];   // best L admitted (ordered key, 0: none)
  int minp[MAXQ];
  uint64_t qtag[MAXQ];
  float sq[MAXQ];
  float cq[MAXQ];
};

// Compact query q's global buffer to its best C upper bounds and refresh cap / tauL / theta: one wave a query, so a
// workgroup's waves compact as many queries at once, with no barrier. Selecting by bits takes about a microsecond a
// query; a bitonic sort by the whole workgroup took 15, one query after the other (3 of the 4 ms of a pass over 4M rows).
// ou / ol / orow: where the slice's list goes, or null to keep it in the buffer.
__device__ __forceinline__ void compact(float* gu, float* gl, int* gr, QState& st, int q, int K, float* ou = nullptr,
                                        float* ol = nullptr, int* orow = nullptr) {
  constexpr int PER = CAND / 64;
  const int lane = threadIdx.x & 63;
  const float bound = st.tauL[q];
  const int n = min(st.cnt[q], CAND);
  int held = 0;
  uint32_t ku[PER], kl[PER];
  int rows[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int e = i * 64 + lane;
    const bool ok = e < n;
    const float u = ok ? gu[e] : 0.f;
    ku[i] = ok && !(u < bound) ? ord_key(u) : 0;  // (entries that the bound has overtaken go)
    kl[i] = ku[i] ? ord_key(gl[e]) : 0;
    rows[i] = ok ? gr[e] : -1;
    held += __popcll(__ballot(ku[i] != 0));
  }
  uint32_t cut = 1;  // entries above it stay, and of those at it as many as there is room for
  int room = C;
  if (held >= C) {
    cut = wave_select(ku, C);
#pragma unroll
    for (int i = 0; i < PER; ++i) room -= __popcll(__ballot(ku[i] > cut));
  }
  if (ou) { gu = ou; gl = ol; gr = orow; }
  int at = 0;
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const unsigned long long ties = __ballot(ku[i] == cut);
    const bool keep = ku[i] > cut || (ku[i] == cut && rank_in(ties) < room);
    room -= __popcll(ties);
    const unsigned long long kept = __ballot(keep);
    if (keep) {
      const int p = at + rank_in(kept);
      gu[p] = key_value(ku[i]);
      gl[p] = key_value(kl[i]);
      gr[p] = rows[i];
    } else {
      kl[i] = 0;
    }
    at += __popcll(kept);
  }
  if (ou && lane >= at) { gu[lane] = -INFINITY; gl[lane] = -INFINITY; gr[lane] = -1; }
  uint32_t kth = 0;
  if (at >= K) kth = wave_select(kl, K);  // any subset's K-th best L is a valid bound
  if (lane == 0) {
    st.cnt[q] = at;
    if (held > C) st.dropped[q] = 1;
    if (at == C) st.cap[q] = key_value(cut);
    if (at >= K) st.tauL[q] = fmaxf(st.tauL[q], key_value(kth));
    st.theta[q] = fmaxf(st.cap[q], st.tauL[q]);
  }
}

// Stage 1 over both planes, U = L = the exact score (the fallback scan): 8 waves, four accumulators per query tile.
__global__ __launch_bounds__(512) void stage1_exact_kernel(
    float* __restrict__ out_u, float* __restrict__ out_l, int* __restrict__ out_r, float* __restrict__ out_drop,
    float* __restrict__ cand_u, float* __restrict__ cand_l, int* __restrict__ cand_r,
    const signed char* __restrict__ qv, const float* __restrict__ qmeta, const signed char* __restrict__ hi,
    const signed char* __restrict__ lo, const float* __restrict__ rmeta, int Q, int N, int D, int K,
    const int* __restrict__ row_prio, const uint64_t* __restrict__ row_tags, const float* __restrict__ row_exp,
    const int* __restrict__ q_minp, const uint64_t* __restrict__ q_tags, float now) {
  constexpr int TH = 512, NWV = TH / 64;
  constexpr int KB = 2;  // k-steps per load batch (16 B per lane per plane and step)
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int NQT = (Q + QT - 1) / QT;
  const int QLD = D + 16;  // padded LDS row (bytes): the 16 query rows of a fragment spread over the banks
  signed char* qh = reinterpret_cast<signed char*>(smem);           // [NQT*16][QLD]
  signed char* ql = qh + (size_t)NQT * QT * QLD;                    // [NQT*16][QLD]
  QState& st = *reinterpret_cast<QState*>(ql + (size_t)NQT * QT * QLD);
  // [2] some query's buffer must be compacted, by rounds in turn: a wave that is a round ahead must not be taken for this
  // one's (the others would miss its barrier)
  int* need = reinterpret_cast<int*>(&st + 1);

  const int nwg = gridDim.x, wg = blockIdx.x;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int g = lane >> 4, col = lane & 15;
  const int DS = D / 64;
  // queries: qv [Q][2][D] (qh, ql) -> LDS, zero rows past Q
  for (int v = threadIdx.x; v < NQT * QT * 2 * (D / 16); v += TH) {
    const int r = v / (2 * (D / 16)), rem = v % (2 * (D / 16));
    const int plane = rem / (D / 16), c16 = (rem % (D / 16)) * 16;
    i32x4 x = i32x4{0, 0, 0, 0};
    if (r < Q) x = *reinterpret_cast<const i32x4*>(qv + ((size_t)r * 2 + plane) * D + c16);
    *reinterpret_cast<i32x4*>((plane ? ql : qh) + (size_t)r * QLD + c16) = x;
  }
  if (threadIdx.x < MAXQ) {
    const int q = threadIdx.x;
    st.cnt[q] = 0;
    st.theta[q] = -INFINITY;
    st.cap[q] = -INFINITY;
    st.tauL[q] = -INFINITY;
    st.dropped[q] = 0;
    st.top[q] = 0;
    st.minp[q] = q < Q ? q_minp[q] : 0x7fffffff;
    st.qtag[q] = q < Q ? q_tags[q] : 0ull;
    st.sq[q] = q < Q ? qmeta[2 * q] : 0.f;
    st.cq[q] = q < Q ? qmeta[2 * q + 1] : 0.f;
  }
  if (threadIdx.x < 2) need[threadIdx.x] = 0;
  __syncthreads();

  float* my_u = cand_u + (size_t)wg * MAXQ * CAND;
  float* my_l = cand_l + (size_t)wg * MAXQ * CAND;
  int* my_r = cand_r + (size_t)wg * MAXQ * CAND;
  const int per = ((N + nwg - 1) / nwg + 15) / 16 * 16;
  const int r0 = wg * per, r1 = min(N, r0 + per);
  const int ngroups = (max(0, r1 - r0) + 15) / 16;
  const int nrounds = (ngroups + NWV - 1) / NWV;

  auto frag_off = [&](int grp_, int s) -> size_t {  // byte offset of this lane's fragment, k-step s
    return (((size_t)((r0 + grp_ * 16) >> 4) * DS + s) * 64 + lane) * 16;
  };
  // branch-free: k-steps past D re-read the last one (never used: compute stops at DS) -- a
  // conditional load splits the block and the wait-count pass then drains every load in flight
  auto load = [&](const signed char* plane, int grp_, int m, i32x4 (&dst)[KB]) {
#pragma unroll
    for (int u = 0; u < KB; ++u)
      dst[u] = __builtin_nontemporal_load(reinterpret_cast<const i32x4*>(plane + frag_off(grp_, min(m + u, DS - 1))));
  };
  i32x4 hA[KB], hB[KB], lA[KB], lB[KB];
  if (wid < ngroups) {
    load(hi, wid, 0, hA);
    load(lo, wid, 0, lA);
  }

  for (int round = 0; round < nrounds; ++round) {
    const int grp = round * NWV + wid;
    if (grp < ngroups) {
      const int gbase = r0 + grp * 16;
      // the rows' (s_r, b_r) are read here, ahead of the next batches: a global load issued
      // after them would make the epilogue's wait drain every row load in flight
      float2 rmv[4];
#pragma unroll
      for (int r = 0; r < 4; ++r)
        rmv[r] = *reinterpret_cast<const float2*>(rmeta + 2 * (size_t)min(gbase + 4 * g + r, r1 - 1));
      i32x4 acc_hh[MAXQ / QT], acc_lh[MAXQ / QT], acc_hl[MAXQ / QT], acc_ll[MAXQ / QT];
#pragma unroll
      for (int t = 0; t < MAXQ / QT; ++t) {
        acc_hh[t] = i32x4{0, 0, 0, 0};
        acc_lh[t] = i32x4{0, 0, 0, 0};
        acc_hl[t] = i32x4{0, 0, 0, 0};
        acc_ll[t] = i32x4{0, 0, 0, 0};
      }
      auto compute = [&](const i32x4 (&ah)[KB], const i32x4 (&al)[KB], int m) {
#pragma unroll
        for (int u = 0; u < KB; ++u) {
          if (m + u >= DS) break;
#pragma unroll
          for (int t = 0; t < MAXQ / QT; ++t) {
            if (t < NQT) {
              const size_t qo = (size_t)(t * QT + col) * QLD + 64 * (m + u) + 16 * g;
              const i32x4 bh = *reinterpret_cast<const i32x4*>(qh + qo);
              const i32x4 bl = *reinterpret_cast<const i32x4*>(ql + qo);
              acc_hh[t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(ah[u], bh, acc_hh[t], 0, 0, 0);
              acc_lh[t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(ah[u], bl, acc_lh[t], 0, 0, 0);
              acc_hl[t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(al[u], bh, acc_hl[t], 0, 0, 0);
              acc_ll[t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(al[u], bl, acc_ll[t], 0, 0, 0);
            }
          }
        }
      };
      for (int m = 0; m < DS; m += 2 * KB) {
        if (m + KB < DS) {
          load(hi, grp, m + KB, hB);
          load(lo, grp, m + KB, lB);
        }
        compute(hA, lA, m);
        if (m + 2 * KB < DS) {
          load(hi, grp, m + 2 * KB, hA);
          load(lo, grp, m + 2 * KB, lA);
        } else if (grp + NWV < ngroups) {  // the next group's first batch stays in flight
          load(hi, grp + NWV, 0, hA);
          load(lo, grp + NWV, 0, lA);
        }
        if (m + KB < DS) compute(hB, lB, m + KB);
      }
      // lane holds rows gbase + 4g + r for queries t*16 + col
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = gbase + 4 * g + r;
        if (row >= r1) continue;
        const float2 rm = rmv[r];
#pragma unroll
        for (int t = 0; t < MAXQ / QT; ++t) {
          const int q = t * QT + col;
          if (t >= NQT || q >= Q) continue;
          const float U = exact_score(acc_hh[t][r], acc_hl[t][r], acc_lh[t][r], acc_ll[t][r], rm.x, st.sq[q]);
          if (!(U > st.theta[q])) {
            if (U > st.tauL[q]) st.dropped[q] = 1;  // refused for capacity, not by the k-th bound
            continue;
          }
          if (row_prio[row] < st.minp[q]) continue;
          if ((row_tags[row] & st.qtag[q]) != st.qtag[q]) continue;
          const float ex = row_exp[row];
          if (ex != 0.f && !(ex > now)) continue;
          const int pos = atomicAdd(&st.cnt[q], 1);
          if (pos < CAND) {
            my_u[q * CAND + pos] = U;
            my_l[q * CAND + pos] = U;
            my_r[q * CAND + pos] = row;
          }
          if (pos == CAND - NWV * 16) need[round & 1] = 1;  // a buffer must absorb a round
        }
      }
    }
    __syncthreads();
    if (need[round & 1]) {
      __syncthreads();
      if (threadIdx.x == 0) need[round & 1] = 0;
      for (int q = wid; q < Q; q += NWV)
        if (st.cnt[q] > C) compact(my_u + q * CAND, my_l + q * CAND, my_r + q * CAND, st, q, K);
    }
    __syncthreads();
  }
  for (int q = wid; q < Q; q += NWV) {
    const size_t o = ((size_t)q * nwg + wg) * C;
    compact(my_u + q * CAND, my_l + q * CAND, my_r + q * CAND, st, q, K, out_u + o, out_l + o, out_r + o);
    if (lane == 0) out_drop[(size_t)q * nwg + wg] = st.dropped[q] ? st.cap[q] : -INFINITY;
  }
}

// Stage 1, the bound scan (profiles/r6_q16_stage1.md). 8 waves, two per SIMD (the 32x32 accumulators of 64 queries
// and two 4-k-step batches need ~170 registers); a wave owns 32-row groups and runs
// v_mfma_i32_32x32x32_i8 (rows x 32 queries): per byte of index it reads half the LDS query
// fragments of the 16x16x64 form (4 KiB per KiB of rows instead of 8) at the same MFMA cycles.
// The A fragments come straight from the 16-row fragment-major planes: lane (r = l & 31,
// h = l >> 5) of k-half kh of k-step s takes row tile 2G + r/16, lane position 16 (2 kh + h) +
// r % 16 -- 16 B, in 256-B runs. The group streams in batches of 4 k-steps, double-buffered, both of
// the next group's first batches in flight over the epilogue. Everything that decides what stays in
// flight is static: the k-step count is a template constant (queries zero-padded to DSC*64
// dims and whole tiles, loads past D clamped), the row loads are unconditional (clamped to the
// slice's last tile), the load batches are pinned by sched_barrier, and waves go on by themselves, without a
// barrier a round -- a branchy load block, a fenced __syncthreads, a load from scratch memory or loads left to the scheduler
// each made the wait-count pass drain the row loads in flight (the first form: 3.2 TB/s).
// Bound by the row stream: 64 queries of 4M rows, 938 -> 731 us at 1,024 dimensions (4.4 -> 5.6 TB/s; 700 if no bound ever
// reached its query's threshold), 64 of 131,000 rows 300 -> 87.
// Candidate stores are made visible by a full barrier only before a compaction, which a wave asks for when it finds a
// buffer at LIM or beyond. Until all have come, each of the others finishes at most the group it is in: LIM + 8 x 32 entries.
// Compacting early (two lists' worth) keeps the thresholds tight, and so the admissions few, now that a compaction costs a
// microsecond.
constexpr int LIM = 2 * C;
// Slices share what they know: after rounds 0, 7, 15, 31, .. each publishes the best L it has admitted per query. The K-th
// best of those is the L of K different rows, so it bounds the answer as tauL does, from the rows of all slices instead of
// one: of 4M rows, a slice then admits a row or two a query after the second round instead of some 260. In round 1 every
// slice works it out for all queries; later one slice a query, for all to read a round after (for all in each: 18 us a time).
__device__ __forceinline__ bool publishes(int round) { return round == 0 || (round >= 7 && ((round + 1) & round) == 0); }
__global__ void clear_kernel(uint32_t* p, int n) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) p[i] = 0;
}
// `pub` [Q][slices] and [Q], cleared before the launch; null: slices of one round, which have no use for it.
// FULL: D is DSC * 64. NTQ: tiles of 32 queries, one of which takes half the products and LDS reads (8 queries of 4M rows, 1,024
// dimensions: 746 us with two, 728).
template <int DSC, bool FULL, int NTQ>
__global__ __launch_bounds__(512) void stage1_bound_kernel(
    float* __restrict__ out_u, float* __restrict__ out_l, int* __restrict__ out_r, float* __restrict__ out_drop,
    float* __restrict__ cand_u, float* __restrict__ cand_l, int* __restrict__ cand_r,
    const signed char* __restrict__ qv, const float* __restrict__ qmeta, const signed char* __restrict__ hi,
    const float* __restrict__ rmeta, int Q, int N, int D, int K, const int* __restrict__ row_prio,
    const uint64_t* __restrict__ row_tags, const float* __restrict__ row_exp, const int* __restrict__ q_minp,
    const uint64_t* __restrict__ q_tags, float now, uint32_t* pub) {
  constexpr int TH = 512, NWV = TH / 64, KB = DSC >= 8 ? 4 : 2, ROWS = 32 * NTQ;
  constexpr int QLD = DSC * 64 + 16;  // padded LDS row (bytes)
  static_assert(DSC % (2 * KB) == 0, "k-steps in whole batch pairs");
  typedef int i32x16 __attribute__((ext_vector_type(16)));
  extern __shared__ __attribute__((aligned(16))) char smem[];
  signed char* qh = reinterpret_cast<signed char*>(smem);  // [ROWS][QLD]
  signed char* ql = qh + (size_t)ROWS * QLD;                // [ROWS][QLD]
  QState& st = *reinterpret_cast<QState*>(ql + (size_t)ROWS * QLD);
  int* need = reinterpret_cast<int*>(&st + 1);  // [0] some query's buffer must be compacted, [1] waves that are done
  // [NWV][32] per group row: (s_r, b_r), then the filter words (priority, expiry, tags)
  float2* rm_lds = reinterpret_cast<float2*>(need + 4);
  int* pr_lds = reinterpret_cast<int*>(rm_lds + NWV * 32);
  float* ex_lds = reinterpret_cast<float*>(pr_lds + NWV * 32);
  uint64_t* tg_lds = reinterpret_cast<uint64_t*>(ex_lds + NWV * 32);
  uint32_t* first = reinterpret_cast<uint32_t*>(tg_lds + NWV * 32);  // [ROWS][65] the first round's lower bounds

  const int nwg = gridDim.x, wg = blockIdx.x;
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lr = lane & 31, lh = lane >> 5;
  const int DS = FULL ? DSC : D / 64;
  uint32_t* tau = pub + (size_t)Q * nwg;  // [Q] K-th best bounds over the slices
  for (int v = threadIdx.x; v < ROWS * 2 * (DSC * 4); v += TH) {
    const int r = v / (2 * DSC * 4), rem = v % (2 * DSC * 4);
    const int plane = rem / (DSC * 4), c16 = (rem % (DSC * 4)) * 16;
    i32x4 x = i32x4{0, 0, 0, 0};
    if (r < Q && c16 < D) x = *reinterpret_cast<const i32x4*>(qv + ((size_t)r * 2 + plane) * D + c16);
    *reinterpret_cast<i32x4*>((plane ? ql : qh) + (size_t)r * QLD + c16) = x;
  }
  if (threadIdx.x < MAXQ) {
    const int q = threadIdx.x;
    st.cnt[q] = 0;
    st.theta[q] = -INFINITY;
    st.cap[q] = -INFINITY;
    st.tauL[q] = -INFINITY;
    st.dropped[q] = 0;
    st.top[q] = 0;
    st.minp[q] = q < Q ? q_minp[q] : 0x7fffffff;
    st.qtag[q] = q < Q ? q_tags[q] : 0ull;
    st.sq[q] = q < Q ? qmeta[2 * q] : 0.f;
    st.cq[q] = q < Q ? qmeta[2 * q + 1] : 0.f;
  }
  if (threadIdx.x < 2) need[threadIdx.x] = 0;
  __syncthreads();

  float* my_u = cand_u + (size_t)wg * MAXQ * CAND;
  float* my_l = cand_l + (size_t)wg * MAXQ * CAND;
  int* my_r = cand_r + (size_t)wg * MAXQ * CAND;
  const int per = ((N + nwg - 1) / nwg + 31) / 32 * 32;
  const int r0 = wg * per, r1 = min(N, r0 + per);
  const int ngroups = (max(0, r1 - r0) + 31) / 32;
  if (ngroups > 0) {  // workgroup-uniform
    const int nrounds = (ngroups + NWV - 1) / NWV;
    const int last_tile = (r1 - 1) >> 4;
    static_assert(LIM + NWV * 32 <= CAND, "a buffer must absorb a round");
    // this lane's two 16-B A pieces (k-halves) of k-step m + u, group grp_: a base that the wave shares and 32 bits of the
    // lane's own, so that no addresses are kept in registers
    auto load = [&](int grp_, int m, i32x4 (&dst)[KB][2]) {
      const int tile = (r0 >> 4) + 2 * min(grp_, ngroups - 1);
      const signed char* base = hi + (size_t)tile * DS * 1024;
      const unsigned own = (tile < last_tile && lr > 15 ? DS * 1024 : 0) + (lr & 15) * 16 + lh * 256;
#pragma unroll
      for (int u = 0; u < KB; ++u)
#pragma unroll
        for (int kh = 0; kh < 2; ++kh)
          dst[u][kh] = __builtin_nontemporal_load(reinterpret_cast<const i32x4*>(base + min(m + u, DS - 1) * 1024 + kh * 512 + own));
    };
    // (s_r, b_r) and the filter words of row gbase + lr of a group, issued ahead of its batches and of the last ones of the
    // group before: the epilogue reads them back from this wave's LDS slot (16 B per 1-KiB row)
    float2 rm_next;
    int pr_next;
    float ex_next;
    uint64_t tg_next;
    auto load_words = [&](int grp_) {
      const int rowc = max(0, min(r0 + grp_ * 32 + lr, r1 - 1));
      rm_next = *reinterpret_cast<const float2*>(rmeta + 2 * (size_t)rowc);
      pr_next = row_prio[rowc];
      ex_next = row_exp[rowc];
      tg_next = row_tags[rowc];
    };
    auto lds_barrier = [] {  // the row loads stay in flight across it
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
    };
    auto flag = [&](int i) {
      return __builtin_amdgcn_readfirstlane(__hip_atomic_load(need + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP));
    };
    // Every wave that finds the flag set comes here, and the barrier holds it until all have.
    auto compact_all = [&] {
      __syncthreads();  // candidate stores complete and visible
      if (threadIdx.x == 0) need[0] = 0;
      for (int q = wid; q < Q; q += NWV)  // (those that would be due soon with them)
        if (st.cnt[q] > C + C / 2) compact(my_u + q * CAND, my_l + q * CAND, my_r + q * CAND, st, q, K);
      __syncthreads();
    };
    // the K-th best bound that the slices have published for a query (a few 1e-4 below it), 0: fewer than K have one
    auto kth_published = [&](int q) {
      constexpr int PER = MAX_WG / 64;
      uint32_t key[PER];
      int have = 0, own = lane;
      asm volatile("" : "+v"(own));  // (no addresses from before the loop)
#pragma unroll
      for (int i = 0; i < PER; ++i) {
        const int w = i * 64 + own;
        key[i] = w < nwg ? __hip_atomic_load(pub + q * nwg + w, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0;
      }
#pragma unroll
      for (int i = 0; i < PER; ++i) have += __popcll(__ballot(key[i] != 0));
      return have < K ? 0u : wave_select_floor<13>(key, K);
    };
    auto raise = [&](int q, uint32_t k) {
      if (k && key_value(k) > st.tauL[q]) {
        st.tauL[q] = key_value(k);
        st.theta[q] = fmaxf(st.cap[q], key_value(k));
      }
    };
    // one round; X and Y hold the group's first two batches on entry and the next group's on exit
    auto body = [&](int round, i32x4 (&X)[KB][2], i32x4 (&Y)[KB][2]) {
      const int grp = round * NWV + wid, next = grp + NWV;
      const int gbase = r0 + grp * 32;
      i32x16 acc_hh[NTQ], acc_lh[NTQ];
#pragma unroll
      for (int t = 0; t < NTQ; ++t)
#pragma unroll
        for (int j = 0; j < 16; ++j) {
          acc_hh[t][j] = 0;
          acc_lh[t][j] = 0;
        }
      auto compute = [&](const i32x4 (&ah)[KB][2], int m) {
#pragma unroll
        for (int u = 0; u < KB; ++u) {
#pragma unroll
          for (int kh = 0; kh < 2; ++kh)
#pragma unroll
            for (int t = 0; t < NTQ; ++t) {
              const int qo = (32 * t + lr) * QLD + 64 * (m + u) + 32 * kh + 16 * lh;
              const i32x4 bh = *reinterpret_cast<const i32x4*>(qh + qo);
              const i32x4 bl = *reinterpret_cast<const i32x4*>(ql + qo);
              acc_hh[t] = __builtin_amdgcn_mfma_i32_32x32x32_i8(ah[u][kh], bh, acc_hh[t], 0, 0, 0);
              acc_lh[t] = __builtin_amdgcn_mfma_i32_32x32x32_i8(ah[u][kh], bl, acc_lh[t], 0, 0, 0);
            }
        }
      };
      // sched_barrier pins each batch's loads where they are issued: left to the scheduler they
      // sink next to their first use and only ~1 load per wave stays in flight
      // double-buffered batches, both of the next group in flight over the epilogue (a third buffer, two batches ahead,
      // spilled registers at 64 queries)
#pragma unroll
      for (int m = 0; m < DSC; m += 2 * KB) {
        const bool more = m + 2 * KB < DSC;
        __builtin_amdgcn_sched_barrier(0);
        compute(X, m);
        __builtin_amdgcn_sched_barrier(0);
        if (m == 0 && lh == 0) {  // the words of this group, older than X
          rm_lds[wid * 32 + lr] = rm_next;
          pr_lds[wid * 32 + lr] = pr_next;
          ex_lds[wid * 32 + lr] = ex_next;
          tg_lds[wid * 32 + lr] = tg_next;
        }
        if (!more) load_words(next);
        load(more ? grp : next, more ? m + 2 * KB : 0, X);
        __builtin_amdgcn_sched_barrier(0);
        compute(Y, m + KB);
        __builtin_amdgcn_sched_barrier(0);
        load(more ? grp : next, more ? m + 3 * KB : KB, Y);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (pub && round == 1) {
        for (int q = wid; q < Q; q += NWV) raise(q, kth_published(q));
        lds_barrier();  // no wave goes on without the first bounds
      } else if (pub && round > 1) {
        if (publishes(round - 1) && wid == 0 && wg < Q) {
          const uint32_t k = kth_published(wg);
          if (lane == 0) __hip_atomic_fetch_max(tau + wg, k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        if (round > 2 && publishes(round - 2) && wid == 0 && lane < Q)
          raise(lane, __hip_atomic_load(tau + lane, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
      }
      if (round == 0) {
        // The first groups show what their best rows reach before any is admitted: of every four rows the best lower bound
        // that passes the query's filters, 64 of 256 rows, whose K-th best the query begins with. (With all 256 rows
        // admitted for every query, 64 queries of 131,000 rows took 538 us a lookup, 450 so.)
        const float2* rmw = rm_lds + wid * 32;
#pragma unroll
        for (int t = 0; t < NTQ; ++t) {
          const int q = 32 * t + lr, minp = st.minp[q];
          const uint64_t want = st.qtag[q];
          const float sq = st.sq[q], cq = st.cq[q] * 1.0001f;
#pragma unroll
          for (int f = 0; f < 4; ++f) {
            uint32_t best = 0;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const int ri = r + 8 * f + 4 * lh;
              const float2 rm = rmw[ri];
              const float ex = ex_lds[wid * 32 + ri];
              const float sc = fmaf((float)acc_hh[t][4 * f + r], 65536.f, (float)acc_lh[t][4 * f + r] * 256.f) * (rm.x * sq);
              const float e = fmaf(rm.y, cq, 1e-6f);
              if (gbase + ri < r1 && (ex == 0.f || ex > now) && pr_lds[wid * 32 + ri] >= minp &&
                  (tg_lds[wid * 32 + ri] & want) == want && is_finite(sc - e))
                best = max(best, ord_key(sc - e));
            }
            first[q * 65 + (wid * 2 + lh) * 4 + f] = best;
          }
        }
        lds_barrier();
        for (int q = wid; q < Q; q += NWV) {
          const uint32_t key[1] = {first[q * 65 + lane]};
          if (__popcll(__ballot(key[0] != 0)) >= K) raise(q, wave_select_floor<13>(key, K));
        }
        lds_barrier();
      }
      if (grp < ngroups) {
        // lane holds queries 32 t + lr, rows gbase + (j & 3) + 8 (j >> 2) + 4 lh (j = 0..15).
        // First only whether any lane's bound reaches its query's k-th lower bound tauL (theta is no lower): seven
        // operations a pair, and once the bounds are tight most groups end there. (All of it for every group took 230 of
        // the 940 us of 4M rows and 64 queries, as the waves' loads ran dry meanwhile.) Then the pairs (t, j) that some lane
        // reaches, each behind a branch of the wave's: unrolled without, they do not fit the registers.
        const int nrow = r1 - gbase;  // rows ri < nrow are in the slice
        const float2* rmw = rm_lds + wid * 32;  // written by this wave (LDS order holds)
        float tl[NTQ], sqv[NTQ], cqv[NTQ];
#pragma unroll
        for (int t = 0; t < NTQ; ++t) {
          const int q = 32 * t + lr;
          tl[t] = q < Q ? st.tauL[q] : INFINITY;
          sqv[t] = st.sq[q];
          cqv[t] = st.cq[q] * 1.0001f;
        }
        unsigned reach = 0;  // bit 16 t + j
#pragma unroll
        for (int j = 0; j < 16; ++j) {
          const float2 rm = rmw[(j & 3) + 8 * (j >> 2) + 4 * lh];
#pragma unroll
          for (int t = 0; t < NTQ; ++t) {
            const float U = fmaf(fmaf((float)acc_hh[t][j], 256.f, (float)acc_lh[t][j]), rm.x * (256.f * sqv[t]),
                                 fmaf(rm.y, cqv[t], 2e-6f));  // (a margin over the bounds below)
            if (__any(U > tl[t])) reach |= 1u << (16 * t + j);
          }
        }
        if (reach) {
          // (what this path reads and writes is named here: addresses kept in registers from before the loop go to scratch
          // memory, and each load from there waits for all row loads in flight)
          int own = lr, half = 4 * lh + wid * 32, at = wg * (MAXQ * CAND);
          asm volatile("" : "+v"(own), "+v"(half), "+s"(at));
#pragma unroll
          for (int t = 0; t < NTQ; ++t) {
            const int q = 32 * t + own;
#pragma unroll
            for (int j = 0; j < 16; ++j) {
              if (!((reach >> (16 * t + j)) & 1u)) continue;
              const int rw = (j & 3) + 8 * (j >> 2) + half, ri = rw - wid * 32;
              const float2 rm = rm_lds[rw];
              const float sc = fmaf((float)acc_hh[t][j], 65536.f, (float)acc_lh[t][j] * 256.f) * (rm.x * sqv[t]);
              const float e = fmaf(rm.y, cqv[t], 1e-6f);  // margin: fp32 rounding of sc and e
              if (ri >= nrow || !(sc + e > tl[t])) continue;
              if (!(sc + e > st.theta[q])) {  // refused for capacity, not by the k-th bound
                st.dropped[q] = 1;
                continue;
              }
              const float ex = ex_lds[rw];
              if (pr_lds[rw] < st.minp[q] || (tg_lds[rw] & st.qtag[q]) != st.qtag[q] ||
                  (ex != 0.f && !(ex > now)))
                continue;
              const int pos = atomicAdd(&st.cnt[q], 1);
              atomicMax(&st.top[q], ord_key(sc - e));
              if (pos < CAND) {
                const unsigned to = at + q * CAND + pos;
                cand_u[to] = sc + e;
                cand_l[to] = sc - e;
                cand_r[to] = gbase + ri;
              }
              if (pos >= LIM) __hip_atomic_store(need, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            }
          }
        }
      }
      // (LDS only: the row loads stay in flight)
      // Round 1 begins with a barrier of its own: a wave that waits there must not meet others in a compaction's. So no wave
      // leaves round 0 before all have admitted its rows, and all find the same flag. Later rounds have no other barrier.
      if (round == 0) lds_barrier();
      if (flag(0)) compact_all();
      if (pub && publishes(round) && threadIdx.x < Q)
        __hip_atomic_store(pub + threadIdx.x * nwg + wg, st.top[threadIdx.x], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    i32x4 bA[KB][2], bB[KB][2];
    load_words(wid);
    load(wid, 0, bA);
    load(wid, KB, bB);
    for (int round = 0; round < nrounds; ++round) body(round, bA, bB);
    // done: the others may still ask for a compaction
    if (lane == 0) __hip_atomic_fetch_add(need + 1, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    for (;;) {
      const int done = flag(1);
      if (flag(0)) compact_all();
      else if (done == NWV) break;
      else __builtin_amdgcn_s_sleep(4);
    }
  }
  __syncthreads();
  // The lists. Buffers of at most C entries, all of a wave's queries at once, so that their loads wait together.
  constexpr int QW = ROWS / NWV;
  int most = 0;
#pragma unroll
  for (int i = 0; i < QW; ++i) most = max(most, wid + NWV * i < Q ? st.cnt[wid + NWV * i] : 0);
  if (most <= C) {
    float u[QW], l[QW];
    int row[QW];
#pragma unroll
    for (int i = 0; i < QW; ++i) {
      const int q = min(wid + NWV * i, Q - 1), at = q * CAND + max(0, min(lane, st.cnt[q] - 1));
      const bool ok = wid + NWV * i < Q && lane < st.cnt[q];
      u[i] = ok ? my_u[at] : -INFINITY;
      l[i] = ok ? my_l[at] : -INFINITY;
      row[i] = ok ? my_r[at] : -1;
    }
#pragma unroll
    for (int i = 0; i < QW; ++i) {
      const int q = wid + NWV * i;
      if (q >= Q) break;
      const bool keep = row[i] >= 0 && !(u[i] < st.tauL[q]);  // (entries that the bound has overtaken go)
      const unsigned long long kept = __ballot(keep), rest = ~kept;
      const size_t o = ((size_t)q * nwg + wg) * C + (keep ? rank_in(kept) : (int)__popcll(kept) + rank_in(rest));
      out_u[o] = keep ? u[i] : -INFINITY;
      out_l[o] = keep ? l[i] : -INFINITY;
      out_r[o] = keep ? row[i] : -1;
      if (lane == 0) out_drop[(size_t)q * nwg + wg] = st.dropped[q] ? st.cap[q] : -INFINITY;
    }
    return;
  }
  for (int q = wid; q < Q; q += NWV) {
    const size_t o = ((size_t)q * nwg + wg) * C;
    compact(my_u + q * CAND, my_l + q * CAND, my_r + q * CAND, st, q, K, out_u + o, out_l + o, out_r + o);
    if (lane == 0) out_drop[(size_t)q * nwg + wg] = st.dropped[q] ? st.cap[q] : -INFINITY;
  }
}

// Stage 2: one workgroup per query (see the header), 16 list entries a thread in registers. EXACT: the lists hold exact
// scores. Both selections go by bits (topk_select.h); with sorted buffers the launch took 130 us for 16,384 entries.
template <bool EXACT>
__global__ __launch_bounds__(THREADS) void stage2_kernel(
    float* __restrict__ out_s, int* __restrict__ out_rows, int* __restrict__ unsafe,
    const float* __restrict__ lu, const float* __restrict__ ll, const int* __restrict__ lr,
    const float* __restrict__ ldrop, int nwg, const signed char* __restrict__ qv,
    const float* __restrict__ qmeta, const signed char* __restrict__ hi, const signed char* __restrict__ lo,
    const float* __restrict__ rmeta, int D, int K) {
  constexpr int PER = MAX_WG * C / THREADS;  // entries a thread
  constexpr int CL = 8 * THREADS;            // re-ranked entries at a time
  constexpr int RR = CL / THREADS + 1;
  constexpr int MOVED = 4;
  static_assert(MOVED <= PER && MOVED * THREADS <= CL, "entries that move have room");
  __shared__ int red[2 * NW];
  __shared__ Selection sel;
  __shared__ int crow[EXACT ? 1 : CL + MAXK];
  __shared__ uint32_t ckey[EXACT ? 1 : CL + MAXK];
  __shared__ float best_s[MAXK];
  __shared__ int best_r[MAXK];
  __shared__ int ncand;
  __shared__ uint32_t picked;
  const int q = blockIdx.x;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int total = nwg * C;
  const float* u = lu + (size_t)q * total;
  const float* l = ll + (size_t)q * total;
  const int* r = lr + (size_t)q * total;
  float* os = out_s + (size_t)q * K;
  int* orow = out_rows + (size_t)q * K;
  // ---- A: tau = the K-th best lower bound over every slice's list (no bound with fewer than K entries)
  uint32_t key[PER], ukey[PER];
  int row[PER], have = 0, per = (total + THREADS - 1) / THREADS;  // a thread's first `per` may hold an entry
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int e = i * THREADS + threadIdx.x;
    row[i] = -1;
    if (i >= per) continue;
    row[i] = e < total ? r[e] : -1;
    have += __popcll(__ballot(row[i] >= 0));
  }
  // what C and B read is on its way with the lists
  const float sq = qmeta[2 * q];
  const int DS = D / 64;
  // a lane holds 16 dimensions of a row: k-step lane / 4, lane group lane % 4 of it (D <= 1024)
  const bool on = !EXACT && lane < DS * 4;
  i32x4 qa = i32x4{0, 0, 0, 0}, qb = qa;
  if (on) {
    const signed char* qp = qv + (size_t)q * 2 * D + 16 * lane;
    qa = *reinterpret_cast<const i32x4*>(qp);
    qb = *reinterpret_cast<const i32x4*>(qp + D);
  }
  const uint32_t none = ord_key(-INFINITY);
  uint32_t drop = none;
  if (!EXACT)
    for (int i = threadIdx.x; i < nwg; i += THREADS) drop = max(drop, ord_key(ldrop[(size_t)q * nwg + i]));
  if (threadIdx.x == 0) ncand = 0;
  __syncthreads();
  int at = 0;
  if (lane == 0) at = atomicAdd(&ncand, have);
  at = __shfl(at, 0, 64);
  __syncthreads();
  have = ncand;
  uint32_t tau = 1;
  if (EXACT || have > MOVED * THREADS) {
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int e = min(i * THREADS + (int)threadIdx.x, total - 1);
      key[i] = row[i] >= 0 ? ord_key(l[e]) : 0;
      ukey[i] = !EXACT && row[i] >= 0 ? ord_key(u[e]) : 0;
    }
    if (have >= K) tau = block_select<PER, NW>(key, K, red);
  } else {
    // Slices that share their bounds list a row or two each, and few slices a dozen: such entries move together, up to
    // MOVED a thread, which one wave selects from where there is one, and their bounds one load instead of 16 in turn (64 queries of 4M
    // rows: 67 -> 53 us; 3 of 20,011, 1,204 entries in 79 lists, where those of more than 1,024 stayed, 23 -> 18).
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      if (i >= per) {
        ukey[i] = 0;
        continue;
      }
      const unsigned long long m = __ballot(row[i] >= 0);
      const int p = at + rank_in(m);
      if (row[i] >= 0) { crow[p] = row[i]; ckey[p] = i * THREADS + threadIdx.x; }
      at += __popcll(m);
      row[i] = -1;
      ukey[i] = 0;
    }
    __syncthreads();
    per = (have + THREADS - 1) / THREADS;
    uint32_t low[MOVED];
#pragma unroll
    for (int i = 0; i < MOVED; ++i) {
      const int at = i * THREADS + threadIdx.x;
      low[i] = 0;
      if (at < have) {
        const int e = ckey[at];
        row[i] = crow[at];
        ukey[i] = ord_key(u[e]);
        low[i] = ord_key(l[e]);
      }
    }
    if (per > 1) {
      if (have >= K) tau = block_select<MOVED, NW>(low, K, red);
    } else {
      if ((int)threadIdx.x < have) ckey[threadIdx.x] = low[0];  // (each reads its own before)
      __syncthreads();
      if (have >= K) tau = lds_select(ckey, have, K, &picked);
    }
  }
  // ---- B: a slice that refused a row for capacity at a level >= tau may have lost a top-k row
  if (EXACT) {  // the lists hold exact scores
    if (threadIdx.x == 0) unsafe[q] = 0;
    write_best(key, row, tau, K, sel, os, orow);
    return;
  }
  const bool lost = __syncthreads_or(drop > none && drop >= tau);
  if (threadIdx.x == 0) unsafe[q] = lost;
  // ---- C: re-rank every listed row whose upper bound reaches tau, exactly
  int cand = 0;
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    if (i >= per) continue;
    if (ukey[i] < tau) row[i] = -1;
    cand += __popcll(__ballot(row[i] >= 0));
  }
  if (lane == 0) red[wid] = cand;
  if (threadIdx.x == 0) ncand = 0;
  __syncthreads();
  cand = 0;
#pragma unroll
  for (int w = 0; w < NW; ++w) cand += red[w];
  int kept = 0;  // best entries so far, ahead of the next ones in crow / ckey
  const int step = cand <= CL ? PER : CL / THREADS;
#pragma unroll 1
  for (int part = 0; part < PER; part += step) {
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      if (i < part || i >= part + step || i >= per) continue;
      const unsigned long long m = __ballot(row[i] >= 0);
      int at = 0;
      if (lane == 0 && m) at = atomicAdd(&ncand, (int)__popcll(m));
      at = __shfl(at, 0, 64) + kept + rank_in(m);
      if (row[i] >= 0) crow[at] = row[i];
    }
    __syncthreads();
    const int n = kept + ncand;
    constexpr int RB = 4;  // rows a wave reads at once: the launch is a chain of such reads
    for (int j0 = kept + wid * RB; j0 < n; j0 += NW * RB) {
      i32x4 a[RB], b[RB];
      int rw[RB];
      float sr[RB];
#pragma unroll
      for (int k = 0; k < RB; ++k) {
        rw[k] = crow[min(j0 + k, n - 1)];
        sr[k] = rmeta[2 * (size_t)rw[k]];
        if (on) {
          const size_t off = (((size_t)(rw[k] >> 4) * DS + (lane >> 2)) * 64 + 16 * (lane & 3) + (rw[k] & 15)) * 16;
          a[k] = *reinterpret_cast<const i32x4*>(hi + off);
          b[k] = *reinterpret_cast<const i32x4*>(lo + off);
        } else {
          a[k] = b[k] = i32x4{0, 0, 0, 0};
        }
      }
#pragma unroll
      for (int k = 0; k < RB; ++k) {
        int hh = 0, hl = 0, lh = 0, lls = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          hh = __builtin_amdgcn_sdot4(qa[e], a[k][e], hh, false);
          hl = __builtin_amdgcn_sdot4(qa[e], b[k][e], hl, false);
          lh = __builtin_amdgcn_sdot4(qb[e], a[k][e], lh, false);
          lls = __builtin_amdgcn_sdot4(qb[e], b[k][e], lls, false);
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
          hh += __shfl_xor(hh, o, 64);
          hl += __shfl_xor(hl, o, 64);
          lh += __shfl_xor(lh, o, 64);
          lls += __shfl_xor(lls, o, 64);
        }
        if (lane == 0 && j0 + k < n) ckey[j0 + k] = ord_key(exact_score(hh, hl, lh, lls, sr[k], sq));
      }
    }
    __syncthreads();
    const bool last = part + step >= PER;
    float* bs = last ? os : best_s;
    int* br = last ? orow : best_r;
    if (n <= 64) {
      write_best_few(ckey, crow, n, K, bs, br);
    } else if (n <= THREADS) {
      const uint32_t ck[1] = {(int)threadIdx.x < n ? ckey[threadIdx.x] : 0};
      const int cr[1] = {(int)threadIdx.x < n ? crow[threadIdx.x] : -1};
      write_best(ck, cr, n > K ? lds_select(ckey, n, K, &picked) : 1, K, sel, bs, br);
    } else {
      uint32_t ck[RR];
      int cr[RR];
#pragma unroll
      for (int i = 0; i < RR; ++i) {
        const int e = i * THREADS + threadIdx.x;
        ck[i] = e < n ? ckey[e] : 0;
        cr[i] = e < n ? crow[e] : -1;
      }
      write_best(ck, cr, block_select<RR, NW>(ck, K, red), K, sel, bs, br);
    }
    if (!last) {
      __syncthreads();
      kept = min(n, K);
      if (threadIdx.x < kept) {
        ckey[threadIdx.x] = ord_key(best_s[threadIdx.x]);
        crow[threadIdx.x] = best_r[threadIdx.x];
      }
      if (threadIdx.x == 0) ncand = 0;
      __syncthreads();
    }
  }
}

// ---- queries ------------------------------------------------------------------------------------------
// x / y rounded as IEEE does, whatever the compiler may do with a float division (fast-math): the double quotient
// rounds to the same float, and the empty asm keeps the two steps apart, and a rounding to 16 bits behind them.
__device__ __forceinline__ float div_rn(float x, float y) {
  double d = (double)x / (double)y;
  asm volatile("" : "+v"(d));
  float f = (float)d;
  asm volatile("" : "+v"(f));
  return f;
}

// One workgroup a query: normalised (if asked), then rounded to bf16, or to 16-bit fixed point as q16_quantize does:
// s_q = max|x| / 32512, v = round(x / s_q) = 256 qh + ql, c_q = s_q ||v||_2 (a hair above). NaN goes where torch's
// operations take it: a norm or a maximum of a query that holds one is one (s_q is then 1), and in v it is 0. One launch in
// place of the 28 elementwise ones that took as long as the search of a small index. x is read once, of up to PQ * 256
// dimensions, as it may lie in the host's memory; so may the query's filters (minp, tags), which go to fminp and ftags.
constexpr int PQ = 8;
__global__ __launch_bounds__(256) void prepare_kernel(const float* __restrict__ x, int D, int normalize, bf16* __restrict__ out,
                                                      signed char* __restrict__ qv, float* __restrict__ qmeta,
                                                      const int* __restrict__ minp, const uint64_t* __restrict__ tags,
                                                      int* __restrict__ fminp, uint64_t* __restrict__ ftags) {
  __shared__ double red[4];
  __shared__ uint32_t redm[4];
  const int q = blockIdx.x, lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  x += (size_t)q * D;
  if (fminp && threadIdx.x == 0) {
    fminp[q] = minp[q];
    ftags[q] = tags[q];
  }
  float xs[PQ];
#pragma unroll
  for (int k = 0; k < PQ; ++k) xs[k] = k * 256 + (int)threadIdx.x < D ? x[k * 256 + threadIdx.x] : 0.f;
  auto each = [&](auto f) {  // f(dimension, value) of this thread's dimensions
#pragma unroll
    for (int k = 0; k < PQ; ++k)
      if (k * 256 + (int)threadIdx.x < D) f(k * 256 + (int)threadIdx.x, xs[k]);
    for (int i = PQ * 256 + threadIdx.x; i < D; i += 256) f(i, x[i]);
  };
  auto sum = [&](double v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    __syncthreads();
    if (lane == 0) red[wid] = v;
    __syncthreads();
    return red[0] + red[1] + red[2] + red[3];
  };
  // (what is not finite is told by its bits: the compiler is told that there is none)
  auto size = [](float v) { return __float_as_uint(v) & 0x7fffffffu; };
  constexpr uint32_t INF = 0x7f800000u;
  float by = 1.f;
  if (normalize) {
    double ss = 0.;
    each([&](int, float v) { ss += (double)v * (double)v; });
    ss = sum(ss);
    const long long over = __double_as_longlong(ss) - 0x7ff0000000000000ll;  // the norm is infinite (0) or NaN (above)
    by = fmaxf((float)sqrt(ss), 1e-12f);
    if (over >= 0 || size(by) == INF) {  // finite values become 0 or NaN, the others NaN
      each([&](int i, float v) {
        if (out) {
          reinterpret_cast<uint16_t*>(out)[(size_t)q * D + i] = over > 0 || size(v) >= INF ? 0x7fc0 : __float_as_uint(v) >> 16 & 0x8000;
        } else {
          qv[(size_t)q * 2 * D + i] = 0;
          qv[(size_t)q * 2 * D + D + i] = 0;
        }
      });
      if (!out && threadIdx.x == 0) {
        qmeta[2 * q] = 1.f;
        qmeta[2 * q + 1] = 0.f;
      }
      return;
    }
  }
  auto at = [&](float v) { return normalize ? div_rn(v, by) : v; };
  if (out) {
    each([&](int i, float v) { out[(size_t)q * D + i] = (bf16)at(v); });
    return;
  }
  uint32_t mb = 0;  // magnitudes in their bits' order, NaN above all
  each([&](int, float v) { mb = max(mb, size(at(v))); });
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) mb = max(mb, (uint32_t)__shfl_xor((int)mb, o, 64));
  if (lane == 0) redm[wid] = mb;
  __syncthreads();
  mb = max(max(redm[0], redm[1]), max(redm[2], redm[3]));
  const float sc = mb > 0 && mb <= INF ? div_rn(__uint_as_float(mb), 32512.f) : 1.f;
  double vv = 0.;
  each([&](int i, float x) {
    const float f = rintf(div_rn(at(x), sc));
    const int v = size(f) > INF ? 0 : (int)fminf(fmaxf(f, -32512.f), 32512.f), h = (v + 128) >> 8;
    qv[(size_t)q * 2 * D + i] = (signed char)h;
    qv[(size_t)q * 2 * D + D + i] = (signed char)(v - 256 * h);
    vv += (double)v * (double)v;  // whole numbers below 2^53: exact in any order
  });
  vv = sum(vv);
  if (threadIdx.x == 0) {
    qmeta[2 * q] = sc;
    qmeta[2 * q + 1] = (float)((double)sc * sqrt(vv)) * (1.f + 1e-6f);
  }
}

}  // namespace q16
}  // namespace pa

// workspace: lists [3][Q][nwg][C] (U, L, row) + drop levels [Q][nwg] + published bounds [Q][nwg] and [Q] + per-(slice, query)
// candidate buffers [3][nwg][64][CAND]
extern "C" long long pa_q16_topk_workspace_bytes(int Q, int N) {
  const long long w = pa::q16::num_wg(N);
  return 3LL * Q * w * pa::q16::C * 4 + (2LL * w + 1) * Q * 4 + 3LL * w * pa::q16::MAXQ * pa::q16::CAND * 4;
}

// queries_q: [Q][2][D] int8 (qh, ql); qmeta [Q][2] (s_q, c_q); hi / lo: [N/16][D/64][64][16]
// int8; rmeta [N][2] (s_r, b_r). Outputs scores / rows [Q][K] and unsafe [Q] (stage-1 mode only:
// 1 = rerun this batch with exact = 1). Returns 0, -1 for an unsupported shape, or a HIP error.
extern "C" int pa_q16_topk(float* out_scores, int* out_rows, int* unsafe, void* workspace, const void* queries_q,
                           const float* qmeta, const void* hi, const void* lo, const float* rmeta, int Q, int N,
                           int D, int K, const int* row_priority, const uint64_t* row_tags,
                           const float* row_expiry, const int* q_min_priority, const uint64_t* q_tags, float now,
                           int exact, hipStream_t st) {
  using namespace pa::q16;
  if (Q <= 0) return 0;
  if (D % 64 != 0 || D > MAXD || K < 1 || K > MAXK || Q > MAXQ) return -1;
  if (N <= 0) {
    (void)hipMemsetAsync(out_rows, 0xff, (size_t)Q * K * sizeof(int), st);
    (void)hipMemsetAsync(unsafe, 0, (size_t)Q * sizeof(int), st);
    return (int)hipGetLastError();
  }
  const int nwg = num_wg(N);
  float* lu = reinterpret_cast<float*>(workspace);
  float* ll = lu + (size_t)Q * nwg * C;
  int* lr = reinterpret_cast<int*>(ll + (size_t)Q * nwg * C);
  float* ldrop = reinterpret_cast<float*>(lr + (size_t)Q * nwg * C);
  uint32_t* pub = reinterpret_cast<uint32_t*>(ldrop + (size_t)Q * nwg);
  float* cu = ldrop + 2 * (size_t)Q * nwg + Q;
  float* cl = cu + (size_t)nwg * MAXQ * CAND;
  int* cr = reinterpret_cast<int*>(cl + (size_t)nwg * MAXQ * CAND);
  const int nqt = (Q + QT - 1) / QT;
  const size_t lds = (size_t)nqt * QT * (D + 16) * 2 + sizeof(QState) + 16;
  static bool attr_set = false;
  if (!attr_set) {
#define PA_X(D) stage1_bound_kernel<D, true, 1>, stage1_bound_kernel<D, false, 1>, stage1_bound_kernel<D, true, 2>, stage1_bound_kernel<D, false, 2>
    for (auto* k : {PA_X(4), PA_X(8), PA_X(16)})
      (void)hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
#undef PA_X
    (void)hipFuncSetAttribute((const void*)stage1_exact_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    attr_set = true;
  }
  const signed char* qv = (const signed char*)queries_q;
  const signed char* h = (const signed char*)hi;
  const signed char* l = (const signed char*)lo;
  if (exact) {
    hipLaunchKernelGGL(stage1_exact_kernel, dim3(nwg), dim3(512), lds, st, lu, ll, lr, ldrop, cu, cl, cr, qv, qmeta,
                       h, l, rmeta, Q, N, D, K, row_priority, row_tags, row_expiry, q_min_priority, q_tags, now);
    hipLaunchKernelGGL(stage2_kernel<true>, dim3(Q), dim3(THREADS), 0, st, out_scores, out_rows, unsafe, lu, ll, lr,
                       ldrop, nwg, qv, qmeta, h, l, rmeta, D, K);
  } else {
    const int dsc = D <= 256 ? 4 : (D <= 512 ? 8 : 16);
    const int tiles = Q > 32 ? 2 : 1;
    const size_t ldsb = (size_t)(32 * tiles) * (dsc * 64 + 16) * 2 + sizeof(QState) + 16 + 8 * 32 * 24 + 32 * tiles * 65 * 4;
    if (N > MIN_ROWS_PER_WG * nwg) hipLaunchKernelGGL(clear_kernel, dim3(8), dim3(512), 0, st, pub, Q * (nwg + 1));
    else pub = nullptr;
    const bool full = D == dsc * 64;
#define PA_X(D) (full ? (tiles == 1 ? stage1_bound_kernel<D, true, 1> : stage1_bound_kernel<D, true, 2>)    \
                      : (tiles == 1 ? stage1_bound_kernel<D, false, 1> : stage1_bound_kernel<D, false, 2>))
    auto* bound = dsc == 4 ? PA_X(4) : dsc == 8 ? PA_X(8) : PA_X(16);
#undef PA_X
    hipLaunchKernelGGL(bound, dim3(nwg), dim3(512), ldsb, st, lu, ll, lr, ldrop, cu, cl, cr, qv, qmeta, h, rmeta, Q, N, D,
                       K, row_priority, row_tags, row_expiry, q_min_priority, q_tags, now, pub);
    hipLaunchKernelGGL(stage2_kernel<false>, dim3(Q), dim3(THREADS), 0, st, out_scores, out_rows, unsafe, lu, ll, lr,
                       ldrop, nwg, qv, qmeta, h, l, rmeta, D, K);
  }
  return (int)hipGetLastError();
}

// x fp32 [Q][D] -> bf16 [Q][D] (out), or, with out null, int8 [Q][2][D] (qv) and fp32 [Q][2] (qmeta). With fminp, the queries'
// filters minp [Q] and tags [Q] are copied to fminp and ftags.
extern "C" int pa_prepare_queries(const float* x, int Q, int D, int normalize, void* out, void* qv, float* qmeta, const int* minp,
                                  const uint64_t* tags, int* fminp, uint64_t* ftags, hipStream_t st) {
  if (Q <= 0) return 0;
  hipLaunchKernelGGL(pa::q16::prepare_kernel, dim3(Q), dim3(256), 0, st, x, D, normalize, (pa::bf16*)out, (signed char*)qv,
                     qmeta, minp, tags, fminp, ftags);
  return (int)hipGetLastError();
}
