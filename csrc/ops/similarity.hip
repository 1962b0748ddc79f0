// HBM-resident semantic index: fused filter + cosine similarity + top-k
// (backs EnhancedMemory.semantic_search,
// reference pilott/memory/enhanced_memory.py:93-131).
//
// index   [N, D] bf16, rows L2-normalised on insert (so cosine == dot)
// queries [Q, D] bf16, L2-normalised
// per-row filter metadata: priority (int32), tag bitmask (uint64), expiry (f32
// seconds, 0 = never); per-query: min priority, required tag bitmask.
// A row qualifies for query q iff prio >= minp[q] && (tags & qtags[q]) == qtags[q]
// && (expiry == 0 || expiry > now) — the reference's candidate-index semantics
// (priority index range, tag-set intersection, is_expired) evaluated in-kernel.
//
// Stage 1 (one pass over the index for up to 64 queries): each workgroup owns a
// slice of rows; its 16 waves take 16-row groups and multiply them by EVERY query
// tile with v_mfma_f32_16x16x32_bf16 — index rows stream from HBM straight into
// the A operand once (the index is stored in 16-row tiles, fragment-major:
// [N/16][D/32][64 lanes][8], so each wave load is 1 KiB contiguous instead of
// 16 rows x 64 B — half the load-path work per streamed byte), the (<= 64) queries sit in LDS as B operands, so a 205 GB
// 100M x 1024 index is read exactly once per batch of agent queries. Scores
// above a query's running threshold (and passing the filters) are appended to
// that query's candidate buffer (global workspace, per workgroup); one wave cuts a
// full buffer to its k best (topk_select.h) and raises the threshold to the k-th. Each
// slice writes its top-k. Stage 2 (one WG per query) merges the slices' lists.
#include "topk_select.h"

#include <algorithm>

namespace pa {

constexpr int SIM_CAND = 512;     // candidate buffer per (slice, query), power of two
constexpr int SIM_MAXK = 64;
constexpr int SIM_QT = 16;        // queries per MFMA tile (N = 16)
constexpr int SIM_MAXQ = 64;      // queries per pass (4 tiles resident in LDS)
constexpr int SIM_MAXD = 1024;    // LDS query capacity per query (bf16)
// A round of 16 waves x 16 rows a slice at least, 128 KB of row loads in flight per CU. Few queries of an index of which no CU
// has more than 8 waves' rows take cosine_short_kernel; with many queries their work on the first round is what they wait for,
// and the merge has more lists to read (both stages, slices of 256 rows and of 128, x 1,024: 40 queries of 5,000 rows 34.8 us and
// 41.0, 64 48.8 and 53.5, 64 of 32,768 52.5 and 60.9; 17 of 5,000, 29.1 and 27.9, are the other way round).
constexpr int SIM_ROUND = 256, SIM_SHORT = 32768, SIM_FEW_Q = 16;  // rows of a round; rows and queries of a short index
constexpr int SIM_THREADS = 4 * SIM_ROUND;
constexpr int SIM_LIM = 2 * SIM_MAXK;  // entries of a buffer between rounds; a round may admit 256 more
constexpr int SIM_KB = 8;         // k-steps per row-load batch (two batches in flight)
constexpr int SIM_MAX_WG = 256;    // one resident workgroup per CU: the threshold warm-up is paid once per CU

inline bool sim_short(int Q, int N) { return Q <= SIM_FEW_Q && N <= SIM_SHORT; }
inline int sim_short_waves(int N) { return N <= 4 * 16 * SIM_MAX_WG ? 4 : (N + 16 * SIM_MAX_WG - 1) / (16 * SIM_MAX_WG); }  // at most 8
inline int sim_num_wg(int Q, int N) {
  const int rows = sim_short(Q, N) ? 16 * sim_short_waves(N) : SIM_ROUND;
  return std::max(1, std::min(SIM_MAX_WG, (N + rows - 1) / rows));
}

// Cut query buffer `gs/gr` to its best K and raise the threshold: one wave, no barrier, about a microsecond (a bitonic sort
// by the workgroup took ten, one query after the other). os / orow: where the slice's list goes, or null to keep it.
__device__ __forceinline__ void compact_global(float* gs, int* gr, int* cnt, float* theta, int K, float* os = nullptr,
                                               int* orow = nullptr) {
  constexpr int PER = SIM_CAND / 64;
  const int lane = threadIdx.x & 63, n = min(*cnt, SIM_CAND);
  uint32_t key[PER];
  int row[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int e = i * 64 + lane;
    key[i] = e < n ? ord_key(gs[e]) : 0;
    row[i] = e < n ? gr[e] : -1;
  }
  uint32_t cut = 1;  // entries above it stay, and of those at it as many as there is room for
  int room = K, at = 0;
  if (n >= K) {
    cut = wave_select(key, K);
#pragma unroll
    for (int i = 0; i < PER; ++i) room -= __popcll(__ballot(key[i] > cut));
  }
  if (os) { gs = os; gr = orow; }
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const unsigned long long ties = __ballot(key[i] == cut);
    const bool keep = key[i] > cut || (key[i] == cut && rank_in(ties) < room);
    room -= __popcll(ties);
    const unsigned long long kept = __ballot(keep);
    if (keep) {
      const int p = at + rank_in(kept);
      gs[p] = key_value(key[i]);
      gr[p] = row[i];
    }
    at += __popcll(kept);
  }
  if (os && lane >= at && lane < K) { gs[lane] = -INFINITY; gr[lane] = -1; }
  if (lane == 0) {
    *cnt = at;
    if (at == K) *theta = key_value(cut);
  }
}

__global__ __launch_bounds__(SIM_THREADS) void cosine_stage1_kernel(
    float* __restrict__ ws_s, int* __restrict__ ws_r, float* __restrict__ cand_s, int* __restrict__ cand_r,
    const bf16* __restrict__ queries, const bf16* __restrict__ index, int Q, int N, int D, int K,
    const int* __restrict__ row_prio, const uint64_t* __restrict__ row_tags,
    const float* __restrict__ row_exp, const int* __restrict__ q_minp, const uint64_t* __restrict__ q_tags,
    float now) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int NQT = (Q + SIM_QT - 1) / SIM_QT;
  const int QLD = D + 8;  // padded LDS row: the 16 query rows of a B fragment hit distinct bank slots
  bf16* qt = reinterpret_cast<bf16*>(smem);                                     // [NQT*16][QLD]
  int* cnt = reinterpret_cast<int*>(smem + (size_t)NQT * SIM_QT * QLD * 2);      // [MAXQ]
  float* theta = reinterpret_cast<float*>(cnt + SIM_MAXQ);                    // [MAXQ]
  int* minp = reinterpret_cast<int*>(theta + SIM_MAXQ);                       // [MAXQ]
  uint64_t* qtag = reinterpret_cast<uint64_t*>(minp + SIM_MAXQ);              // [MAXQ]
  int* need = reinterpret_cast<int*>(qtag + SIM_MAXQ);  // [2] some buffer is full, by rounds in turn: a wave that is a
                                                        // round ahead must not be taken for this one's
  // [waves][16] the filter words of a group's rows (tags, priority, expiry), and [NQT*16][65] the first round's scores
  uint64_t* tg_lds = reinterpret_cast<uint64_t*>(need + 4);
  int* pr_lds = reinterpret_cast<int*>(tg_lds + SIM_THREADS / 4);
  float* ex_lds = reinterpret_cast<float*>(pr_lds + SIM_THREADS / 4);
  uint32_t* first = reinterpret_cast<uint32_t*>(ex_lds + SIM_THREADS / 4);

  const int nwg = gridDim.x, wg = blockIdx.x;
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 4, col = lane & 15;
  for (int v = threadIdx.x; v < NQT * SIM_QT * D / 8; v += SIM_THREADS) {
    const int r = (v * 8) / D, c = (v * 8) % D;
    bf16x8 x;
    if (r < Q) x = *reinterpret_cast<const bf16x8*>(queries + (size_t)r * D + c);
    else {
#pragma unroll
      for (int j = 0; j < 8; ++j) x[j] = (bf16)0.f;
    }
    *reinterpret_cast<bf16x8*>(qt + (size_t)r * QLD + c) = x;
  }
  if (threadIdx.x < SIM_MAXQ) {
    const int q = threadIdx.x;
    cnt[q] = 0;
    theta[q] = -INFINITY;
    minp[q] = q < Q ? q_minp[q] : 0x7fffffff;
    qtag[q] = q < Q ? q_tags[q] : 0ull;
  }
  if (threadIdx.x < 2) need[threadIdx.x] = 0;
  __syncthreads();

  float* my_s = cand_s + (size_t)wg * SIM_MAXQ * SIM_CAND;
  int* my_r = cand_r + (size_t)wg * SIM_MAXQ * SIM_CAND;
  const int per = ((N + nwg - 1) / nwg + 15) / 16 * 16;  // slices start on 16-row tiles
  const int r0 = wg * per, r1 = min(N, r0 + per);
  const int ngroups = (max(0, r1 - r0) + 15) / 16;
  constexpr int NW = SIM_THREADS / 64;
  const int nrounds = (ngroups + NW - 1) / NW;
  const int ksteps = D / 32;

  // Row loads are double-buffered in batches of SIM_KB k-steps (bufA / bufB) and
  // the first batch of a wave's NEXT 16-row group is issued before the round's
  // candidate work and barrier, so ~2 x SIM_KB KiB per wave stay in flight across
  // group and round boundaries (a round-synchronous loop drains the stream at
  // every barrier: 3.5-3.8 TB/s before).
  auto tile_ptr = [&](int grp_) {
    return index + ((size_t)((r0 + grp_ * 16) >> 4) * ksteps) * 512 + lane * 8;
  };
  auto load_batch = [&](const bf16* ap, int m, bf16x8 (&dst)[SIM_KB]) {
#pragma unroll
    for (int u = 0; u < SIM_KB; ++u)
      dst[u] = (m + u < ksteps) ? __builtin_nontemporal_load(reinterpret_cast<const bf16x8*>(ap + 512 * (m + u)))
                                : bf16x8{};
  };
  bf16x8 bufA[SIM_KB], bufB[SIM_KB];
  if (wid < ngroups) load_batch(tile_ptr(wid), 0, bufA);

  for (int round = 0; round < nrounds; ++round) {
    const int grp = round * NW + wid;
    const int gbase = r0 + grp * 16;
    f32x4 acc[SIM_MAXQ / SIM_QT];
#pragma unroll
    for (int t = 0; t < SIM_MAXQ / SIM_QT; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (grp < ngroups) {
      // packed tile gbase/16: k-step m is 64 lanes x 16 B contiguous (1 KiB per wave load)
      const bf16* ap = tile_ptr(grp);
      // the rows' filter words ride along, older than the group's later batches: read where a row is admitted, each was
      // a load to wait for behind the row stream
      const int rowc = min(gbase + col, r1 - 1);
      const int pr = row_prio[rowc];
      const float ex = row_exp[rowc];
      const uint64_t tg = row_tags[rowc];
      auto compute = [&](const bf16x8 (&av)[SIM_KB], int m) {
#pragma unroll
        for (int u = 0; u < SIM_KB; ++u) {
          if (m + u >= ksteps) break;
#pragma unroll
          for (int t = 0; t < SIM_MAXQ / SIM_QT; ++t) {
            if (t < NQT) {
              const bf16x8 b = *reinterpret_cast<const bf16x8*>(qt + (size_t)(t * SIM_QT + col) * QLD + 32 * (m + u) + 8 * g);
              acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av[u], b, acc[t], 0, 0, 0);
            }
          }
        }
      };
      for (int m = 0; m < ksteps; m += 2 * SIM_KB) {
        if (m + SIM_KB < ksteps) load_batch(ap, m + SIM_KB, bufB);
        if (m == 0 && g == 0) {
          tg_lds[wid * 16 + col] = tg;
          pr_lds[wid * 16 + col] = pr;
          ex_lds[wid * 16 + col] = ex;
        }
        compute(bufA, m);
        if (m + 2 * SIM_KB < ksteps) load_batch(ap, m + 2 * SIM_KB, bufA);
        else if (grp + NW < ngroups) load_batch(tile_ptr(grp + NW), 0, bufA);  // next group's first batch
        if (m + SIM_KB < ksteps) compute(bufB, m + SIM_KB);
      }
    }
    // lane holds rows gbase + 4g + r for queries t*16 + col
    auto passes = [&](int at, int q) {  // the row's words (its place in the LDS arrays) against a query's filters
      const float ex = ex_lds[at];
      return pr_lds[at] >= minp[q] && (tg_lds[at] & qtag[q]) == qtag[q] && (ex == 0.f || ex > now);
    };
    if (round == 0) {
      // The first groups show their best before any row is admitted: of every four rows the best score that passes the
      // query's filters, whose K-th best is where the query begins. (With all 256 rows admitted for every
      // query, the first round was most of a small index's pass: 64 queries of 131,000 rows 292 us a lookup, 261 so.)
#pragma unroll
      for (int t = 0; t < SIM_MAXQ / SIM_QT; ++t) {
        if (t >= NQT) break;
        const int q = t * SIM_QT + col;
        uint32_t best = 0;
        if (grp < ngroups) {
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (gbase + 4 * g + r < r1 && passes(wid * 16 + 4 * g + r, q) && is_finite(acc[t][r])) best = max(best, ord_key(acc[t][r]));
        }
        first[q * 65 + wid * 4 + g] = best;
      }
      __syncthreads();
      for (int q = wid; q < Q; q += NW) {
        const uint32_t key[1] = {lane < NW * 4 ? first[q * 65 + lane] : 0};
        if (__popcll(__ballot(key[0] != 0)) >= K) {
          const uint32_t k = wave_select_floor<13>(key, K);
          // (rows that reach it are admitted: just below it, also where it is 0)
          if (lane == 0) theta[q] = fminf(key_value(k - 1), key_value(k) - 1e-30f);
        }
      }
      __syncthreads();
    }
    if (grp < ngroups) {
      unsigned reach = 0;  // bit 4 t + r: some lane's score is above its query's threshold
#pragma unroll
      for (int t = 0; t < SIM_MAXQ / SIM_QT; ++t) {
        if (t >= NQT) break;
        const float th = t * SIM_QT + col < Q ? theta[t * SIM_QT + col] : INFINITY;
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (__any(acc[t][r] > th)) reach |= 1u << (4 * t + r);
      }
      if (reach) {
#pragma unroll
        for (int t = 0; t < SIM_MAXQ / SIM_QT; ++t) {
          const int q = t * SIM_QT + col;
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            if (!((reach >> (4 * t + r)) & 1u)) continue;
            const int row = gbase + 4 * g + r;
            const float sc = acc[t][r];
            if (row >= r1 || q >= Q || !(sc > theta[q]) || !passes(wid * 16 + 4 * g + r, q)) continue;
            const int pos = atomicAdd(&cnt[q], 1);
            if (pos < SIM_CAND) {
              my_s[q * SIM_CAND + pos] = sc;
              my_r[q * SIM_CAND + pos] = row;
            }
            if (pos == SIM_LIM) need[round & 1] = 1;
          }
        }
      }
    }
    __syncthreads();
    static_assert(SIM_LIM + NW * 16 <= SIM_CAND, "a buffer must absorb a round");
    if (need[round & 1]) {
      __syncthreads();
      if (threadIdx.x == 0) need[round & 1] = 0;
      for (int q = wid; q < Q; q += NW)  // (those that would be due soon with them)
        if (cnt[q] > SIM_MAXK) compact_global(my_s + q * SIM_CAND, my_r + q * SIM_CAND, &cnt[q], &theta[q], K);
      __syncthreads();
    }
  }
  __syncthreads();
  for (int q = wid; q < Q; q += NW) {
    const size_t o = ((size_t)q * nwg + wg) * K;
    compact_global(my_s + q * SIM_CAND, my_r + q * SIM_CAND, &cnt[q], &theta[q], K, ws_s + o, ws_r + o);
  }
}

// Few queries of a short index: a workgroup's slice is one 16-row tile a wave. All of a tile is on its way before the queries
// are in LDS, and a slice's scores are chosen from in LDS, a wave a query, with no threshold and no buffers in memory (each
// a trip that the whole launch waited for). Bound by latency: 3 queries of 20,011 rows x 1,024 15.2 -> 9.0 us (slices of 128 rows
// through cosine_stage1_kernel before), of which the rows' 41 MB are 6; 16 of 32,768 25 -> 16.5, 1 of 1,000 x 256 8.9 -> 4.5.
template <int KS>
__global__ __launch_bounds__(512) void cosine_short_kernel(
    float* __restrict__ ws_s, int* __restrict__ ws_r, const bf16* __restrict__ queries, const bf16* __restrict__ index, int Q, int N,
    int D, int K, const int* __restrict__ row_prio, const uint64_t* __restrict__ row_tags, const float* __restrict__ row_exp,
    const int* __restrict__ q_minp, const uint64_t* __restrict__ q_tags, float now) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int QLD = D + 8, NW = blockDim.x >> 6, rows = 16 * NW, ksteps = D / 32;
  bf16* qt = reinterpret_cast<bf16*>(smem);                                // [16][QLD], the first Q of them
  uint32_t* keys = reinterpret_cast<uint32_t*>(smem + SIM_QT * QLD * 2);   // [16][rows]
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 4, col = lane & 15, r0 = blockIdx.x * rows + wid * 16;  // (the first row of a tile is below N or not at all)
  const bf16* ap = index + (size_t)(min(r0, (N - 1) & ~15) >> 4) * ksteps * 512 + lane * 8;
  bf16x8 a[KS];
#pragma unroll
  for (int m = 0; m < KS; ++m)
    a[m] = m < ksteps ? __builtin_nontemporal_load(reinterpret_cast<const bf16x8*>(ap + 512 * m)) : bf16x8{};
  // the words of this lane's four rows and of its query
  int pr[4];
  float ex[4];
  uint64_t tg[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int row = min(r0 + 4 * g + r, N - 1);
    pr[r] = row_prio[row];
    ex[r] = row_exp[row];
    tg[r] = row_tags[row];
  }
  const int q = min(col, Q - 1), minp = q_minp[q];
  const uint64_t qtag = q_tags[q];
  for (int v = threadIdx.x; v < Q * D / 8; v += blockDim.x) {
    const int r = (v * 8) / D, c = (v * 8) % D;
    *reinterpret_cast<bf16x8*>(qt + (size_t)r * QLD + c) = *reinterpret_cast<const bf16x8*>(queries + (size_t)r * D + c);
  }
  __syncthreads();
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  const bf16* qr = qt + (size_t)q * QLD + 8 * g;
#pragma unroll
  for (int m = 0; m < KS; ++m)
    if (m < ksteps) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[m], *reinterpret_cast<const bf16x8*>(qr + 32 * m), acc, 0, 0, 0);
  // lane holds rows r0 + 4 g + r for query col
  constexpr uint32_t LOWEST = 0x007fffffu, HIGHEST = 0xff800000u;  // -inf, inf
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const bool passes = r0 + 4 * g + r < N && pr[r] >= minp && (tg[r] & qtag) == qtag && (ex[r] == 0.f || ex[r] > now);
    const uint32_t key = ord_key(acc[r]);  // (neither -inf nor what is no number: by their places in the order)
    keys[col * rows + wid * 16 + 4 * g + r] = passes && key > LOWEST && key <= HIGHEST ? key : 0;
  }
  __syncthreads();
  for (int i = wid; i < Q; i += NW) {
    uint32_t key[2];
    int have = 0, at = 0;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      key[j] = 64 * j + lane < rows ? keys[i * rows + 64 * j + lane] : 0;
      have += __popcll(__ballot(key[j] != 0));
    }
    uint32_t cut = 1;  // entries above it stay, and of those at it as many as there is room for
    int room = K;
    if (have >= K) {
      cut = wave_select(key, K);
#pragma unroll
      for (int j = 0; j < 2; ++j) room -= __popcll(__ballot(key[j] > cut));
    }
    const size_t o = ((size_t)i * gridDim.x + blockIdx.x) * K;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const unsigned long long ties = __ballot(key[j] == cut);
      const bool keep = key[j] > cut || (key[j] == cut && rank_in(ties) < room);
      room -= __popcll(ties);
      const unsigned long long kept = __ballot(keep);
      if (keep) {
        ws_s[o + at + rank_in(kept)] = key_value(key[j]);
        ws_r[o + at + rank_in(kept)] = blockIdx.x * rows + 64 * j + lane;
      }
      at += __popcll(kept);
    }
    if (lane >= at && lane < K) { ws_s[o + lane] = -INFINITY; ws_r[o + lane] = -1; }
  }
}

// Stage 2: one workgroup per query picks the best K of the slices' lists, PER entries a thread. The best of every four
// threads' entries are 256 keys, whose K-th is reached by K entries at least and, unless the best lie together, by few more:
// those are ranked. Only where they are more than fit does the selection count all keys bit by bit, with a barrier a bit (3
// queries, 251 lists of 5: 9.2 -> 5.2 us; 16 queries, 250 lists of 20: 19.9 -> 9.5).
template <int PER>
__global__ __launch_bounds__(1024) void cosine_stage2_kernel(float* __restrict__ out_s, int* __restrict__ out_r,
                                                             const float* __restrict__ ws_s, const int* __restrict__ ws_r,
                                                             int nwg, int K) {
  __shared__ Selection sel;
  __shared__ int red[2 * 16];
  __shared__ uint32_t best[256];
  const int q = blockIdx.x, total = nwg * K, lane = threadIdx.x & 63;
  const float* s = ws_s + (size_t)q * total;
  const int* r = ws_r + (size_t)q * total;
  uint32_t key[PER], top = 0;
  int row[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int e = i * 1024 + threadIdx.x;
    row[i] = e < total ? r[e] : -1;
    key[i] = row[i] >= 0 ? ord_key(s[e]) : 0;
    top = max(top, key[i]);
  }
  top = max(top, (uint32_t)__shfl_xor((int)top, 1, 64));
  top = max(top, (uint32_t)__shfl_xor((int)top, 2, 64));
  if ((lane & 3) == 0) best[threadIdx.x >> 2] = top;
  if (threadIdx.x == 0) sel.n = 0;
  __syncthreads();
  uint32_t b[4], from = 1;
  int have = 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    b[i] = best[64 * i + lane];
    have += __popcll(__ballot(b[i] != 0));
  }
  if (have >= K) from = max(1u, wave_select_floor<13>(b, K));
#pragma unroll
  for (int i = 0; i < PER; ++i)
    if (key[i] >= from) {
      const int p = atomicAdd(&sel.n, 1);
      if (p < SEL) { sel.key[p] = key[i]; sel.row[p] = row[i]; }
    }
  __syncthreads();
  out_s += (size_t)q * K;
  out_r += (size_t)q * K;
  if (sel.n <= SEL) return write_ranked(sel, K, out_s, out_r);
  const uint32_t kth = block_select<PER, 16>(key, K, red);  // (more than SEL entries: more than K)
  write_best(key, row, kth, K, sel, out_s, out_r);
}

}  // namespace pa

// workspace = stage-1 top-k lists [Q][nwg][K] (score, row) and, but for a short index, per-(slice, query) candidate buffers
// [nwg][64][CAND] (score, row). Q > 64: what the largest of its passes of 64 needs (a last one of few queries has more slices of
// a short index).
extern "C" long long pa_cosine_topk_workspace_bytes(int Q, int N, int K) {
  if (Q > pa::SIM_MAXQ)
    return std::max(pa_cosine_topk_workspace_bytes(pa::SIM_MAXQ, N, K), pa_cosine_topk_workspace_bytes((Q - 1) % pa::SIM_MAXQ + 1, N, K));
  const long long w = pa::sim_num_wg(Q, N);
  return Q * w * K * 8 + (pa::sim_short(Q, N) ? 0 : w * pa::SIM_MAXQ * pa::SIM_CAND * 8);
}

extern "C" int pa_cosine_topk(float* out_scores, int* out_rows, void* workspace,
                              const void* queries, const void* index, int Q, int N, int D, int K,
                              const int* row_priority, const uint64_t* row_tags,
                              const float* row_expiry, const int* q_min_priority,
                              const uint64_t* q_tags, float now, int n_valid, hipStream_t st) {
  (void)n_valid;
  if (Q <= 0) return 0;
  if (D % 32 != 0 || D > pa::SIM_MAXD || K < 1 || K > pa::SIM_MAXK || Q > pa::SIM_MAXQ) return -1;
  if (N <= 0) {
    // empty index: every query gets an empty result (the reference raised here)
    (void)hipMemsetAsync(out_rows, 0xff, (size_t)Q * K * sizeof(int), st);
    return (int)hipGetLastError();
  }
  const int nwg = pa::sim_num_wg(Q, N);
  float* ws_s = reinterpret_cast<float*>(workspace);
  int* ws_r = reinterpret_cast<int*>(ws_s + (size_t)Q * nwg * K);
  float* cand_s = reinterpret_cast<float*>(ws_r + (size_t)Q * nwg * K);
  int* cand_r = reinterpret_cast<int*>(cand_s + (size_t)nwg * pa::SIM_MAXQ * pa::SIM_CAND);
  const int nqt = (Q + pa::SIM_QT - 1) / pa::SIM_QT, threads = pa::SIM_ROUND * 4;
  const size_t lds = (size_t)nqt * pa::SIM_QT * (D + 8) * 2 + pa::SIM_MAXQ * (4 + 4 + 4 + 8) + 16 +
                     threads / 4 * 16 + (size_t)nqt * pa::SIM_QT * 65 * 4;
  if (pa::sim_short(Q, N)) {
    const int waves = pa::sim_short_waves(N);
    auto* scan = D <= 256 ? pa::cosine_short_kernel<8> : D <= 512 ? pa::cosine_short_kernel<16> : pa::cosine_short_kernel<32>;
    hipLaunchKernelGGL(scan, dim3(nwg), dim3(64 * waves), pa::SIM_QT * ((D + 8) * 2 + 16 * waves * 4), st, ws_s, ws_r,
                       (const pa::bf16*)queries, (const pa::bf16*)index, Q, N, D, K, row_priority, row_tags, row_expiry, q_min_priority,
                       q_tags, now);
  } else {
    static bool attr_set = false;
    if (!attr_set) {
      (void)hipFuncSetAttribute((const void*)pa::cosine_stage1_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
      attr_set = true;
    }
    hipLaunchKernelGGL(pa::cosine_stage1_kernel, dim3(nwg), dim3(threads), lds, st, ws_s, ws_r, cand_s, cand_r, (const pa::bf16*)queries,
                       (const pa::bf16*)index, Q, N, D, K, row_priority, row_tags, row_expiry, q_min_priority, q_tags, now);
  }
  static_assert(pa::SIM_MAX_WG * pa::SIM_MAXK <= 16 * 1024, "stage 2 holds all lists");
  auto* merge = nwg * K <= 1024 ? pa::cosine_stage2_kernel<1>
                                : nwg * K <= 4096 ? pa::cosine_stage2_kernel<4> : pa::cosine_stage2_kernel<16>;
  hipLaunchKernelGGL(merge, dim3(Q), dim3(1024), 0, st, out_scores, out_rows, ws_s, ws_r, nwg, K);
  return (int)hipGetLastError();
}
