// Grouped projections: many small weight matrices, each applied to its own rows.
//
//   dense   every row goes through every group, group h reading its own columns of x and writing
//           its own columns of out (per-head up-projections of latent attention)
//   sorted  row p belongs to one group: mixture-of-experts layers, rows sorted by expert into
//           tiles of at most TM rows (table_route_kernel below)
//
// Weights are packed per group like the other projections ([N/16, K/32, 64, 8], one 16-B lane
// vector per MFMA operand). The MFMA's A operand is W and its B operand x, so a lane's four
// accumulators are four consecutive outputs of one row: 8-byte stores, and the gated pair
// (tiles 2i: gate, 2i + 1: up) is lane-local. Sorted rows go in tiles of 16 to 128, as the caller asks (experts: 16
// and 32 up to 24 rows on average, one group: up to 64); more run the ping-pong kernels (gemm_prefill.hip pa_expert_tiles).
//
// Epilogues: plain, the gated unit of packed_epi.h (limit, alpha, cubic, bias), or the square of relu; of dense rows
// also the product times sigmoid(gate), and the gated unit whose second factor is the row's embedding in a table.
// Sorted rows may have weights: the product is that of weight * x.
#include "packed_epi.h"

extern "C" int pa_expert_tiles(void* y, const void* x, const void* wp, long long wstride, int groups, int N, int K, int ldx, int ldy,
                               const int* tiles, int max_tiles, const int* n_tiles, const int* order, int x_div,
                               int out_order, int epi, float limit, float alpha, float cubic, float bias, const float* row_w,
                               const int* live, int always, hipStream_t st);

namespace pa {
namespace gg {

struct Args {
  const void* x;
  const void* w;
  void* out;
  long long wstride;       // elements per group
  int ldx, xg, ldo, og;    // row strides and per-group column offsets (dense)
  int rows, N16, K32;      // dense rows; N16 = packed 16-row tiles per group
  const int4* tiles;       // sorted: {group, first position, rows, 0}
  const int* n_tiles;
  const int* order;        // sorted: position -> token * top + k
  int x_div;               // sorted: x row = order / x_div (0: x row = position)
  int out_order;           // sorted: out row = order[position] (0: out row = position)
  float limit, alpha, cubic, bias;
  // dense, optional: after a group's N columns of out, the rotated part of the row's head (r columns of
  // x at the group's offset + rskip, the first rd turned by the row's position), padded to rp columns
  const int* positions;
  const float* cos_sin;
  int rskip, r, rp, rd;
  int wide;  // out rows and group offsets are multiples of 8 elements
  const float* row_w;      // sorted, optional: by order[position], the weight of x's row
  // dense, optional: gate [rows, ldg], columns as out's; table rows ids[row], its columns at tcol as out's
  const void *gate, *table;
  const int* ids;
  int ldg, ldt, tcol, vocab;
  const int* skip;  // dense, optional: rows that are not 0 here stay as they are
};

// all of a tile's rows (64 at most) are left out
__device__ __forceinline__ bool skipped(const Args& A, int start, int n) {
  if (!A.skip) return false;
  const int lane = threadIdx.x & 63;
  return __all(lane >= n || A.skip[start + min(lane, n - 1)] != 0);
}

// The rotated columns of `n` rows from `start` of group grp (one workgroup), of those that are not left out.
template <typename T>
__device__ __forceinline__ void rotate_rows(const Args& A, int grp, int start, int n) {
  const int half = A.rd >> 1, N = A.N16 * 16;
  if (sizeof(T) == 2 && half % 8 == 0 && A.rd == A.r && A.rskip % 8 == 0 && A.xg % 8 == 0 && A.og % 8 == 0 &&
      A.ldo % 8 == 0) {
    // 8 pairs a thread, 16-byte accesses
    const int hp = half >> 3;
    for (int e = threadIdx.x; e < n * hp; e += 256) {
      const int t = start + e / hp, j = (e % hp) * 8;
      if (A.skip && A.skip[t]) continue;
      const bf16* src = (const bf16*)A.x + (size_t)t * A.ldx + (size_t)grp * A.xg + A.rskip + j;
      bf16* dst = (bf16*)A.out + (size_t)t * A.ldo + (size_t)grp * A.og + N + j;
      const float* cs = A.cos_sin + (size_t)A.positions[t] * A.rd + j;
      const bf16x8 u = *reinterpret_cast<const bf16x8*>(src), v = *reinterpret_cast<const bf16x8*>(src + half);
      float c[8], s[8];
      __builtin_memcpy(c, cs, 32);
      __builtin_memcpy(s, cs + half, 32);
      bf16x8 a, b;
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        a[k] = (bf16)((float)u[k] * c[k] - (float)v[k] * s[k]);
        b[k] = (bf16)((float)v[k] * c[k] + (float)u[k] * s[k]);
      }
      *reinterpret_cast<bf16x8*>(dst) = a;
      *reinterpret_cast<bf16x8*>(dst + half) = b;
    }
    for (int e = threadIdx.x; e < n * (A.rp - A.r); e += 256) {
      const int t = start + e / (A.rp - A.r);
      if (A.skip && A.skip[t]) continue;
      ((T*)A.out)[(size_t)t * A.ldo + (size_t)grp * A.og + N + A.r + e % (A.rp - A.r)] = (T)0.f;
    }
    return;
  }
  const int per = max(1, 256 / A.rp), i0 = threadIdx.x / A.rp;  // rows at a time
  for (int j = threadIdx.x % A.rp; j < A.rp && i0 < per; j += 256) {
#pragma unroll 4
    for (int i = i0; i < n; i += per) {
      const int t = start + i;
      if (A.skip && A.skip[t]) continue;
      const T* src = (const T*)A.x + (size_t)t * A.ldx + (size_t)grp * A.xg + A.rskip;
      float v = 0.f;
      if (j < A.r) {
        v = (float)src[j];
        const float* cs = A.cos_sin + (size_t)A.positions[t] * A.rd;
        if (j < half) v = v * cs[j] - (float)src[j + half] * cs[half + j];
        else if (j < A.rd) v = v * cs[j - half] + (float)src[j - half] * cs[j];
      }
      ((T*)A.out)[(size_t)t * A.ldo + (size_t)grp * A.og + N + j] = (T)v;
    }
  }
}

__device__ __forceinline__ float glu(float g, float u, const Args& A) {
  return pk::gated_unit(g, u, A.limit, A.alpha, A.cubic, A.bias);
}

enum { PLAIN = 0, GLU = 1, RELU2 = 2, GATED = 3, TABLE = 4 };

// where the second factor of a dense row's outputs lies (GATED, TABLE)
template <typename T, int EPI>
__device__ __forceinline__ const T* factor_row(const Args& A, int row, int grp) {
  if constexpr (EPI == GATED) return (const T*)A.gate + (size_t)row * A.ldg + (size_t)grp * A.og;
  return (const T*)A.table + (size_t)min(max(A.ids[row], 0), A.vocab - 1) * A.ldt + A.tcol;
}
template <int EPI>
__device__ __forceinline__ float times(float a, float f, const Args& A) {
  if constexpr (EPI == GATED) return a / (1.f + __expf(-f));
  return glu(a, f, A);
}

// A wave's outputs: 16 NT of a group's columns from nt0 on, of the rows m * 16 + c < n from `start`.
template <int MT, int NT, int EPI>
__device__ __forceinline__ void store_rows(const Args& A, int grp, int start, int n, int nt0, const f32x4 (&acc)[MT][NT]) {
  const int lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4;
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    if (16 * m + c >= n) continue;
    const int at = start + 16 * m + c;
    if (A.skip && A.skip[at]) continue;
    bf16* o = (bf16*)A.out + (size_t)at * A.ldo + (size_t)grp * A.og + 4 * g;
    if constexpr (EPI == GATED) {
      const bf16* f = factor_row<bf16, EPI>(A, at, grp) + 4 * g;
#pragma unroll
      for (int i = 0; i < NT; ++i) {
        if (nt0 + i >= A.N16) break;
        const bf16x4 fv = *reinterpret_cast<const bf16x4*>(f + (nt0 + i) * 16);
        bf16x4 v;
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = (bf16)times<EPI>(acc[m][i][j], (float)fv[j], A);
        *reinterpret_cast<bf16x4*>(o + (nt0 + i) * 16) = v;
      }
    } else if (NT % 2 == 0 && A.N16 % 2 == 0 && A.wide) {
      // 16-byte stores: lanes of neighbouring lane groups trade halves
      const struct { bf16* y; int ldy; } row{o - 4 * g, 0};
#pragma unroll
      for (int i = 0; i + 1 < NT; i += 2) {
        if (nt0 + i >= A.N16) break;
        pk::store_pair_wide<pk::EP_PLAIN>(row, 0, nt0 + i, g, acc[m][i], acc[m][i + 1]);
      }
    } else {
#pragma unroll
      for (int i = 0; i < NT; ++i) {
        if (nt0 + i >= A.N16) break;
        bf16x4 v;
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = (bf16)acc[m][i][j];
        *reinterpret_cast<bf16x4*>(o + (nt0 + i) * 16) = v;
      }
    }
  }
}

// Sorted rows: the NT tiles from nt on of the row 16 m + c (GLU: a gate and an up tile).
template <int EPI, int NT>
__device__ __forceinline__ void store_sorted(const Args& A, int start, int n, int m, int nt, const f32x4 (&a)[NT]) {
  const int lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4;
  if (16 * m + c >= n || nt >= A.N16) return;
  const int p = start + 16 * m + c;
  bf16* o = (bf16*)A.out + (size_t)(A.out_order ? A.order[p] : p) * A.ldo + 4 * g;
  if constexpr (EPI == GLU) {
    const float rw = A.row_w ? A.row_w[A.order[p]] : 1.f;
    bf16x4 v;
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = (bf16)glu(a[0][j] * rw, a[1][j] * rw, A);
    *reinterpret_cast<bf16x4*>(o + nt * 8) = v;
    return;
  }
  if constexpr (NT == 2) {
    if (A.N16 % 2 == 0 && A.wide) {
      const struct { bf16* y; int ldy; } row{o - 4 * g, 0};
      pk::store_pair_wide<EPI == RELU2 ? pk::EP_RELU2 : pk::EP_PLAIN>(row, 0, nt, g, a[0], a[1]);
      return;
    }
  }
#pragma unroll
  for (int i = 0; i < NT; ++i) {
    if (nt + i >= A.N16) break;
    bf16x4 v;
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = (bf16)(EPI == RELU2 ? pk::relu2(a[i][j]) : a[i][j]);
    *reinterpret_cast<bf16x4*>(o + (nt + i) * 16) = v;
  }
}

// Tiles of 16 MT rows and 16 NT outputs a wave, straight from memory: dense rows (PLAIN, GATED), and sorted ones (PLAIN, GLU,
// RELU2) of few inputs (sorted_rows).
template <int MT, int NT, int KU, int EPI, bool SORTED = false>
__global__ __launch_bounds__(256) void gemm_kernel(const Args A) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int c = lane & 15, g = lane >> 4;
  int grp = blockIdx.z, start = blockIdx.y * (16 * MT), n = min(16 * MT, A.rows - start);
  if constexpr (SORTED) {
    if ((int)blockIdx.y >= A.n_tiles[0]) return;
    const int4 tl = A.tiles[blockIdx.y];
    grp = tl.x;
    start = tl.y;
    n = tl.z;
  } else {
    if (skipped(A, start, n)) return;
  }
  if (A.rp && blockIdx.x == 0) {
    rotate_rows<bf16>(A, grp, start, n);
    return;
  }
  const int nt0 = (((int)blockIdx.x - (A.rp ? 1 : 0)) * 4 + wid) * NT;
  if (nt0 >= A.N16) return;
  const bf16* wp = (const bf16*)A.w + (size_t)grp * A.wstride + lane * 8;
  const bf16* wt[NT];
#pragma unroll
  for (int i = 0; i < NT; ++i) wt[i] = wp + (size_t)min(nt0 + i, A.N16 - 1) * A.K32 * 512;
  const bf16* xr[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    int row = start + min(16 * m + c, n - 1);
    if (SORTED && A.x_div) row = A.order[row] / A.x_div;
    xr[m] = (const bf16*)A.x + (size_t)row * A.ldx + (SORTED ? 0 : (size_t)grp * A.xg) + 8 * g;
  }
  f32x4 acc[MT][NT];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int i = 0; i < NT; ++i) acc[m][i] = f32x4{0.f, 0.f, 0.f, 0.f};
  bf16x8 a[KU][NT], b[KU][MT];
  auto load = [&](int s, bf16x8 (&aa)[KU][NT], bf16x8 (&bb)[KU][MT]) {
#pragma unroll
    for (int k = 0; k < KU; ++k) {
#pragma unroll
      for (int i = 0; i < NT; ++i) aa[k][i] = *reinterpret_cast<const bf16x8*>(wt[i] + (size_t)(s + k) * 512);
#pragma unroll
      for (int m = 0; m < MT; ++m) bb[k][m] = *reinterpret_cast<const bf16x8*>(xr[m] + (size_t)(s + k) * 32);
    }
  };
  load(0, a, b);
  for (int s = 0; s < A.K32; s += KU) {
    bf16x8 an[KU][NT], bn[KU][MT];
    if (s + KU < A.K32) load(s + KU, an, bn);
#pragma unroll
    for (int k = 0; k < KU; ++k)
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int i = 0; i < NT; ++i)
          acc[m][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[k][i], b[k][m], acc[m][i], 0, 0, 0);
#pragma unroll
    for (int k = 0; k < KU; ++k) {
#pragma unroll
      for (int i = 0; i < NT; ++i) a[k][i] = an[k][i];
#pragma unroll
      for (int m = 0; m < MT; ++m) b[k][m] = bn[k][m];
    }
  }
  if constexpr (SORTED) {
#pragma unroll
    for (int m = 0; m < MT; ++m) store_sorted<EPI, NT>(A, start, n, m, nt0, acc[m]);
  } else {
    store_rows<MT, NT, EPI>(A, grp, start, n, nt0, acc);
  }
}

// Many dense rows of groups with few inputs (the heads of a latent attention): 64 rows of a group's inputs whole in LDS,
// every one of its outputs from there. In gemm_kernel each wave fetches them by itself, in pieces of 64 bytes, for every
// 64 outputs. Units of 8 inputs, [K / 8][64 rows][8] and a row of padding, so that rows are written and fragments read
// without conflicts. 4,096 rows, 16 heads: 128 -> 512 beside 64 rotated 43 -> 34 us (88 MB:
// 18 us at the rate of a copy). 512 -> 128 stays there: 29 us, here 31, as the rows arrive before the first product; and so
// do fewer than two workgroups a CU (512 rows of 16 heads: 10 us, here 11), and gated outputs of many workgroups and fewer
// inputs (4,096 rows, 16 heads of 1,024, times a gate: of 64 inputs 117 us, here 145, of 128 136, 149; 8 heads 46, 38 and 51,
// 42).
constexpr int HEAD_UNIT = 65 * 16, HEAD_K32 = 8;

template <int EPI>
__global__ __launch_bounds__(256, 2) void head_rows_kernel(const Args A) {
  constexpr int NT = 4;
  extern __shared__ __attribute__((aligned(16))) char xs[];
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), c = lane & 15, g = lane >> 4;
  const int grp = blockIdx.y, start = blockIdx.x * 64, n = min(64, A.rows - start), U = 4 * A.K32;
  if (skipped(A, start, n)) return;
  const bf16* x = (const bf16*)A.x + (size_t)start * A.ldx + (size_t)grp * A.xg;
  const unsigned inv = ((1u << 20) + U - 1) / U;  // e / U of e < 4096
  bf16x8 v[HEAD_K32];
  auto unit = [&](int k, int& j) {
    const unsigned e = k * 256 + threadIdx.x;
    j = e * inv >> 20;
    return (int)e - j * U;
  };
#pragma unroll
  for (int k = 0; k < HEAD_K32; ++k)
    if (k < A.K32) {
      int j;
      const int u = unit(k, j);
      v[k] = *reinterpret_cast<const bf16x8*>(x + (size_t)min(j, n - 1) * A.ldx + 8 * u);
    }
#pragma unroll
  for (int k = 0; k < HEAD_K32; ++k)
    if (k < A.K32) {
      int j;
      const int u = unit(k, j);
      *reinterpret_cast<bf16x8*>(xs + u * HEAD_UNIT + j * 16) = v[k];
    }
  if (A.rp) rotate_rows<bf16>(A, grp, start, n);
  __syncthreads();
  const bf16* wp = (const bf16*)A.w + (size_t)grp * A.wstride + lane * 8;
  const char* xf = xs + g * HEAD_UNIT + c * 16;
  for (int nt0 = wid * NT; nt0 < A.N16; nt0 += 4 * NT) {
    const bf16* wt[NT];
#pragma unroll
    for (int i = 0; i < NT; ++i) wt[i] = wp + (size_t)min(nt0 + i, A.N16 - 1) * A.K32 * 512;
    f32x4 acc[4][NT];
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
      for (int i = 0; i < NT; ++i) acc[m][i] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto load = [&](int s, bf16x8 (&a)[NT]) {  // (past the end: the last step's again)
#pragma unroll
      for (int i = 0; i < NT; ++i) a[i] = *reinterpret_cast<const bf16x8*>(wt[i] + (size_t)min(s, A.K32 - 1) * 512);
    };
    auto step = [&](int s, const bf16x8 (&a)[NT]) {
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        const bf16x8 b = *reinterpret_cast<const bf16x8*>(xf + s * (4 * HEAD_UNIT) + m * 256);
#pragma unroll
        for (int i = 0; i < NT; ++i) acc[m][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], b, acc[m][i], 0, 0, 0);
      }
    };
    bf16x8 a0[NT], a1[NT];
    load(0, a0);
    load(1, a1);
    int s = 0;
    for (; s + 1 < A.K32; s += 2) {
      step(s, a0);
      load(s + 2, a0);
      step(s + 1, a1);
      load(s + 3, a1);
    }
    if (s < A.K32) step(s, a0);
    store_rows<4, NT, EPI>(A, grp, start, n, nt0, acc);
  }
}

// Sorted rows in tiles of 16 MT = 16 to 128: the rows of a group go through its weights together, so that these leave
// memory once. A workgroup loads its rows (wherever they lie) in whole lines, 64 WK k a stage, and its waves read the
// fragments from LDS: a wave's own fragment loads, 16 rows x 64 B an instruction, cost more than the weights. 8 waves lie
// side by side over a pair of 16-output tiles each; with WK > 1, WK of them share one pair and split the k-steps of a
// stage, which leaves more workgroups. Weights and rows are one in-order ring of loads, D stages deep; the stage barrier
// waits for LDS alone. NTW: weights that no other tile reads are loaded non-temporal.
// Bound by the weights' bytes: 64 experts of 2 x 1408 x 2048 and 2048 x 1408 and a shared one, both products, us before ->
// after: 64 tokens 215 -> 182 (5.4 TB/s), 400 275 -> 228, 1000 456 -> 295 (the ping-pong kernels are the
// faster ones from 25 rows a group on: GROUP_TILES in models/common.py); a dense 2 x 8192 x 2048 gate and up of 64 rows
// 30 -> 17, of 256 rows 45 -> 33.
template <int MT, int WK, int EPI, bool NTW>
__global__ __launch_bounds__(512, MT == 8 ? 4 : 2) void rows_kernel(const Args A) {
  constexpr int WN = 8 / WK, NT = 2, KW = 2, D = 2;
  constexpr int TM = 16 * MT, KC = 64 * WK, XLD = KC * 2 + 16;
  constexpr int LR = KC / 8, RL = 512 / LR, XL = (TM + RL - 1) / RL;  // threads a row, rows a load, loads a stage
  extern __shared__ __attribute__((aligned(16))) char smem[];  // [2][TM][XLD], then the partial sums
  // A group's tiles read the same weights: the same block of outputs of each goes to one XCD, in turn, and finds them in
  // its L2 (the first block's XCD moves with the group, so that all have as many). Not with the 11 blocks or so of WK =
  // 1, which do not divide over 8 XCDs, and where most groups have one tile.
  const int blocks = (A.N16 + WN * NT - 1) / (WN * NT);
  int tile, block;
  if constexpr (WK == 1) {
    tile = blockIdx.x / blocks;
    block = blockIdx.x % blocks;
  } else {
    const int b8 = (blocks + 7) >> 3, seq = blockIdx.x >> 3;
    tile = seq / b8;
    block = seq % b8 * 8;
  }
  if (tile >= A.n_tiles[0]) return;
  const int4 tl = A.tiles[tile];
  const int grp = tl.x, start = tl.y, n = tl.z;
  if (WK > 1) block += (blockIdx.x + grp) & 7;
  if (block >= blocks) return;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, c = lane & 15, g = lane >> 4;
  const int wk = wid % WK, wn = wid / WK, xrow = threadIdx.x / LR, xu = threadIdx.x % LR;
  const int nt0 = (block * WN + wn) * NT, KS = A.K32, nst = (KS * 32 + KC - 1) / KC;
  const bf16x8* wt[NT];
#pragma unroll
  for (int j = 0; j < NT; ++j)
    wt[j] = reinterpret_cast<const bf16x8*>((const bf16*)A.w + (size_t)grp * A.wstride +
                                            (size_t)min(nt0 + j, A.N16 - 1) * KS * 512) + lane;
  const bf16* xr[XL];
#pragma unroll
  for (int i = 0; i < XL; ++i) {
    const int pos = start + min(xrow + RL * i, n - 1);
    xr[i] = (const bf16*)A.x + (size_t)(A.x_div ? A.order[pos] / A.x_div : pos) * A.ldx;
  }
  f32x4 acc[MT][NT];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[m][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  bf16x8 wb[D][KW][NT], xb[D][XL];
  // (past the end: the last ones again, unconditional, so that the waits stay counted)
  auto load = [&](int st, int d) {
    __builtin_amdgcn_sched_barrier(0);
    const int k = min(st * KC + 8 * xu, KS * 32 - 8);
#pragma unroll
    for (int i = 0; i < XL; ++i) xb[d][i] = *reinterpret_cast<const bf16x8*>(xr[i] + k);
#pragma unroll
    for (int u = 0; u < KW; ++u) {
      const int ks = min(st * (KC / 32) + wk * KW + u, KS - 1);
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        if constexpr (NTW) wb[d][u][j] = __builtin_nontemporal_load(wt[j] + (size_t)ks * 64);
        else wb[d][u][j] = wt[j][(size_t)ks * 64];
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };
#pragma unroll
  for (int d = 0; d < D; ++d) load(d, d);
  for (int st0 = 0; st0 < nst; st0 += D) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      const int st = st0 + d;
      if (st < nst) {  // uniform
        char* slot = smem + (st & 1) * TM * XLD;
#pragma unroll
        for (int i = 0; i < XL; ++i)
          if (TM % RL == 0 || xrow + RL * i < TM)
            *reinterpret_cast<bf16x8*>(slot + (xrow + RL * i) * XLD + 16 * xu) = xb[d][i];
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
#pragma unroll
        for (int u = 0; u < KW; ++u) {
          if (st * (KC / 32) + wk * KW + u < KS) {
#pragma unroll
            for (int m = 0; m < MT; ++m) {
              const bf16x8 b = *reinterpret_cast<const bf16x8*>(slot + (16 * m + c) * XLD + (wk * KW + u) * 64 + 16 * g);
#pragma unroll
              for (int j = 0; j < NT; ++j)
                acc[m][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wb[d][u][j], b, acc[m][j], 0, 0, 0);
            }
          }
        }
        load(st + D, d);
      }
    }
  }
  if constexpr (WK == 1) {
#pragma unroll
    for (int m = 0; m < MT; ++m) store_sorted<EPI, NT>(A, start, n, m, nt0, acc[m]);
  } else {
    __syncthreads();
    f32x4* red = reinterpret_cast<f32x4*>(smem);  // [WK][WN][MT][NT][64]
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int j = 0; j < NT; ++j) red[(((wk * WN + wn) * MT + m) * NT + j) * 64 + lane] = acc[m][j];
    __syncthreads();
    for (int t = wid; t < WN * MT; t += 8) {
      f32x4 v[NT];
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        v[j] = red[(t * NT + j) * 64 + lane];
#pragma unroll
        for (int w = 1; w < WK; ++w) v[j] += red[((w * WN * MT + t) * NT + j) * 64 + lane];
      }
      store_sorted<EPI, NT>(A, start, n, t % MT, (block * WN + t / MT) * NT, v);
    }
  }
}

template <int MT, int WK, bool NTW>
static int launch_rows(const Args& A, int epi, int max_tiles, hipStream_t st) {
  constexpr int TN = (8 / WK) * 32;
  constexpr int x = 2 * 16 * MT * (128 * WK + 16), sums = WK > 1 ? 8 * MT * 2 * 1024 : 0, lds = x > sums ? x : sums;
  static_assert(lds <= 160 * 1024, "LDS of a CU");
  static bool attr = false;
  if (!attr) {
    for (auto* k : {rows_kernel<MT, WK, PLAIN, NTW>, rows_kernel<MT, WK, GLU, NTW>, rows_kernel<MT, WK, RELU2, NTW>})
      (void)hipFuncSetAttribute((const void*)k, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    attr = true;
  }
  const int blocks = (A.N16 * 16 + TN - 1) / TN;
  hipLaunchKernelGGL((epi == 1 ? rows_kernel<MT, WK, GLU, NTW> : epi == 2 ? rows_kernel<MT, WK, RELU2, NTW> : rows_kernel<MT, WK, PLAIN, NTW>),
                     dim3((WK > 1 ? (blocks + 7) / 8 * 8 : blocks) * max_tiles), dim3(512), lds, st, A);
  return (int)hipGetLastError();
}

// Tiles of 16 and 32 rows whose stages of LDS do not pay: a wave's fragments straight from memory (gemm_kernel). us at 16
// rows a tile, rows_kernel against gemm_kernel: 64 experts of 2 x 256 x K and 96 rows, K = 256 6.9, 5.6, 512 9.3, 8.5, 1024
// 13.7, 14.2; of 2048 x K 16.3, 13.1, 25.4, 23.8, 38.9, 45.0. Few tiles end with their slowest (16 of 1024 x 512, 64 rows 6.6,
// 6.5; 24 of 2048 x 512 12.7, 13.3); few outputs leave rows_kernel few workgroups a group (64 of 128 x 2048, 600 rows 22, 16).
static bool few_inputs(const Args& A, bool glu, int max_tiles) {
  if (max_tiles > 65535) return false;  // (a dimension of its grid)
  const bool narrow = A.N16 <= 16 && max_tiles >= (A.K32 <= 16 ? 64 : 96);
  return A.K32 <= (glu ? 4 : 8) || narrow || (A.K32 <= 16 && max_tiles * A.N16 >= 1536);
}

// Waves over k (WK): 4 for few rows; with 64-row tiles of many groups 2 (T = 400: 228 us both products, 4: 246, 1: 254),
// with those of one group as many as leave at most two workgroups a CU (2 x 8192 x 2048 outputs of 128 rows: 4 26 us, of 256: 2
// 33 us, 4 45; of 512: 1 46 us, 2 57); 1 with 128 rows, whose accumulators fill a wave. Non-temporal weights where
// no more than every third tile is a group's second (64 tokens 192 -> 182 us; 400 tokens 240 -> 250).
static int sorted_rows(const Args& A, int epi, int tm, int groups, int max_tiles, hipStream_t st) {
  if (tm <= 32 && few_inputs(A, epi == 1, max_tiles)) {
#define PA_S(MT, NT, KU, G)                                                                                               \
  hipLaunchKernelGGL((gemm_kernel<MT, NT, KU, G, true>), dim3((A.N16 + 4 * NT - 1) / (4 * NT), max_tiles), dim3(256), 0, st, A)
#define PA_SK(MT, NT, G)                     \
  do {                                       \
    if (A.K32 % 4 == 0) PA_S(MT, NT, 4, G);  \
    else if (A.K32 % 2 == 0) PA_S(MT, NT, 2, G); \
    else PA_S(MT, NT, 1, G);                 \
  } while (0)
    if (tm == 16) {
      if (epi == 1) PA_SK(1, 2, GLU);
      else if (epi == 2) PA_SK(1, 1, RELU2);
      else PA_SK(1, 1, PLAIN);
    } else {
      if (epi == 1) PA_SK(2, 2, GLU);
      else if (epi == 2) PA_SK(2, 1, RELU2);
      else PA_SK(2, 1, PLAIN);
    }
#undef PA_SK
#undef PA_S
    return (int)hipGetLastError();
  }
  const bool once = (max_tiles - groups) * 2 <= groups;
  auto fits = [&](int wk) { return (A.N16 * 16 + 256 / wk - 1) / (256 / wk) * max_tiles <= 512; };
  if (tm == 16) return once ? launch_rows<1, 4, true>(A, epi, max_tiles, st) : launch_rows<1, 4, false>(A, epi, max_tiles, st);
  if (tm == 32) return once ? launch_rows<2, 4, true>(A, epi, max_tiles, st) : launch_rows<2, 4, false>(A, epi, max_tiles, st);
  if (tm == 128) return launch_rows<8, 1, false>(A, epi, max_tiles, st);
  if (tm != 64) return -2;
  if (groups == 1 && fits(4)) return once ? launch_rows<4, 4, true>(A, epi, max_tiles, st) : launch_rows<4, 4, false>(A, epi, max_tiles, st);
  if (groups == 1 && !fits(2)) return launch_rows<4, 1, false>(A, epi, max_tiles, st);
  return launch_rows<4, 2, false>(A, epi, max_tiles, st);
}

// Dense rows through one group of few outputs (TABLE): 8 waves share a tile of 16 MT rows and 16 NT outputs, each every
// eighth step of K, and add up through LDS.
template <int MT, int NT>
__global__ __launch_bounds__(512) void split_k_kernel(const Args A) {
  extern __shared__ __attribute__((aligned(16))) f32x4 red[];  // [8][MT NT][64]
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, c = lane & 15, g = lane >> 4;
  // tiles of the same rows next to each other on one XCD: they share its copy of x
  const int cols = (A.N16 + NT - 1) / NT, tiles = cols * ((A.rows + 16 * MT - 1) / (16 * MT)), per = (tiles + 7) >> 3;
  const int tile = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per || tile >= tiles) return;
  const int nt0 = tile % cols * NT, start = tile / cols * (16 * MT), n = min(16 * MT, A.rows - start);
  const bf16 *wt[NT], *xr[MT];
#pragma unroll
  for (int i = 0; i < NT; ++i) wt[i] = (const bf16*)A.w + (size_t)min(nt0 + i, A.N16 - 1) * A.K32 * 512 + lane * 8;
#pragma unroll
  for (int m = 0; m < MT; ++m) xr[m] = (const bf16*)A.x + (size_t)(start + min(16 * m + c, n - 1)) * A.ldx + 8 * g;
  f32x4 acc[MT][NT];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int i = 0; i < NT; ++i) acc[m][i] = f32x4{0.f, 0.f, 0.f, 0.f};
  constexpr int U = MT * NT == 1 ? 8 : 4;  // steps whose loads go out together
  for (int s = wid; s < A.K32; s += 8 * U) {
    bf16x8 a[U][NT], b[U][MT];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = min(s + 8 * u, A.K32 - 1);
#pragma unroll
      for (int i = 0; i < NT; ++i) a[u][i] = *reinterpret_cast<const bf16x8*>(wt[i] + (size_t)k * 512);
#pragma unroll
      for (int m = 0; m < MT; ++m) b[u][m] = *reinterpret_cast<const bf16x8*>(xr[m] + (size_t)k * 32);
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (s + 8 * u < A.K32) {
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
          for (int i = 0; i < NT; ++i) acc[m][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[u][i], b[u][m], acc[m][i], 0, 0, 0);
      }
  }
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int i = 0; i < NT; ++i) red[((wid * MT + m) * NT + i) * 64 + lane] = acc[m][i];
  __syncthreads();
  for (int t = wid; t < MT * NT; t += 8) {  // tile (m, i): the same lanes again
    const int m = t / NT, i = t % NT, row = start + 16 * m + c;
    f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < 8; ++w) v += red[((w * MT + m) * NT + i) * 64 + lane];
    if (16 * m + c >= n || nt0 + i >= A.N16) continue;
    const int col = (nt0 + i) * 16 + 4 * g;
    const bf16x4 f = *reinterpret_cast<const bf16x4*>(factor_row<bf16, TABLE>(A, row, 0) + col);
    bf16x4 o;
#pragma unroll
    for (int j = 0; j < 4; ++j) o[j] = (bf16)times<TABLE>(v[j], (float)f[j], A);
    *reinterpret_cast<bf16x4*>((bf16*)A.out + (size_t)row * A.ldo + col) = o;
  }
}

// fp32: one output (or gated pair) per thread, weights row-major [G, 16 N16, 32 K32] in the same
// row order as the packed ones. The exact path; not tuned.
template <int EPI>
__global__ __launch_bounds__(256) void gemm_f32_kernel(const Args A) {
  constexpr bool PAIR = EPI == GLU;
  constexpr int TM = 16;
  __shared__ float xs[TM][33], w0[16][33], w1[16][33];
  const int tn = threadIdx.x & 15, tm = threadIdx.x >> 4;
  int grp, start, n;
  if (A.tiles) {
    if ((int)blockIdx.y >= A.n_tiles[0]) return;
    const int4 tl = A.tiles[blockIdx.y];
    grp = tl.x; start = tl.y; n = tl.z;
  } else {
    grp = blockIdx.z;
    start = blockIdx.y * TM;
    n = min(TM, A.rows - start);
  }
  if (A.rp && blockIdx.x == 0) {
    rotate_rows<float>(A, grp, start, n);
    return;
  }
  const int bx = (int)blockIdx.x - (A.rp ? 1 : 0);
  const int K = A.K32 * 32;
  const float* wg = (const float*)A.w + (size_t)grp * A.wstride + (size_t)bx * (PAIR ? 32 : 16) * K;
  float a0 = 0.f, a1 = 0.f;
  for (int k0 = 0; k0 < K; k0 += 32) {
    __syncthreads();
    for (int e = threadIdx.x; e < TM * 32; e += 256) {
      const int m = e >> 5, k = e & 31, p = start + min(m, n - 1);
      int row = p;
      if (A.tiles && A.x_div) row = A.order[p] / A.x_div;
      xs[m][k] = ((const float*)A.x)[(size_t)row * A.ldx + (A.tiles ? 0 : (size_t)grp * A.xg) + k0 + k];
      w0[m][k] = wg[(size_t)m * K + k0 + k];
      if (PAIR) w1[m][k] = wg[(size_t)(16 + m) * K + k0 + k];
    }
    __syncthreads();
#pragma unroll 8
    for (int k = 0; k < 32; ++k) {
      a0 += xs[tm][k] * w0[tn][k];
      if (PAIR) a1 += xs[tm][k] * w1[tn][k];
    }
  }
  if (tm >= n) return;
  const int p = start + tm;
  const int orow = (A.tiles && A.out_order) ? A.order[p] : p;
  float* o = (float*)A.out + (size_t)orow * A.ldo + (A.tiles ? 0 : (size_t)grp * A.og) + bx * 16 + tn;
  if constexpr (PAIR) {
    const float rw = A.row_w ? A.row_w[A.order[p]] : 1.f;
    *o = glu(a0 * rw, a1 * rw, A);
  } else if constexpr (EPI == GATED || EPI == TABLE) {
    *o = times<EPI>(a0, factor_row<float, EPI>(A, p, grp)[bx * 16 + tn], A);
  } else {
    *o = EPI == RELU2 ? pk::relu2(a0) : a0;
  }
}

// Routing by token id, for every expert layer of the model (blockIdx.x: the layer):
// layer l's table [vocab, top] (int32, at tables + desc[0]) names the token's experts. Rows with
// slot < 0 (padding) are left out. Writes, at the layer's offsets,
//   order[p] = token * top + k, positions sorted by expert;  tiles: at most tm rows of one expert each.
// Bound by a workgroup's instructions and by the wait for an id and then its table row, 1,024 positions at a time. So steps of more
// than one and a half slices of ROUTE_SLICE positions count in one launch, a workgroup a slice, and place in another. 8 layers of 64 experts,
// 6 a token, back to back, us in one launch and in two: 4,096 tokens 35.0, 10.9, 2,048 19.5, 10.5, 1,300 13.5, 10.4, 1,000 (in one) 11.6; in
// a step, whose tables are not in the caches, 4,096 64, 18.
constexpr int ROUTE_DESC = 8;  // {table offset, vocab, top, experts, order offset, tile offset, max tiles, 0}
constexpr int ROUTE_EMAX = 2048, ROUTE_SLICE = 4096;
enum { ROUTE_ALL = 0, ROUTE_COUNT = 1, ROUTE_PLACE = 2 };

template <int PART>
__global__ __launch_bounds__(1024) void table_route_kernel(const int* __restrict__ tables, const int* __restrict__ desc,
                                                           const int* __restrict__ ids, const int* __restrict__ slots,
                                                           int T, int tm, int* __restrict__ order,
                                                           int4* __restrict__ tiles, int* __restrict__ n_tiles,
                                                           int* __restrict__ counts) {  // [layers, slices, ROUTE_EMAX]
  __shared__ int cnt[ROUTE_EMAX], base[ROUTE_EMAX], tbase[ROUTE_EMAX], ws[2][16];
  const int* d = desc + blockIdx.x * ROUTE_DESC;
  const int V = d[1], top = d[2], E = d[3];
  const int* tab = tables + d[0];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  const int p0 = PART == ROUTE_ALL ? 0 : blockIdx.y * ROUTE_SLICE, p1 = PART == ROUTE_ALL ? T * top : min(T * top, p0 + ROUTE_SLICE);
  constexpr int U = PART == ROUTE_ALL ? 1 : ROUTE_SLICE / 1024;
  int* mine = counts + ((size_t)blockIdx.x * gridDim.y + blockIdx.y) * ROUTE_EMAX;
  auto expert = [&](int p) {
    const int t = p / top;
    if (slots[t] < 0) return -1;
    const int e = tab[(size_t)min(max(ids[t], 0), V - 1) * top + (p - t * top)];
    return min(max(e, 0), E - 1);
  };
  if constexpr (PART != ROUTE_PLACE) {
    for (int e = threadIdx.x; e < E; e += 1024) cnt[e] = 0;
    __syncthreads();
#pragma unroll U
    for (int p = p0 + threadIdx.x; p < p1; p += 1024) {
      const int e = expert(p);
      if (e >= 0) atomicAdd(&cnt[e], 1);
    }
    __syncthreads();
  }
  if constexpr (PART == ROUTE_COUNT) {
    for (int e = threadIdx.x; e < E; e += 1024) mine[e] = cnt[e];
    return;
  }
  constexpr int EPT = ROUTE_EMAX / 1024;
  int before[EPT];  // an expert's rows in the slices ahead of this one
  if constexpr (PART == ROUTE_PLACE) {
#pragma unroll
    for (int k = 0; k < EPT; ++k) {
      const int e = threadIdx.x + k * 1024;
      if (e >= E) break;
      int all = 0, ahead = 0;
      const int* from = counts + (size_t)blockIdx.x * gridDim.y * ROUTE_EMAX + e;
#pragma unroll 8
      for (int y = 0; y < (int)gridDim.y; ++y) {
        const int n = from[(size_t)y * ROUTE_EMAX];
        ahead += y < (int)blockIdx.y ? n : 0;
        all += n;
      }
      cnt[e] = all;
      before[k] = ahead;
    }
  }
  // exclusive scans of the row and tile counts, 1,024 experts at a time
  int carry_r = 0, carry_t = 0;
  for (int e0 = 0; e0 < E; e0 += 1024) {
    const int e = e0 + threadIdx.x;
    const int r = e < E ? cnt[e] : 0, q = (r + tm - 1) / tm;
    int sr = r, sq = q;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int a = __shfl_up(sr, o, 64), b = __shfl_up(sq, o, 64);
      if (lane >= o) { sr += a; sq += b; }
    }
    if (lane == 63) { ws[0][wid] = sr; ws[1][wid] = sq; }
    __syncthreads();
    int or_ = carry_r, oq = carry_t, tr = 0, tq = 0;
    for (int w = 0; w < 16; ++w) {
      if (w < wid) { or_ += ws[0][w]; oq += ws[1][w]; }
      tr += ws[0][w];
      tq += ws[1][w];
    }
    if (e < E) { base[e] = or_ + sr - r; tbase[e] = oq + sq - q; }
    carry_r += tr;
    carry_t += tq;
    __syncthreads();
  }
  if (PART == ROUTE_ALL || blockIdx.y == 0) {
    int4* tl = tiles + d[5];
    for (int e = threadIdx.x; e < E; e += 1024)
      for (int i = 0, k = tbase[e]; i < cnt[e]; i += tm, ++k)
        if (k < d[6]) tl[k] = int4{e, base[e] + i, min(tm, cnt[e] - i), 0};
    if (threadIdx.x == 0) n_tiles[blockIdx.x] = min(carry_t, d[6]);
  }
  if constexpr (PART == ROUTE_PLACE)
#pragma unroll
    for (int k = 0; k < EPT; ++k)
      if ((int)threadIdx.x + k * 1024 < E) base[threadIdx.x + k * 1024] += before[k];  // (by the thread that read it for the tiles)
  __syncthreads();
  int* ord = order + d[4];
#pragma unroll U
  for (int p = p0 + threadIdx.x; p < p1; p += 1024) {
    const int e = expert(p);
    if (e >= 0) ord[atomicAdd(&base[e], 1)] = p;
  }
}

}  // namespace gg
}  // namespace pa

// The slices of pa_table_route's counts, each ROUTE_EMAX ints a layer; 0: it needs none. `most`: the largest top of the layers.
extern "C" int pa_table_route_slices(int T, int most) {
  const long long rows = (long long)T * most, n = (rows + pa::gg::ROUTE_SLICE - 1) / pa::gg::ROUTE_SLICE;
  return 2 * rows > 3 * pa::gg::ROUTE_SLICE && n <= 65535 ? (int)n : 0;
}
extern "C" int pa_table_route_counts() { return pa::gg::ROUTE_EMAX; }

extern "C" int pa_table_route(const int* tables, const int* desc, int layers, const int* ids, const int* slots, int T,
                              int tm, int* order, int* tiles, int* n_tiles, int* counts, int slices, hipStream_t st) {
  if (layers <= 0 || T <= 0) return 0;
#define PA_ROUTE(PART, Y)                                                                                                                 \
  hipLaunchKernelGGL((pa::gg::table_route_kernel<pa::gg::PART>), dim3(layers, Y), dim3(1024), 0, st, tables, desc, ids, slots, T, tm, order, \
                     (int4*)tiles, n_tiles, counts)
  if (slices > 0) {
    PA_ROUTE(ROUTE_COUNT, slices);
    PA_ROUTE(ROUTE_PLACE, slices);
  } else {
    PA_ROUTE(ROUTE_ALL, 1);
  }
#undef PA_ROUTE
  return (int)hipGetLastError();
}

// tm: rows per sorted tile (16, 32, 64, 128 or 256; dense: the kernel's choice by row count). always: so many of the last
// groups hold every row (pa_expert_tiles; the others do not look at it)
extern "C" int pa_grouped_gemm(int fp32, const void* x, const void* w, void* out, long long wstride, int groups,
                               int ldx, int xg, int ldo, int og, int rows, int N16, int K32, const int* tiles,
                               int max_tiles, const int* n_tiles, const int* order, int x_div, int out_order, int tm,
                               int epi, float limit, float alpha, float cubic, float bias, const int* positions,
                               const float* cos_sin, int rskip, int r, int rp, int rd, const float* row_w, const void* gate,
                               int ldg, const void* table, const int* ids, int ldt, int tcol, int vocab, const int* skip,
                               const int* live, int always, hipStream_t st) {
  if (skip && (fp32 || tiles || epi == 4)) return -1;
  if (N16 <= 0 || K32 <= 0 || (epi == 1 && N16 % 2)) return -1;
  if (row_w && (!tiles || epi != 1 || !x_div)) return -1;
  if (tiles ? epi > 2 : epi == 1 || epi == 2 || (epi == 3 && !gate) || (epi == 4 && (!table || !ids))) return -1;
  if (tiles ? max_tiles <= 0 : rows <= 0) return 0;
  const pa::gg::Args A{x, w, out, wstride, ldx, xg, ldo, og, rows, N16, K32, (const int4*)tiles, n_tiles,
                       order, x_div, out_order, limit, alpha, cubic, bias, positions, cos_sin, rskip, r, rp, rd,
                       ldo % 8 == 0 && og % 8 == 0 && ((uintptr_t)out & 15) == 0, row_w, gate, table, ids, ldg, ldt, tcol, vocab, skip};
  const int rot = rp > 0 ? 1 : 0;  // one more column of workgroups
  if (fp32) {
    if (tiles && tm != 16) return -2;
    const dim3 grid((epi == 1 ? N16 / 2 : N16) + rot, tiles ? max_tiles : (rows + 15) / 16, tiles ? 1 : groups);
    if (epi == 1) hipLaunchKernelGGL((pa::gg::gemm_f32_kernel<pa::gg::GLU>), grid, dim3(256), 0, st, A);
    else if (epi == 2) hipLaunchKernelGGL((pa::gg::gemm_f32_kernel<pa::gg::RELU2>), grid, dim3(256), 0, st, A);
    else if (epi == 3) hipLaunchKernelGGL((pa::gg::gemm_f32_kernel<pa::gg::GATED>), grid, dim3(256), 0, st, A);
    else if (epi == 4) hipLaunchKernelGGL((pa::gg::gemm_f32_kernel<pa::gg::TABLE>), grid, dim3(256), 0, st, A);
    else hipLaunchKernelGGL((pa::gg::gemm_f32_kernel<pa::gg::PLAIN>), grid, dim3(256), 0, st, A);
    return (int)hipGetLastError();
  }
  if (tiles && tm == 256)
    return pa_expert_tiles(out, x, w, wstride, groups, N16 * 16, K32 * 32, ldx, ldo, tiles, max_tiles, n_tiles, order, x_div,
                           out_order, epi == 1 ? pa::pk::EP_GLU : epi == 2 ? pa::pk::EP_RELU2 : pa::pk::EP_PLAIN, limit, alpha, cubic, bias, row_w, live, always, st);
  if (epi == 4) {  // tiles as large as leave most of the chip busy
#define PA_SK(MT, NT)                                                                                                       \
  do {                                                                                                                      \
    constexpr int lds = 8 * MT * NT * 1024;                                                                                 \
    static bool attr = false;                                                                                               \
    if (!attr) {                                                                                                            \
      (void)hipFuncSetAttribute((const void*)pa::gg::split_k_kernel<MT, NT>, hipFuncAttributeMaxDynamicSharedMemorySize, lds); \
      attr = true;                                                                                                          \
    }                                                                                                                       \
    hipLaunchKernelGGL((pa::gg::split_k_kernel<MT, NT>), dim3(((N16 + NT - 1) / NT * ((rows + 16 * MT - 1) / (16 * MT)) + 7) / 8 * 8), \
                       dim3(512), lds, st, A);                                                                              \
  } while (0)
    auto fills = [&](int t) { return (N16 + t - 1) / t * ((rows + 16 * t - 1) / (16 * t)) >= 192; };
    if (groups != 1) return -1;
    if (fills(4)) PA_SK(4, 4);
    else if (fills(2)) PA_SK(2, 2);
    else PA_SK(1, 1);
#undef PA_SK
    return (int)hipGetLastError();
  }
  if (tiles) return pa::gg::sorted_rows(A, epi, tm, groups, max_tiles, st);
  // dense: 64-row tiles once they fill the chip
  const int head_wgs = (rows + 63) / 64 * groups;
  tm = (N16 + 15) / 16 * ((rows + 63) / 64) * groups < 256 ? 16 : 64;
#define PA_GG(MT, NT, KU, G)                                                                                   \
  hipLaunchKernelGGL((pa::gg::gemm_kernel<MT, NT, KU, G>),                                                     \
                     dim3((N16 + 4 * NT - 1) / (4 * NT) + rot, (rows + 16 * MT - 1) / (16 * MT), groups), dim3(256), 0, st, A)
#define PA_GGK(MT, NT, G)                      \
  do {                                         \
    if (K32 % 4 == 0) PA_GG(MT, NT, 4, G);     \
    else if (K32 % 2 == 0) PA_GG(MT, NT, 2, G);\
    else PA_GG(MT, NT, 1, G);                  \
  } while (0)
  if (tm == 16) {
    if (epi == 3) PA_GGK(1, 1, pa::gg::GATED);
    else PA_GGK(1, 1, pa::gg::PLAIN);
  } else if (K32 <= pa::gg::HEAD_K32 && N16 >= 16 && head_wgs >= 512 &&
             (epi != 3 || head_wgs <= 768 || (K32 == 8 && N16 <= 32))) {
    const dim3 grid((rows + 63) / 64, groups);
    const int lds = 4 * K32 * pa::gg::HEAD_UNIT;
    if (epi == 3) hipLaunchKernelGGL((pa::gg::head_rows_kernel<pa::gg::GATED>), grid, dim3(256), lds, st, A);
    else hipLaunchKernelGGL((pa::gg::head_rows_kernel<pa::gg::PLAIN>), grid, dim3(256), lds, st, A);
  } else {
    if (epi == 3) PA_GG(4, 4, 1, pa::gg::GATED);
    else PA_GG(4, 4, 1, pa::gg::PLAIN);
  }
#undef PA_GGK
#undef PA_GG
  return (int)hipGetLastError();
}
