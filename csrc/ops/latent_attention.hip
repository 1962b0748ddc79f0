// Paged latent attention (queries absorbed into the latent space), for prefill chunks, decode
// rows and mixed batches in one launch.
//
// The cache holds one row per token for all heads: [latent c (Rp) | rotated key part (rp)],
// D = Rp + rp (rp 0: a latent without positions), pages of 16 tokens, fragment-major [D/8][16][8] (latent_cache.hip). With
//   q~_h = [W_uk,h^T q_h | rot(q_h)]          (absorbed before the launch)
//   score_h(i, j) = q~_h(i) . row(j) * scale,  o~_h(i) = sum_j softmax_j score * c(j)
// every head reads the same rows: keys are the whole row, values its first Rp dims, and the
// W_uv up-projection of o~ follows the launch. The MFMA columns are (token, head) pairs,
// consecutive rows of q~ [T, H, D], so any head count fills them.
//
//   S^T[keys x cols] = rows . Q^T      A = key rows (one 1-KB run of a page per k-step), B = Q^T
//   O^T[dims x cols] += c^T . P^T      A = c^T by LDS transpose reads (ds_read_b64_tr_b16) of the
//                                      SAME tile, B = P^T = the S^T accumulator's own registers
// so the rows are read from HBM once and stored once; no transposed copy exists anywhere.
//
// A window of W keys (0: none) limits position i to keys i - W + 1 .. i: tiles wholly outside an
// item's range are never read.
//
// Items come from the scheduler like paged_attention's (seq, q_begin, nq | part<<8 | nparts<<20,
// partial slot):
//   nq <= dec_tokens: split over keys. The 8 waves take every 8th page with a private LDS tile and
//                     merge; nparts > 1 divides the item's own (windowed) key range evenly, the
//                     partials go to memory and merge_kernel, a second launch, combines them: at
//                     16 x Rp floats a partition, one last arriver would read for longer than all
//                     partitions compute, while the launch spreads the columns over the chip.
//   otherwise:        128 columns per workgroup, 16 per wave; all waves share double-buffered 32-key
//                     tiles that arrive by direct global -> LDS loads. A step with few such items
//                     has them cut into partitions of their keys too (8 slots each).
//
// Steps of few tokens have the heads' products with W_uv behind the merge in the same launch (merge_heads_kernel).
//
// Prompt portions of the widest latents have a second form (latent_expand.h), whose units the same launches run.
#include "common.h"
#include "latent_expand.h"

#include <algorithm>
#include <type_traits>

namespace pa {
namespace la {

constexpr float NEG_BIG = -1.0e30f;
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) bf16x4 lds_bf16x4;
typedef __attribute__((address_space(3))) void lds_void;
typedef const __attribute__((address_space(1))) void glb_void;

struct Args {
  void* out;             // [T, H, Rp]
  float* part_o;         // [slots, NB, 16, Rp]
  float* part_ml;        // [slots, NB, 16, 2]
  const void* q;         // [T, H, D]
  const void* pages;
  const int4* items;
  const int* n_items;
  const int *q_start, *q_len, *ctx_len, *block_table;
  int max_blocks, H, NB, Rp, D, dec_tokens, window;
  float scale_log2;
  Expand X;
};

// requests whose keys are expanded take no part in the absorbed form
template <bool XP>
__device__ __forceinline__ bool expanded(const Args& A, int s) { return XP && A.X.base[s] != X_NONE; }

// ---------------------------------------------------------------------------
// Any sizes, bf16 or fp32: one workgroup per (token of an item, head). The exact path.
template <typename T>
__global__ __launch_bounds__(256) void simple_kernel(const Args A) {
  extern __shared__ __attribute__((aligned(16))) float sm[];
  float* sq = sm;           // D
  float* sp = sm + A.D;     // 256
  float* red = sp + 256;    // 4
  const int h = blockIdx.x, n = A.n_items[0];
  for (int item = blockIdx.y; item < n; item += gridDim.y) {
    const int4 it = A.items[item];
    const int s = it.x, nq = it.z & 0xff, part = (it.z >> 8) & 0xfff;
    if (part > 0) continue;  // partition 0 takes the whole range
    const int ctx = A.ctx_len[s], ql = A.q_len[s];
    const int* bt = A.block_table + (size_t)s * A.max_blocks;
    for (int i = 0; i < nq; ++i) {
      const int tok = it.y + i, pos = ctx - ql + tok;
      const int lo = A.window > 0 ? max(0, pos - A.window + 1) : 0;
      const size_t row = (size_t)(A.q_start[s] + tok) * A.H + h;
      __syncthreads();
      for (int d = threadIdx.x; d < A.D; d += 256) sq[d] = (float)((const T*)A.q)[row * A.D + d];
      __syncthreads();
      float m = NEG_BIG, l = 0.f, o[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
      for (int k0 = lo; k0 <= pos; k0 += 256) {
        const int key = k0 + threadIdx.x;
        float sc = NEG_BIG;
        if (key <= pos) {
          const T* kr = (const T*)A.pages + (size_t)bt[key >> 4] * A.D * 16 + (key & 15) * 8;
          float a = 0.f;
          for (int d = 0; d < A.D; d += 8)
#pragma unroll
            for (int j = 0; j < 8; ++j) a += sq[d + j] * (float)kr[(size_t)d * 16 + j];
          sc = a * A.scale_log2;
        }
        const float wm = wave_max(sc);
        if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = wm;
        __syncthreads();
        const float mn = fmaxf(m, fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3])));
        const float alpha = exp2f(m - mn), p = key <= pos ? exp2f(sc - mn) : 0.f;
        m = mn;
        sp[threadIdx.x] = p;
        __syncthreads();
        l = l * alpha + block_sum<4>(p, red);
        const int nk = min(256, pos + 1 - k0);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int d = threadIdx.x + 256 * e;
          if (d >= A.Rp) break;
          float a = o[e] * alpha;
          for (int k = 0; k < nk; ++k) {
            const int kk = k0 + k;
            a += sp[k] * (float)((const T*)A.pages)[(size_t)bt[kk >> 4] * A.D * 16 + (size_t)(d >> 3) * 128 +
                                                    (kk & 15) * 8 + (d & 7)];
          }
          o[e] = a;
        }
        __syncthreads();
      }
      const float inv = 1.f / l;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int d = threadIdx.x + 256 * e;
        if (d < A.Rp) ((T*)A.out)[row * A.Rp + d] = (T)(o[e] * inv);
      }
    }
  }
}

// ---------------------------------------------------------------------------
// c^T operand: lanes 16g + i of the result hold dim i of keys 4g .. 4g + 3; each lane names the
// 8 bytes (key 4g + i/4, dims 4 (i%4) .. + 3) of the 4 x 16 block its group transposes
__device__ __forceinline__ bf16x4 tr_read(const char* p) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)p);
}
// The same for pair_item: without alias information the compiler waits there for the direct loads to LDS in flight. (In
// split_item and tile_item it only orders the loop differently: 192 + 64, 4,096 tokens 171 us, without it 167.)
__device__ __forceinline__ bf16x4 tr_read_ahead(const char* __restrict__ p) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)p);
}

constexpr int NW = 8;          // waves per workgroup: two a SIMD, one's softmax under the other's MFMAs
constexpr int MERGE_LD = 132;  // floats per merge row of 128 dims

template <int RT, int PT>
__device__ __forceinline__ void split_item(const Args& A, const int4 it, char* smem) {
  constexpr int NK = RT + PT, D = 32 * NK, RP = 32 * RT;
  const int s = it.x, qb = it.y, nq = it.z & 0xff, part = (it.z >> 8) & 0xfff, nparts = it.z >> 20, pidx = it.w;
  const int cb = blockIdx.x, cols = nq * A.H;
  if (cb * 16 >= cols) return;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, g = lane >> 4, c = lane & 15;
  const int ctx = A.ctx_len[s], ql = A.q_len[s];
  const int pos0 = ctx - ql + qb;
  const int ci = cb * 16 + c;
  const int cpos = pos0 + min(ci, cols - 1) / A.H;  // this column's position
  const int klo = A.window > 0 ? max(0, cpos - A.window + 1) : 0;
  const size_t row0 = (size_t)(A.q_start[s] + qb) * A.H + cb * 16;  // q~ row of column 0
  const size_t row = row0 + min(c, cols - 1 - cb * 16);
  // the item's pages, and this partition's share
  const int p_lo = (A.window > 0 ? max(0, pos0 - A.window + 1) : 0) >> 4, p_hi = (pos0 + nq + 15) >> 4;
  const int per = (p_hi - p_lo + nparts - 1) / nparts;
  const int p_begin = p_lo + part * per, p_end = min(p_hi, p_begin + per);
  const int* bt = A.block_table + (size_t)s * A.max_blocks;

  constexpr bool AHEAD = RT < 16;
  bf16x8 kf[NK];
  auto load = [&](int p, bf16x8 (&k)[NK]) {
    const bf16* b = (const bf16*)A.pages + (size_t)bt[p] * (D * 16) + (g * 16 + c) * 8;
#pragma unroll
    for (int m = 0; m < NK; ++m) k[m] = *reinterpret_cast<const bf16x8*>(b + m * 512);
  };
  // the wave's first page is under way while the queries are staged
  if (AHEAD && p_begin + wid < p_end) load(p_begin + wid, kf);
  // all waves share the 16 columns: their Q^T operands (1 KB per k-step) live in LDS
  char* sq = smem + NW * (RP * 32);
  for (int m = wid; m < NK; m += NW)
    *reinterpret_cast<bf16x8*>(sq + m * 1024 + (g * 16 + c) * 16) =
        *reinterpret_cast<const bf16x8*>((const bf16*)A.q + row * D + 32 * m + 8 * g);
  __syncthreads();
  f32x4 o[2 * RT];
#pragma unroll
  for (int n = 0; n < 2 * RT; ++n) o[n] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m_run = NEG_BIG, l_run = 0.f;
  char* my = smem + wid * (RP * 32);  // 16 keys x RP dims
  const int loff = (g * 16 + c) * 16;  // this lane's 16 B of a k-step
  const int toff = ((c & 3) >> 1) * 256 + (4 * g + (c >> 2)) * 16 + (c & 1) * 8;

  // the widest latents load a later page when they need it: it does not fit the registers beside the
  // outputs' update, and the SIMD's other wave computes meanwhile
  for (int p = p_begin + wid; p < p_end; p += NW) {
    if (!AHEAD) load(p, kf);
    f32x4 sc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int m = 0; m < NK; ++m) {
      const bf16x8 qf = *reinterpret_cast<const bf16x8*>(sq + m * 1024 + loff);
      sc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[m], qf, sc, 0, 0, 0);
      if (m < RT) *reinterpret_cast<bf16x8*>(my + m * 1024 + loff) = kf[m];
    }
    if (AHEAD && p + NW < p_end) load(p + NW, kf);
    float tmax = NEG_BIG;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int key = 16 * p + 4 * g + r;
      sc[r] = (key <= cpos && key >= klo) ? sc[r] * A.scale_log2 : NEG_BIG;
      tmax = fmaxf(tmax, sc[r]);
    }
    tmax = fmaxf(tmax, __shfl_xor(tmax, 16, 64));
    tmax = fmaxf(tmax, __shfl_xor(tmax, 32, 64));
    const float m_new = fmaxf(m_run, tmax);
    if (__any(m_new > m_run)) {
      const float alpha = exp2f(m_run - m_new);
      l_run *= alpha;
#pragma unroll
      for (int n = 0; n < 2 * RT; ++n) o[n] *= alpha;
      m_run = m_new;
    }
    bf16x4 pf;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float e = exp2f(sc[r] - m_run);
      l_run += e;
      pf[r] = (bf16)e;
    }
    // the tile is private to the wave: its LDS operations complete in order
    const s16x4 pb = __builtin_bit_cast(s16x4, pf);
#pragma unroll
    for (int n = 0; n < 2 * RT; ++n) {
      const s16x4 v = __builtin_bit_cast(s16x4, tr_read(my + n * 512 + toff));
      o[n] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(v, pb, o[n], 0, 0, 0);
    }
  }
  l_run += __shfl_xor(l_run, 16, 64);
  l_run += __shfl_xor(l_run, 32, 64);

  // merge the waves, 128 dims at a time
  float* mo = reinterpret_cast<float*>(smem);                           // [NW][16][MERGE_LD]
  float* mm = reinterpret_cast<float*>(smem + NW * 16 * MERGE_LD * 4);  // [NW][16]
  float* ml = mm + NW * 16;
  __syncthreads();
  if (g == 0) {
    mm[wid * 16 + c] = m_run;
    ml[wid * 16 + c] = l_run;
  }
  const int ccol = threadIdx.x >> 5, d4 = (threadIdx.x & 31) * 4;
  const bool cvalid = cb * 16 + ccol < cols;
  float wgt[NW], L = 0.f, mt = NEG_BIG;
#pragma unroll
  for (int nb = 0; nb < (RT + 3) / 4; ++nb) {
    if (nb) __syncthreads();
#pragma unroll
    for (int n = 0; n < 8; ++n)
      if (nb * 8 + n < 2 * RT) *reinterpret_cast<f32x4*>(mo + (wid * 16 + c) * MERGE_LD + 16 * n + 4 * g) = o[nb * 8 + n];
    __syncthreads();
    if (nb == 0) {
#pragma unroll
      for (int w = 0; w < NW; ++w) mt = fmaxf(mt, mm[w * 16 + ccol]);
#pragma unroll
      for (int w = 0; w < NW; ++w) {
        wgt[w] = exp2f(mm[w * 16 + ccol] - mt);
        L += wgt[w] * ml[w * 16 + ccol];
      }
    }
    const int d0 = nb * 128 + d4;
    if (d0 < RP) {
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int w = 0; w < NW; ++w)
        acc += wgt[w] * *reinterpret_cast<const f32x4*>(mo + (w * 16 + ccol) * MERGE_LD + d4);
      if (nparts > 1) {
        *reinterpret_cast<f32x4*>(A.part_o + (((size_t)pidx * A.NB + cb) * 16 + ccol) * RP + d0) = acc;
      } else if (cvalid) {
        const float inv = 1.f / L;
        bf16x4 v;
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = (bf16)(acc[j] * inv);
        *reinterpret_cast<bf16x4*>((bf16*)A.out + (row0 + ccol) * RP + d0) = v;
      }
    }
  }
  if (nparts > 1 && (threadIdx.x & 31) == 0)
    reinterpret_cast<float2*>(A.part_ml)[((size_t)pidx * A.NB + cb) * 16 + ccol] = float2{mt, L};
}

// The partitions of the expanded units. Each part of a tile merges its share of the tile's tokens (groups of four, in turn), a wave
// four tokens of a head, two at a time with 4 dims a lane: all parts' loads of a wave are under way at once. Four tiles in four parts (499 tokens
// after 3,584), 17 MB: with a wave a token of the first parts, the others idle, 11.6 us, so 8.2 (a launch that finds none takes 4.7).
__device__ __forceinline__ void merge_expanded(const Args& A) {
  constexpr int TOK = 4, UNITS = X_COLS / TOK;
  const int lane = threadIdx.x & 63, n = A.X.counts[0] * A.H * UNITS, half = lane >> 5, d = 4 * (lane & 31);
  const int waves = gridDim.x * gridDim.y * 4, w0 = (blockIdx.y * gridDim.x + blockIdx.x) * 4 + (threadIdx.x >> 6);
  for (int w = __builtin_amdgcn_readfirstlane(w0); w < n; w += waves) {
    const int4 it = A.X.att[w / (A.H * UNITS)];
    const int rest = w % (A.H * UNITS), h = rest / UNITS, unit = rest % UNITS, part = it.z & 0xffff, parts = it.z >> 16;
    if (parts <= 1 || unit % parts != part) continue;
    const int left = A.q_len[it.x] - it.y * X_COLS - unit * TOK;  // tokens from the unit's first on
    if (left <= 0) continue;
    const size_t at = (size_t)it.w * A.H * X_COLS + h * X_COLS + unit * TOK, step = (size_t)A.H * X_COLS;
    float2 ml[TOK / 2][X_PARTS];
    f32x4 o[TOK / 2][X_PARTS];
#pragma unroll
    for (int j = 0; j < TOK / 2; ++j) {
      const size_t row = at + min(2 * j + half, left - 1);
#pragma unroll
      for (int p = 0; p < X_PARTS; ++p) {  // (behind the last part: its values again)
        const size_t slot = row + min(p, parts - 1) * step;
        ml[j][p] = reinterpret_cast<const float2*>(A.X.part_ml)[slot];
        o[j][p] = *reinterpret_cast<const f32x4*>(A.X.part_o + slot * X_DIM + d);
      }
    }
#pragma unroll
    for (int j = 0; j < TOK / 2; ++j) {
      float m = NEG_BIG, L = 0.f;
      f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int p = 0; p < X_PARTS; ++p) m = fmaxf(m, ml[j][p].x);
#pragma unroll
      for (int p = 0; p < X_PARTS; ++p) {
        // (written out: left to the compiler, the unrolled sums of products are rounded in other places than one after the other)
        const float f = exp2f(ml[j][p].x - m);
        L = p < parts ? fmaf(f, ml[j][p].y, L) : L;
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = p < parts ? fmaf(f, o[j][p][r], v[r]) : v[r];
      }
      if (2 * j + half >= left) continue;
      const float inv = 1.f / L;
      bf16x4 b;
#pragma unroll
      for (int r = 0; r < 4; ++r) b[r] = (bf16)(v[r] * inv);
      *reinterpret_cast<bf16x4*>((bf16*)A.X.out + (size_t)(A.q_start[it.x] + it.y * X_COLS + unit * TOK + 2 * j + half) * A.X.ldo + h * X_DIM + d) = b;
    }
  }
}

// The partitions of an item, merged: a wave per (item, column), 8 dims per lane and step.
template <int RT, bool XP = false>
__global__ __launch_bounds__(256) void merge_kernel(const Args A) {
  constexpr int RP = 32 * RT;
  const int lane = threadIdx.x & 63;
  const int n = A.n_items[0];
  if constexpr (XP) merge_expanded(A);
  for (int item = blockIdx.y; item < n; item += gridDim.y) {
    const int4 it = A.items[item];
    const int nq = it.z & 0xff, nparts = it.z >> 20;
    if (nparts <= 1 || ((it.z >> 8) & 0xfff) != 0 || expanded<XP>(A, it.x)) continue;
    const int step = nq <= A.dec_tokens ? 1 : 8;  // slots of a partition
    for (int col = blockIdx.x * 4 + (threadIdx.x >> 6); col < nq * A.H; col += gridDim.x * 4) {
      auto slot = [&](int p) { return (size_t)(it.w + p * step) * A.NB * 16 + col; };
      const float2* ml = reinterpret_cast<const float2*>(A.part_ml);
      // lane p holds partition p's weight (64 at a time): the loads of a round are independent
      float gm = NEG_BIG, L = 0.f;
      for (int p0 = 0; p0 < nparts; p0 += 64) gm = fmaxf(gm, p0 + lane < nparts ? ml[slot(p0 + lane)].x : NEG_BIG);
      gm = wave_max(gm);
      float a[(RP + 511) / 512][8];
#pragma unroll
      for (int e = 0; e < (RP + 511) / 512; ++e)
#pragma unroll
        for (int j = 0; j < 8; ++j) a[e][j] = 0.f;
      for (int p0 = 0; p0 < nparts; p0 += 64) {
        float w = 0.f;
        if (p0 + lane < nparts) {
          const float2 v = ml[slot(p0 + lane)];
          w = exp2f(v.x - gm);
          L += w * v.y;
        }
        const int np = min(64, nparts - p0);
#pragma unroll 8
        for (int p = 0; p < np; ++p) {
          const float wp = __shfl(w, p, 64);
#pragma unroll
          for (int e = 0; e < (RP + 511) / 512; ++e) {
            const int d = min(e * 512 + lane * 8, RP - 8);
            const f32x4* s = reinterpret_cast<const f32x4*>(A.part_o + slot(p0 + p) * RP + d);
            const f32x4 x = s[0], y = s[1];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              a[e][j] += wp * x[j];
              a[e][4 + j] += wp * y[j];
            }
          }
        }
      }
      L = wave_sum(L);
      const float inv = 1.f / L;
      bf16* o = (bf16*)A.out + ((size_t)(A.q_start[it.x] + it.y) * A.H + col) * RP;
#pragma unroll
      for (int e = 0; e < (RP + 511) / 512; ++e) {
        const int d = e * 512 + lane * 8;
        if (d < RP) {
          bf16x8 v;
#pragma unroll
          for (int j = 0; j < 8; ++j) v[j] = (bf16)(a[e][j] * inv);
          *reinterpret_cast<bf16x8*>(o + d) = v;
        }
      }
    }
  }
}

template <int RT, int PT, int CT>
__device__ __forceinline__ void tile_item(const Args& A, const int4 it, char* smem) {
  constexpr int NK = RT + PT, D = 32 * NK, RP = 32 * RT, TILE = 32 * D * 2;
  const int s = it.x, qb = it.y, nq = it.z & 0xff, part = (it.z >> 8) & 0xfff, nparts = it.z >> 20;
  const int cols = nq * A.H, cw = blockIdx.x * (16 * NW * CT);
  if (cw >= cols) return;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, g = lane >> 4, c = lane & 15;
  const int ctx = A.ctx_len[s], ql = A.q_len[s];
  const int pos0 = ctx - ql + qb;
  const size_t row0 = (size_t)(A.q_start[s] + qb) * A.H;
  const int* bt = A.block_table + (size_t)s * A.max_blocks;
  int ci[CT], cpos[CT], klo[CT];
  const int loff = (g * 16 + c) * 16;
  bf16x8 qf[CT][NK];
#pragma unroll
  for (int t = 0; t < CT; ++t) {
    ci[t] = cw + (wid * CT + t) * 16 + c;
    const int cc = min(ci[t], cols - 1);
    cpos[t] = pos0 + cc / A.H;
    klo[t] = A.window > 0 ? max(0, cpos[t] - A.window + 1) : 0;
#pragma unroll
    for (int m = 0; m < NK; ++m)
      qf[t][m] = *reinterpret_cast<const bf16x8*>((const bf16*)A.q + (row0 + cc) * D + 32 * m + 8 * g);
  }
  // positions of the workgroup's columns -> its key tiles
  const int f = pos0 + cw / A.H, e = pos0 + min(cw + 16 * NW * CT - 1, cols - 1) / A.H;
  int t_lo = (A.window > 0 ? max(0, f - A.window + 1) : 0) >> 5, t_hi = (e + 32) >> 5;
  if (nparts > 1) {  // this partition's tiles (possibly none)
    const int per = (t_hi - t_lo + nparts - 1) / nparts;
    t_lo += part * per;
    t_hi = min(t_hi, t_lo + per);
  }
  const int nblk = (ctx + 15) >> 4;
  // this wave's columns: keys below all of their windows' starts / above all positions are masked
  // (t needs no mask when every column sees all its 32 keys)
  const int wf = pos0 + min(cw + wid * CT * 16, cols - 1) / A.H;
  const int we = pos0 + min(cw + wid * CT * 16 + 16 * CT - 1, cols - 1) / A.H;
  const int full_lo = A.window > 0 ? we - A.window + 1 : 0, full_hi = wf;

  f32x4 o[CT][2 * RT];
#pragma unroll
  for (int t = 0; t < CT; ++t)
#pragma unroll
    for (int n = 0; n < 2 * RT; ++n) o[t][n] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m_run[CT], l_run[CT];
#pragma unroll
  for (int t = 0; t < CT; ++t) {
    m_run[t] = NEG_BIG;
    l_run[t] = 0.f;
  }
  // direct loads: the tile is two whole pages, copied linearly, 1 KB per wave and instruction
  auto issue = [&](int t, char* dst) {
    const bf16* src0 = (const bf16*)A.pages + (size_t)bt[min(2 * t, nblk - 1)] * (D * 16) + lane * 8;
    const bf16* src1 = (const bf16*)A.pages + (size_t)bt[min(2 * t + 1, nblk - 1)] * (D * 16) + lane * 8;
#pragma unroll
    for (int i = 0; i < (2 * NK + NW - 1) / NW; ++i) {
      const int ch = i * NW + wid;  // wave-uniform
      if (2 * NK % NW == 0 || ch < 2 * NK)
        __builtin_amdgcn_global_load_lds((glb_void*)((ch < NK ? src0 : src1 - NK * 512) + ch * 512),
                                         (lds_void*)(dst + ch * 1024), 16, 0, 0);
    }
  };
  const int toff = ((c & 3) >> 1) * 256 + (4 * g + (c >> 2)) * 16 + (c & 1) * 8;
  if (t_lo < t_hi) issue(t_lo, smem);
  for (int t = t_lo; t < t_hi; ++t) {
    char* cur = smem + ((t - t_lo) & 1) * TILE;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();  // tile t is whole, and nobody reads the other buffer any more
    if (t + 1 < t_hi) issue(t + 1, smem + ((t + 1 - t_lo) & 1) * TILE);
    f32x4 sc[CT][2];
#pragma unroll
    for (int x = 0; x < CT; ++x)
#pragma unroll
      for (int k = 0; k < 2; ++k) sc[x][k] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int m = 0; m < NK; ++m)
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const bf16x8 kf = *reinterpret_cast<const bf16x8*>(cur + k * (D * 32) + m * 1024 + loff);
#pragma unroll
        for (int x = 0; x < CT; ++x) sc[x][k] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qf[x][m], sc[x][k], 0, 0, 0);
      }
    const bool mask = 32 * t < full_lo || 32 * t + 31 > full_hi;  // wave-uniform
    bf16x8 pf[CT];
#pragma unroll
    for (int x = 0; x < CT; ++x) {
      if (mask) {
#pragma unroll
        for (int k = 0; k < 2; ++k)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int key = 32 * t + 16 * k + 4 * g + r;
            if (key > cpos[x] || key < klo[x]) sc[x][k][r] = NEG_BIG;
          }
      }
      float tmax = NEG_BIG;
#pragma unroll
      for (int k = 0; k < 2; ++k)
#pragma unroll
        for (int r = 0; r < 4; ++r) tmax = fmaxf(tmax, sc[x][k][r]);
      tmax = fmaxf(tmax, __shfl_xor(tmax, 16, 64));
      tmax = fmaxf(tmax, __shfl_xor(tmax, 32, 64));
      const float m_new = fmaxf(m_run[x], fmaxf(tmax * A.scale_log2, NEG_BIG));
      if (__any(m_new > m_run[x])) {
        const float alpha = exp2f(m_run[x] - m_new);
        l_run[x] *= alpha;
#pragma unroll
        for (int n = 0; n < 2 * RT; ++n) o[x][n] *= alpha;
        m_run[x] = m_new;
      }
      // a column that has seen no key yet (its window starts in a later tile): every weight is 0
      const float nm = m_run[x] < 0.01f * NEG_BIG ? 0.f : -m_run[x];
#pragma unroll
      for (int k = 0; k < 2; ++k)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float p = __builtin_amdgcn_exp2f(fmaf(sc[x][k][r], A.scale_log2, nm));
          l_run[x] += p;
          pf[x][4 * k + r] = (bf16)p;
        }
    }
#pragma unroll
    for (int n = 0; n < 2 * RT; ++n) {
      const bf16x4 v0 = tr_read(cur + n * 512 + toff), v1 = tr_read(cur + D * 32 + n * 512 + toff);
      bf16x8 v;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        v[j] = v0[j];
        v[4 + j] = v1[j];
      }
#pragma unroll
      for (int x = 0; x < CT; ++x) o[x][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v, pf[x], o[x][n], 0, 0, 0);
    }
  }
#pragma unroll
  for (int x = 0; x < CT; ++x) {
    float l = l_run[x];
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);
    if (ci[x] >= cols) continue;
    if (nparts > 1) {  // 8 slots hold the item's columns in a row
      const size_t pc = (size_t)it.w * A.NB * 16 + ci[x];
      float* po = A.part_o + pc * RP + 4 * g;
#pragma unroll
      for (int n = 0; n < 2 * RT; ++n) *reinterpret_cast<f32x4*>(po + 16 * n) = o[x][n];
      if (g == 0) reinterpret_cast<float2*>(A.part_ml)[pc] = float2{m_run[x], l};
      continue;
    }
    const float inv = 1.f / l;
    bf16* orow = (bf16*)A.out + (row0 + ci[x]) * RP + 4 * g;
#pragma unroll
    for (int n = 0; n < 2 * RT; ++n) {
      bf16x4 v;
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = (bf16)(o[x][n][r] * inv);
      *reinterpret_cast<bf16x4*>(orow + 16 * n) = v;
    }
  }
}

// The same for the widest latents, whose tile loop is bound by LDS reads: there every wave reads the whole tile for its own
// 16 columns, 68 KB for 68 MFMAs. Here two waves share 32 columns. Each takes half the dimensions of the scores (its
// half of the queries fits the registers) and half the dimensions of the outputs, of both column blocks, so a fragment
// read serves two MFMAs: 40 KB a wave. Between the halves, a wave sends the partner its part of the
// partner's scores and gets its own completed, does the softmax of its 16 columns, and the two trade weights. The
// next tile's scores run ahead of this tile's outputs (three tile buffers), so softmax and outputs overlap.
// 4,096 tokens, 16 heads, 512 + 64: 425 -> 318 us; the MFMAs alone, at 2,176 cycles a tile and CU, 116 us: with two
// waves a SIMD and two barriers a tile, scores, outputs, softmax and loads overlap little. Reads 2, 3, 4 steps ahead: 324,
// 318, 321 us, and 4 prompts of 1,024 115, 114, 118: at 4 the registers end. The subtracted maximum is the true one of the
// keys so far: the largest weight is then exactly 1 and, in 16 bits, has no rounding of its own (letting it fall behind
// saves 10 us of rescaling, and peaked rows err up to twice as much). Of a pair's two blocks only the one whose maximum
// moved is rescaled (both together: 337 us).
template <int RT, int PT>
constexpr int pair_lds_bytes() { return 3 * 32 * 32 * (RT + PT) * 2 + NW * (2048 + 2 * (1024 + 64) + 2048); }

template <int RT, int PT>
__device__ __forceinline__ void pair_item(const Args& A, const int4 it, char* smem) {
  constexpr int NK = RT + PT, NH = (NK + 1) / 2, D = 32 * NK, RP = 32 * RT, TILE = 32 * D * 2;
  const int s = it.x, qb = it.y, nq = it.z & 0xff, part = (it.z >> 8) & 0xfff, nparts = it.z >> 20;
  const int cols = nq * A.H, cw = blockIdx.x * (16 * NW);
  if (cw >= cols) return;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, g = lane >> 4, c = lane & 15;
  const int half = __builtin_amdgcn_readfirstlane(wid & 1);
  const int ctx = A.ctx_len[s], ql = A.q_len[s];
  const int pos0 = ctx - ql + qb;
  const size_t row0 = (size_t)(A.q_start[s] + qb) * A.H;
  const int* bt = A.block_table + (size_t)s * A.max_blocks;
  // column block 0: this wave's own, 1: the partner's
  auto col = [&](int x) { return cw + (x ? wid ^ 1 : wid) * 16 + c; };
  const int cpos = pos0 + min(col(0), cols - 1) / A.H;
  const int klo = A.window > 0 ? max(0, cpos - A.window + 1) : 0;
  const int loff = (g * 16 + c) * 16;
  // (the queries of a wave's last step stay in LDS: with them in registers the tile loop spills)
  constexpr int NQ = NH - 1;
  char* qs = smem + 3 * TILE + NW * (2048 + 2 * (1024 + 64)) + wid * 2048 + loff;
  bf16x8 qf[2][NQ];
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int m = 0; m < NH; ++m) {
      const int mm = half * NH + m;
      const bf16* src = (const bf16*)A.q + (row0 + min(col(x), cols - 1)) * D + 32 * min(mm, NK - 1) + 8 * g;
      bf16x8 v = *reinterpret_cast<const bf16x8*>(src);
      if (2 * NH != NK && mm >= NK) v = bf16x8{};  // (an odd number of steps: none is left for the second half)
      if (m < NQ) qf[x][m < NQ ? m : 0] = v;
      else *reinterpret_cast<bf16x8*>(qs + x * 1024) = v;
    }
  const int f = pos0 + cw / A.H, e = pos0 + min(cw + 16 * NW - 1, cols - 1) / A.H;
  int t_lo = (A.window > 0 ? max(0, f - A.window + 1) : 0) >> 5, t_hi = (e + 32) >> 5;
  if (nparts > 1) {  // this partition's tiles (possibly none)
    const int per = (t_hi - t_lo + nparts - 1) / nparts;
    t_lo += part * per;
    t_hi = min(t_hi, t_lo + per);
  }
  const int nblk = (ctx + 15) >> 4, n_t = t_hi - t_lo;
  // (t needs no mask when every column of the wave sees all its 32 keys)
  const int wf = pos0 + min(cw + wid * 16, cols - 1) / A.H, we = pos0 + min(cw + wid * 16 + 15, cols - 1) / A.H;
  const int full_lo = A.window > 0 ? we - A.window + 1 : 0, full_hi = wf;

  f32x4 o[2][RT];
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int n = 0; n < RT; ++n) o[x][n] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m_run = NEG_BIG, l_run = 0.f;
  char* xs = smem + 3 * TILE;                                    // [NW][2][1 KB] scores for the partner
  char* xp = xs + NW * 2048;                                     // [2][NW][1 KB] weights, of tiles in turn
  float* xa = reinterpret_cast<float*>(xp + 2 * NW * 1024);      // [2][NW][16] factors of the outputs so far
  // page ids, 64 at a time, a lane each: read where they are used, their latency was a stall of every tile
  const int swid = __builtin_amdgcn_readfirstlane(wid), grp = swid >> 2;
  int ids = 0, ids_at = -64;
  auto issue = [&](int t, char* dst) {
    if (2 * t >= ids_at + 64) {  // uniform
      ids_at = 2 * t;
      ids = bt[min(2 * t + lane, nblk - 1)];
    }
    const int i0 = __builtin_amdgcn_readlane(ids, 2 * t - ids_at), i1 = __builtin_amdgcn_readlane(ids, 2 * t + 1 - ids_at);
    const char* src0 = (const char*)A.pages + (size_t)i0 * (D * 32);
    const char* src1 = (const char*)A.pages + (size_t)i1 * (D * 32) - NK * 1024;
#pragma unroll
    for (int i = 0; i < (2 * NK + NW - 1) / NW; ++i) {
      const int ch = i * NW + swid;
      if (2 * NK % NW == 0 || ch < 2 * NK)
        __builtin_amdgcn_global_load_lds((glb_void*)((ch < NK ? src0 : src1) + ch * 1024 + lane * 16),
                                         (lds_void*)(dst + ch * 1024), 16, 0, 0);
    }
  };
  const int toff = half * (RT * 512) + ((c & 3) >> 1) * 256 + (4 * g + (c >> 2)) * 16 + (c & 1) * 8;
  f32x4 sc[2];
  // both column blocks' scores over this half of the dimensions; the partner's go to LDS. Fragments are read AHEAD steps
  // before their use: left to itself the compiler, short of registers, reads each right before its MFMAs.
  constexpr int AHEAD = 3;
  auto scores = [&](const char* tile) {
    bf16x8 kb[AHEAD + 1];
    auto frag = [&](int i) {
      const int k = i / NH, m = i % NH, mm = 2 * NH == NK ? half * NH + m : min(half * NH + m, NK - 1);
      bf16x8 v = *reinterpret_cast<const bf16x8*>(tile + k * (D * 32) + mm * 1024 + loff);
      if (2 * NH != NK && m == NH - 1 && half) v = bf16x8{};
      return v;
    };
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) kb[i] = frag(i);
    f32x4 other = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < 2 * NH; ++i) {
      __builtin_amdgcn_sched_barrier(0);
      const int k = i / NH, m = i % NH;
      if (m == 0) other = sc[k] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (i + AHEAD < 2 * NH) kb[(i + AHEAD) % (AHEAD + 1)] = frag(i + AHEAD);
      __builtin_amdgcn_sched_barrier(0);
      const bf16x8 q0 = m < NQ ? qf[0][m < NQ ? m : 0] : *reinterpret_cast<const bf16x8*>(qs);
      const bf16x8 q1 = m < NQ ? qf[1][m < NQ ? m : 0] : *reinterpret_cast<const bf16x8*>(qs + 1024);
      other = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kb[i % (AHEAD + 1)], q1, other, 0, 0, 0);
      sc[k] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kb[i % (AHEAD + 1)], q0, sc[k], 0, 0, 0);
      if (m == NH - 1) *reinterpret_cast<f32x4*>(xs + (wid * 2 + k) * 1024 + lane * 16) = other;
    }
  };
  // softmax of the own columns' completed scores of tile t; weights and factors to LDS
  auto softmax = [&](int t) {
    bf16x8 pf;
#pragma unroll
    for (int k = 0; k < 2; ++k) sc[k] += *reinterpret_cast<const f32x4*>(xs + ((wid ^ 1) * 2 + k) * 1024 + lane * 16);
    if (32 * t < full_lo || 32 * t + 31 > full_hi) {  // wave-uniform
#pragma unroll
      for (int k = 0; k < 2; ++k)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int key = 32 * t + 16 * k + 4 * g + r;
          if (key > cpos || key < klo) sc[k][r] = NEG_BIG;
        }
    }
    float tmax = NEG_BIG;
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
      for (int r = 0; r < 4; ++r) tmax = fmaxf(tmax, sc[k][r]);
    tmax = fmaxf(tmax, __shfl_xor(tmax, 16, 64));
    tmax = fmaxf(tmax, __shfl_xor(tmax, 32, 64));
    const float m_new = fmaxf(m_run, fmaxf(tmax * A.scale_log2, NEG_BIG));
    const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
    m_run = m_new;
    l_run *= alpha;
    // a column that has seen no key yet (its window starts in a later tile): every weight is 0
    const float nm = m_run < 0.01f * NEG_BIG ? 0.f : -m_run;
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float p = __builtin_amdgcn_exp2f(fmaf(sc[k][r], A.scale_log2, nm));
        l_run += p;
        pf[4 * k + r] = (bf16)p;
      }
    const int at = ((t - t_lo) & 1) * NW + wid;
    *reinterpret_cast<bf16x8*>(xp + at * 1024 + lane * 16) = pf;
    if (g == 0) xa[at * 16 + c] = alpha;
  };
  auto outputs = [&](const char* tile, const bf16x8 (&p)[2]) {
    bf16x4 v0[AHEAD + 1], v1[AHEAD + 1];
    auto read = [&](int n) {
      v0[n % (AHEAD + 1)] = tr_read_ahead(tile + n * 512 + toff);
      v1[n % (AHEAD + 1)] = tr_read_ahead(tile + D * 32 + n * 512 + toff);
    };
#pragma unroll
    for (int n = 0; n < AHEAD; ++n) read(n);
#pragma unroll
    for (int n = 0; n < RT; ++n) {
      if (n + AHEAD < RT) read(n + AHEAD);
      __builtin_amdgcn_sched_barrier(0);
      bf16x8 v;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        v[j] = v0[n % (AHEAD + 1)][j];
        v[4 + j] = v1[n % (AHEAD + 1)][j];
      }
#pragma unroll
      for (int x = 0; x < 2; ++x) o[x][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v, p[x], o[x][n], 0, 0, 0);
    }
  };
  // (Waits by the builtin: of a wait in asm the compiler knows nothing, and at the loop's first use of the queries it then
  // waited for every load, the tile's just issued among them.)
  auto lds_barrier = [] {  // tile loads stay in flight across it
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  auto landed = [] {  // and this one waits for them
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0x0070);  // vmcnt(0) lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  if (n_t > 0) {
    issue(t_lo, smem);
    landed();
    if (n_t > 1) issue(t_lo + 1, smem + TILE);
    scores(smem);
    lds_barrier();
    softmax(t_lo);
    landed();
  }
  __builtin_amdgcn_s_waitcnt(0x0070);  // (also for the path past the branch)
  int cur = 0, nxt = 1;  // buffers of tiles i and i + 1
  for (int i = 0; i < n_t; ++i) {
    const int far = 3 - cur - nxt;
    // tile i + 2 goes where i - 1 was, whose outputs everybody has done
    if (i + 2 < n_t) issue(t_lo + i + 2, smem + far * TILE);
    if (i + 1 < n_t) scores(smem + nxt * TILE);
    lds_barrier();
    if (grp && i + 1 < n_t) softmax(t_lo + i + 1);
    const int own = (i & 1) * NW + wid, other = (i & 1) * NW + (wid ^ 1);
    const bf16x8 p[2] = {*reinterpret_cast<const bf16x8*>(xp + own * 1024 + lane * 16),
                         *reinterpret_cast<const bf16x8*>(xp + other * 1024 + lane * 16)};
    const float a0 = xa[own * 16 + c], a1 = xa[other * 16 + c];
    if (__any(a0 != 1.f)) {
#pragma unroll
      for (int n = 0; n < RT; ++n) o[0][n] *= a0;
    }
    if (__any(a1 != 1.f)) {
#pragma unroll
      for (int n = 0; n < RT; ++n) o[1][n] *= a1;
    }
    outputs(smem + cur * TILE, p);
    if (!grp && i + 1 < n_t) softmax(t_lo + i + 1);
    landed();
    cur = nxt;
    nxt = far;
  }
  float l = l_run;
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  if (g == 0) xa[wid * 16 + c] = l;
  lds_barrier();
  const float lx[2] = {l, xa[(wid ^ 1) * 16 + c]};
#pragma unroll
  for (int x = 0; x < 2; ++x) {
    if (col(x) >= cols) continue;
    if (nparts > 1) {  // 8 slots hold the item's columns in a row
      const size_t pc = (size_t)it.w * A.NB * 16 + col(x);
      float* po = A.part_o + pc * RP + half * (16 * RT) + 4 * g;
#pragma unroll
      for (int n = 0; n < RT; ++n) *reinterpret_cast<f32x4*>(po + 16 * n) = o[x][n];
      if (x == 0 && g == 0) reinterpret_cast<float2*>(A.part_ml)[pc] = float2{m_run, l};
      continue;
    }
    const float inv = 1.f / lx[x];
    bf16* orow = (bf16*)A.out + (row0 + col(x)) * RP + half * (16 * RT) + 4 * g;
#pragma unroll
    for (int n = 0; n < RT; ++n) {
      bf16x4 v;
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = (bf16)(o[x][n][r] * inv);
      *reinterpret_cast<bf16x4*>(orow + 16 * n) = v;
    }
  }
}

// A unit of the expanded form: X_COLS tokens of a request, one head, a part of their keys. Four column groups of 32 tokens
// and two waves each, which take the 32-key tiles of a 64-key stage: a fragment read from LDS then serves two MFMAs, as many
// bytes as the MFMAs take time for, and the two waves of a SIMD run the same columns, and the second adds its
// outputs a stage late, so that one's softmax lies under the other's products. Stages arrive by direct loads two ahead (four
// buffers), one barrier each; the two waves' outputs meet in LDS. 4,096 tokens, 16 heads: 125 us back to back with the merge
// launch (MFMAs 38, without the softmax 102, without the loads 104: LDS reads, 1,280 cycles a stage as the MFMAs, and the
// softmax's 1,600 of a SIMD's VALU overlap in part); pair_item takes 318 and two head projections of 32 each, here the
// expansion's 25. 499 tokens after 3,584: 49 and 25 us, 110 and 22 in the absorbed form. (In a step's launches: 132 and 6 for the
// merge, 28; 38 and 12, 27.)
constexpr int X_BLOCK = (2 * X_DIM + X_ROT) * 32, X_STAGE = 4 * X_BLOCK;  // bytes of 16 keys, of a stage

// stages [lo, hi) of 64 keys that the tokens of a tile see
__device__ __forceinline__ void unit_stages(int pos0, int n, int window, int& lo, int& hi) {
  lo = (window > 0 ? max(0, pos0 - window + 1) : 0) >> 6;
  hi = (pos0 + n + 63) >> 6;
}

__device__ __forceinline__ void expanded_unit(const Args& A, const int4 it, int h, char* smem) {
  constexpr int NQ = (X_DIM + X_ROT) / 32, NV = X_DIM / 16;
  const int s = it.x, part = it.z & 0xffff, nparts = it.z >> 16;
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), g = lane >> 4, c = lane & 15;
  const int cg = wid & 3, kp = wid >> 2;
  const int ctx = A.ctx_len[s], ql = A.q_len[s], nq = min(X_COLS, ql - it.y * X_COLS);
  const int pos0 = ctx - ql + it.y * X_COLS;
  const size_t row0 = (size_t)A.q_start[s] + it.y * X_COLS;
  int s_lo, s_hi;
  unit_stages(pos0, nq, A.window, s_lo, s_hi);
  if (nparts > 1) {  // this part's stages (possibly none)
    const int per = (s_hi - s_lo + nparts - 1) / nparts;
    s_lo += part * per;
    s_hi = min(s_hi, s_lo + per);
  }
  const int n_st = s_hi - s_lo, last_blk = ((ctx + 15) >> 4) - 1, base = A.X.base[s];
  // this wave's columns see some / all of the keys in [some_lo, some_hi] / [all_lo, all_hi]
  const int wf = pos0 + min(cg * 32, nq - 1), we = pos0 + min(cg * 32 + 31, nq - 1);
  const int some_lo = A.window > 0 ? wf - A.window + 1 : 0, all_lo = A.window > 0 ? we - A.window + 1 : 0;

  f32x4 o[2][NV];
  float m_run[2], l_run[2];
#pragma unroll
  for (int x = 0; x < 2; ++x) {
#pragma unroll
    for (int n = 0; n < NV; ++n) o[x][n] = f32x4{0.f, 0.f, 0.f, 0.f};
    m_run[x] = NEG_BIG;
    l_run[x] = 0.f;
  }
  static_assert(2 * X_DIM * 32 == NW * 1024 && X_ROT * 32 * 4 == NW * 1024, "a stage is five loads a wave, which the waits below count");
  const char* kx = (const char*)A.X.kx + (size_t)h * (X_DIM * 64) + wid * 1024 + lane * 16;
  const char* kr = (const char*)A.X.kr + (wid & 1) * 1024 + lane * 16;
  auto issue = [&](int st, char* dst) {
    auto blk = [&](int b) { return (size_t)(base + min(4 * st + b, last_blk)); };
#pragma unroll
    for (int b = 0; b < 4; ++b)
      __builtin_amdgcn_global_load_lds((glb_void*)(kx + blk(b) * A.H * (X_DIM * 64)), (lds_void*)(dst + b * X_BLOCK + wid * 1024), 16, 0, 0);
    __builtin_amdgcn_global_load_lds((glb_void*)(kr + blk(wid >> 1) * (X_ROT * 32)),
                                     (lds_void*)(dst + (wid >> 1) * X_BLOCK + 2 * X_DIM * 32 + (wid & 1) * 1024), 16, 0, 0);
  };
  auto buffer = [&](int i) { return smem + (i & 3) * X_STAGE; };
  // (the first stages are under way while the queries arrive and turn)
  if (n_st > 0) issue(s_lo, buffer(0));
  if (n_st > 1) issue(s_lo + 1, buffer(1));
  int cpos[2], klo[2];
  bf16x8 qf[2][NQ];
#pragma unroll
  for (int x = 0; x < 2; ++x) {
    const int col = min(cg * 32 + x * 16 + c, nq - 1);
    cpos[x] = pos0 + col;
    klo[x] = A.window > 0 ? max(0, cpos[x] - A.window + 1) : 0;
    const bf16* src = (const bf16*)A.X.q + (row0 + col) * A.X.ldq + h * (X_DIM + X_ROT) + 8 * g;
#pragma unroll
    for (int m = 0; m < NQ; ++m) qf[x][m] = *reinterpret_cast<const bf16x8*>(src + 32 * m);
    // the rotated part: the two halves turn together
    const float* cs = A.X.cos_sin + (size_t)cpos[x] * X_ROT + 8 * g;
    float co[8], si[8];
    __builtin_memcpy(co, cs, 32);
    __builtin_memcpy(si, cs + X_ROT / 2, 32);
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const float u = (float)qf[x][NQ - 2][k], v = (float)qf[x][NQ - 1][k];
      qf[x][NQ - 2][k] = (bf16)(u * co[k] - v * si[k]);
      qf[x][NQ - 1][k] = (bf16)(v * co[k] + u * si[k]);
    }
  }
  const int loff = (g * 16 + c) * 16;
  const int toff = ((c & 3) >> 1) * 256 + (4 * g + (c >> 2)) * 16 + (c & 1) * 8;
  // Fragments are read AHEAD steps before their use: left to itself the compiler waits for each.
  constexpr int AHEAD = 4;
  f32x4 sc[2][2];
  bf16x8 pf[2];
  auto scores = [&](const char* tile) {
    bf16x8 kb[AHEAD];
    auto frag = [&](int i) {
      const int k = i & 1, m = i >> 1;
      return *reinterpret_cast<const bf16x8*>(tile + k * X_BLOCK + (m < X_DIM / 32 ? m * 1024 : 2 * X_DIM * 32 + (m - X_DIM / 32) * 1024) + loff);
    };
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) kb[i] = frag(i);
#pragma unroll
    for (int i = 0; i < 2 * NQ; ++i) {
      const int k = i & 1, m = i >> 1;
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        if (m == 0) sc[x][k] = f32x4{0.f, 0.f, 0.f, 0.f};
        sc[x][k] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kb[i % AHEAD], qf[x][m], sc[x][k], 0, 0, 0);
      }
      if (i + AHEAD < 2 * NQ) kb[i % AHEAD] = frag(i + AHEAD);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  // the largest of a column's values, which its four lanes hold: rows of 16 lanes, then halves, change places
  auto column_max = [](float v) {
    auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
    r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
  };
  auto softmax = [&](int key0) {
    if (key0 < all_lo || key0 + 31 > wf) {  // wave-uniform
#pragma unroll
      for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int k = 0; k < 2; ++k)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int key = key0 + 16 * k + 4 * g + r;
            if (key > cpos[x] || key < klo[x]) sc[x][k][r] = NEG_BIG;
          }
    }
    float m_new[2];
#pragma unroll
    for (int x = 0; x < 2; ++x) {
      float tmax = NEG_BIG;
#pragma unroll
      for (int k = 0; k < 2; ++k)
#pragma unroll
        for (int r = 0; r < 4; ++r) tmax = fmaxf(tmax, sc[x][k][r]);
      m_new[x] = fmaxf(m_run[x], fmaxf(column_max(tmax) * A.scale_log2, NEG_BIG));
    }
    if (__any(m_new[0] > m_run[0] || m_new[1] > m_run[1])) {
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        const float alpha = __builtin_amdgcn_exp2f(m_run[x] - m_new[x]);
        l_run[x] *= alpha;
#pragma unroll
        for (int n = 0; n < NV; ++n) o[x][n] *= alpha;
        m_run[x] = m_new[x];
      }
    }
#pragma unroll
    for (int x = 0; x < 2; ++x) {
      // a column that has seen no key yet: every weight is 0
      const float nm = m_run[x] < 0.01f * NEG_BIG ? 0.f : -m_run[x];
#pragma unroll
      for (int k = 0; k < 2; ++k)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float p = __builtin_amdgcn_exp2f(fmaf(sc[x][k][r], A.scale_log2, nm));
          l_run[x] += p;
          pf[x][4 * k + r] = (bf16)p;
        }
    }
  };
  auto outputs = [&](const char* tile) {
    bf16x4 v0[AHEAD], v1[AHEAD];
    auto read = [&](int n) {
      v0[n % AHEAD] = tr_read_ahead(tile + X_DIM * 32 + n * 512 + toff);
      v1[n % AHEAD] = tr_read_ahead(tile + X_BLOCK + X_DIM * 32 + n * 512 + toff);
    };
#pragma unroll
    for (int n = 0; n < AHEAD; ++n) read(n);
#pragma unroll
    for (int n = 0; n < NV; ++n) {
      __builtin_amdgcn_sched_barrier(0);
      bf16x8 v;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        v[j] = v0[n % AHEAD][j];
        v[4 + j] = v1[n % AHEAD][j];
      }
#pragma unroll
      for (int x = 0; x < 2; ++x) o[x][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v, pf[x], o[x][n], 0, 0, 0);
      if (n + AHEAD < NV) read(n + AHEAD);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  int late = -1;  // the stage whose outputs the second waves have yet to add
  for (int i = 0; i < n_st; ++i) {
    asm volatile("" ::: "memory");
    if (i + 1 < n_st) __builtin_amdgcn_s_waitcnt(0x0075);  // vmcnt(5) lgkmcnt(0): the next stage's loads stay in flight
    else __builtin_amdgcn_s_waitcnt(0x0070);
    __builtin_amdgcn_s_barrier();  // stage i is whole, and nobody reads stage i - 2 any more
    asm volatile("" ::: "memory");
    if (i + 2 < n_st) issue(s_lo + i + 2, buffer(i + 2));
    if (late >= 0) outputs(buffer(late) + 2 * X_BLOCK);
    late = -1;
    const char* tile = buffer(i) + kp * (2 * X_BLOCK);
    const int key0 = 64 * (s_lo + i) + 32 * kp;
    if (key0 > we || key0 + 31 < some_lo) continue;  // wave-uniform: no column sees the tile
    scores(tile);
    softmax(key0);
    if (kp) late = i;
    else outputs(tile);
  }
  if (late >= 0) outputs(buffer(late) + 2 * X_BLOCK);
  // each of a column group's two waves sends the partner 16 columns and completes the other 16
#pragma unroll
  for (int x = 0; x < 2; ++x) {
    l_run[x] += __shfl_xor(l_run[x], 16, 64);
    l_run[x] += __shfl_xor(l_run[x], 32, 64);
  }
  f32x4* send = reinterpret_cast<f32x4*>(smem) + wid * (NV * 64);
  float2* send_ml = reinterpret_cast<float2*>(smem + NW * NV * 1024) + wid * 16;
  __syncthreads();  // (also the waits for every load to LDS)
#pragma unroll
  for (int n = 0; n < NV; ++n) send[n * 64 + lane] = kp ? o[0][n] : o[1][n];
  if (g == 0) send_ml[c] = kp ? float2{m_run[0], l_run[0]} : float2{m_run[1], l_run[1]};
  __syncthreads();
  const f32x4* got = reinterpret_cast<const f32x4*>(smem) + (wid ^ 4) * (NV * 64);
  const float2 ml = (reinterpret_cast<const float2*>(smem + NW * NV * 1024) + (wid ^ 4) * 16)[c];
  const float m_own = kp ? m_run[1] : m_run[0], l_own = kp ? l_run[1] : l_run[0];
  const float m = fmaxf(m_own, ml.x), f0 = exp2f(m_own - m), f1 = exp2f(ml.x - m), L = f0 * l_own + f1 * ml.y;
  const int col = cg * 32 + kp * 16 + c;
  if (col >= nq) return;
  const size_t pc = ((size_t)(it.w + part) * A.H + h) * X_COLS + col;
  if (nparts > 1 && g == 0) reinterpret_cast<float2*>(A.X.part_ml)[pc] = float2{m, L};
  const float inv = 1.f / L;
  bf16* out = (bf16*)A.X.out + (row0 + col) * A.X.ldo + h * X_DIM + 4 * g;
#pragma unroll
  for (int n = 0; n < NV; ++n) {
    const f32x4 mine = kp ? o[1][n] : o[0][n];
    const f32x4 v = mine * f0 + got[n * 64 + lane] * f1;
    if (nparts > 1) {
      *reinterpret_cast<f32x4*>(A.X.part_o + pc * X_DIM + 16 * n + 4 * g) = v;
      continue;
    }
    bf16x4 b;
#pragma unroll
    for (int r = 0; r < 4; ++r) b[r] = (bf16)(v[r] * inv);
    *reinterpret_cast<bf16x4*>(out + 16 * n) = b;
  }
}

// Which requests of a step are expanded, where their keys go, and the launches' work lists (one workgroup): those of at least
// X_MIN new tokens, however many are cached, and all of them or none. None where they are more than X_REQS or their keys more
// than the workspace's `room` blocks: a launch ends with its longest item, and the absorbed items of one prompt that is left
// take as long as those of all (2 prompts of 256 after 2,500, 8 layers: 3,216 us absorbed, one of them expanded 3,520). None where
// they fill less than half of the columns of more than two tiles: 10 of 50 after 150 beside 200 decode rows 3,292 us refused,
// 3,407 expanded; 60 of 12 after 60 3,033, 3,370; 7 of 72 after 150 beside 30 2,912, 2,800. And none where they are less than twice
// the tokens of the other requests, whose items wait for the units: 2 of 140 after 600 beside 230 rows of 1,500 keys 3,409, 3,464; 4
// of 132 after 700 beside 200 of 1,000 3,615, 3,605. Tiles whose keys are more than a workgroup's average are split. Rows
// behind the last request's are nobody's, and the head products leave them out like the expanded (`skip`): 13 of 512 had them walk
// their whole inputs, W_uv's 11.9 us and W_uk's 7.4, 4.7 and 5.2 without (3,007 -> 2,885 a step of 8 layers).
constexpr int X_MIN = 12;
__global__ __launch_bounds__(1024) void expand_plan_kernel(const Expand X, const int* __restrict__ q_start,
                                                           const int* __restrict__ q_len, const int* __restrict__ ctx_len, int S,
                                                           int T, int H, int window, int room, int max_att, int max_tiles, int slots,
                                                           int* __restrict__ skip) {
  static_assert(X_REQS == 64, "a lane a request");
  __shared__ int ws[16], others[16], tops[16], req[X_REQS], qs[X_REQS], ql[X_REQS], cl[X_REQS], to[X_REQS], tiles[X_REQS];
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  int found = 0, rest = 0, top = 0;
  for (int s0 = 0; s0 < S; s0 += 1024) {
    const int s = s0 + threadIdx.x, n = s < S ? q_len[s] : 0;
    const bool yes = n >= X_MIN && s < S && q_start[s] + n <= T;
    if (s < S) X.base[s] = X_NONE;
    if (!yes) rest += n;
    if (n > 0) top = max(top, q_start[s] + n);
    const unsigned long long b = __ballot(yes);
    if (lane == 0) ws[wid] = __popcll(b);
    __syncthreads();
    int at = found + (int)__popcll(b & ((1ull << lane) - 1));
    for (int w = 0; w < 16; ++w) {
      if (w < wid) at += ws[w];
      found += ws[w];
    }
    if (yes && at < X_REQS) {
      req[at] = s;
      qs[at] = q_start[s];
      ql[at] = n;
      cl[at] = ctx_len[s];
    }
    __syncthreads();
  }
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    rest += __shfl_xor(rest, o, 64);
    top = max(top, __shfl_xor(top, o, 64));
  }
  if (lane == 0) {
    others[wid] = rest;
    tops[wid] = top;
  }
  __syncthreads();
  rest = 0;
  for (int w = 0; w < 16; ++w) {
    rest += others[w];
    top = max(top, tops[w]);
  }
  for (int t = threadIdx.x; t < T; t += 1024) {
    X.form[t] = 0;
    skip[t] = t >= top;
  }
  // every wave works out all of this, a request a lane
  int n = found <= X_REQS ? found : 0, lo = 0, hi, blocks = 0, nt = 0, total = 0, cols = 0, tokens = 0;
  if (lane < n) {
    const int p0 = cl[lane] - ql[lane];
    unit_stages(p0, ql[lane], window, lo, hi);
    blocks = ((cl[lane] + 15) >> 4) - 4 * lo;
    nt = (blocks + 3) >> 2;
    for (int q = 0; q < ql[lane]; q += X_COLS) {
      int a, b;
      unit_stages(p0 + q, min(X_COLS, ql[lane] - q), window, a, b);
      total += b - a;
      cols += X_COLS;
    }
    tokens = ql[lane];
  }
  int used = blocks, all = nt;  // with the lanes before
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int u = __shfl_up(used, o, 64), v = __shfl_up(all, o, 64);
    if (lane >= o) {
      used += u;
      all += v;
    }
    total += __shfl_xor(total, o, 64);
    cols += __shfl_xor(cols, o, 64);
    tokens += __shfl_xor(tokens, o, 64);
  }
  const int listed = __shfl(all, 63, 64);
  if (__shfl(used, 63, 64) > room || listed > max_tiles || (cols > 2 * X_COLS && 2 * tokens < cols) || tokens < 2 * rest) n = 0;
  if (threadIdx.x < n) {
    to[lane] = used - blocks - 4 * lo;
    tiles[lane] = all - nt;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    const int fair = max(8, (total * H + 255) / 256);
    int na = 0, slot = 0;
    for (int i = 0; i < n; ++i)
      for (int q = 0; q < ql[i]; q += X_COLS) {
        unit_stages(cl[i] - ql[i] + q, min(X_COLS, ql[i] - q), window, lo, hi);
        int parts = min(X_PARTS, (hi - lo + fair - 1) / fair);
        if (slot + parts > slots) parts = 1;
        for (int p = 0; p < parts && na < max_att; ++p) X.att[na++] = int4{req[i], q / X_COLS, p | parts << 16, slot};
        if (parts > 1) slot += parts;
      }
    X.counts[0] = na;
    X.counts[1] = n ? listed : 0;
  }
  for (int i = 0; i < n; ++i) {
    unit_stages(cl[i] - ql[i], ql[i], window, lo, hi);
    const int nb = (cl[i] + 15) >> 4;
    if (threadIdx.x == 0) X.base[req[i]] = to[i];
    for (int j = threadIdx.x; 4 * (lo + j) < nb; j += 1024)
      X.tiles[tiles[i] + j] = int4{req[i], 4 * (lo + j), min(4, nb - 4 * (lo + j)), to[i] + 4 * (lo + j)};
    for (int t = threadIdx.x; t < ql[i]; t += 1024) X.form[qs[i] + t] = skip[qs[i] + t] = 1;
  }
}

// Keys and values of the heads: the latents of a block of 16 keys, as the pages hold them, times W_uk,h and W_uv,h. A workgroup keeps the
// weights of one head (256 KB) in registers, 32 of the 256 outputs a wave, and takes its share of the blocks through LDS, X_AHEAD ahead by
// direct loads; the outputs' lanes hold 4 dims of a key: 512 bytes of the workspace a store. 4,096 keys of 16 heads 23 us (17 GFLOP, 34 MB
// written): the products take 14 behind 5 of weights on their way, the stores 4 more (stores of 1 KB as long; four waves of 64 outputs, which
// read half as much LDS, 25; XCDs of 4 or 16 heads 23 and 26). With two heads' weights streamed from L2 past a workgroup's 64 keys, two
// workgroups a CU, arrival, products and stores came one after the other. us so -> now: 100 keys 11.0 -> 5.3, 512 11.6 -> 6.9,
// 1,000 12.5 -> 9.1, 2,000 15.6 -> 14.3, 3,000 23.0 -> 18.9, 4,096 27.6 -> 23.1; 5 heads 4,096 13.7 -> 12.2, 40 heads 512 13.6 -> 11.2, 4,096 60.5 -> 46.0.
constexpr int X_AHEAD = 6, X_RING = 8;  // blocks
__global__ __launch_bounds__(512, 2) void expand_kernel(const Expand X, const bf16* __restrict__ pages, const bf16* __restrict__ wk,
                                                        const bf16* __restrict__ wv, const int* __restrict__ block_table, int max_blocks, int H, int D,
                                                        int shares) {
  extern __shared__ __attribute__((aligned(16))) char smem[];  // [X_RING][X_RANK / 32][1 KB]
  constexpr int KS = X_RANK / 32, NT = 2, P = X_AHEAD, EARLY = 6;
  static_assert(P < X_RING, "a block arrives where nobody reads");
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), g = lane >> 4, c = lane & 15;
  const int h = blockIdx.x % H, n = 4 * X.counts[1], per = (n + shares - 1) / shares, i0 = blockIdx.x / H * per, i1 = min(n, i0 + per);
  if (i0 >= i1) return;
  // a block a lane, 64 from c0 on: its page and its place in the workspace (of a tile's missing blocks: those of its last one)
  int id, to;
  auto places = [&](int c0) {
    const int e = min(c0 + lane, i1 - 1);
    const int4 tl = X.tiles[e >> 2];
    const int b = min(e & 3, tl.z - 1);
    to = tl.w + b;
    id = block_table[(size_t)tl.x * max_blocks + tl.y + b];
  };
  places(i0);
  asm volatile("" ::"v"(id) : "memory");  // (before the weights are under way, which a later wait would be for too)
  const int t16 = wid * NT;  // the wave's first tile of the head's 8 of keys and 8 of values
  const bf16* wp = (t16 < 8 ? wk : wv) + ((size_t)h * 8 + (t16 & 7)) * (KS * 512) + lane * 8;
  bf16x8 a[KS][NT];
#pragma unroll
  for (int s = 0; s < KS; ++s)
#pragma unroll
    for (int i = 0; i < NT; ++i) a[s][i] = *reinterpret_cast<const bf16x8*>(wp + (size_t)(i * KS + s) * 512);
  for (int c0 = i0; c0 < i1; c0 += 64) {
    const int m = min(64, i1 - c0);
    if (c0 > i0) places(c0);
    auto issue = [&](int i) {  // (past the end: the last block again, so that the waits stay counted)
      const bf16* src = pages + (size_t)__builtin_amdgcn_readlane(id, min(i, m - 1)) * (D * 16) + wid * 512 + lane * 8;
      char* dst = smem + (i % X_RING) * (KS * 1024) + wid * 1024;
#pragma unroll
      for (int j = 0; j < KS / 8; ++j)
        __builtin_amdgcn_global_load_lds((glb_void*)(src + j * 4096), (lds_void*)(dst + j * 8192), 16, 0, 0);
    };
    for (int i = 0; i < P; ++i) issue(i);
    for (int i = 0; i < m; ++i) {
      // this wave's two loads of block i have arrived: behind them the loads of P - 1 blocks are under way and, once they
      // are P blocks old, two stores of each of the last P too
      asm volatile("" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      if (i < P) __builtin_amdgcn_s_waitcnt(0x0F70 | (2 * P - 2));
      else __builtin_amdgcn_s_waitcnt(0x0F70 | ((4 * P - 2) & 15) | (4 * P - 2) >> 4 << 14);
      __builtin_amdgcn_s_barrier();  // block i is whole, and nobody reads block i - 1 any more
      asm volatile("" ::: "memory");
      issue(i + P);
      __builtin_amdgcn_sched_barrier(0);
      const char* from = smem + (i % X_RING) * (KS * 1024) + lane * 16;
      f32x4 acc[NT];
#pragma unroll
      for (int j = 0; j < NT; ++j) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
      bf16x8 k[EARLY];  // (left to itself the compiler waits for each pair)
#pragma unroll
      for (int s = 0; s < EARLY; ++s) k[s] = *reinterpret_cast<const bf16x8*>(from + s * 1024);
#pragma unroll
      for (int s = 0; s < KS; ++s) {
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[s][j], k[s % EARLY], acc[j], 0, 0, 0);
        if (s + EARLY < KS) k[s % EARLY] = *reinterpret_cast<const bf16x8*>(from + (s + EARLY) * 1024);
      }
      bf16* dst = (bf16*)X.kx + ((size_t)__builtin_amdgcn_readlane(to, i) * H + h) * (X_DIM * 32) + (2 * t16 + (g >> 1)) * 128 + c * 8 + (g & 1) * 4;
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        bf16x4 v;
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = (bf16)acc[j][r];
        *reinterpret_cast<bf16x4*>(dst + j * 256) = v;
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    // the rotated parts, a block a wave, shared out over the heads
    for (int i = wid; i < m; i += 8) {
      if ((c0 + i) % H != h) continue;
      const bf16x8* src = reinterpret_cast<const bf16x8*>(pages + (size_t)__builtin_amdgcn_readlane(id, i) * (D * 16) + X_RANK * 16) + lane;
      bf16x8* dst = reinterpret_cast<bf16x8*>((bf16*)X.kr + (size_t)__builtin_amdgcn_readlane(to, i) * (X_ROT * 16)) + lane;
      dst[0] = src[0];
      dst[64] = src[64];
    }
    __builtin_amdgcn_s_waitcnt(0x0070);  // every load to LDS has arrived, before others come or the workgroup ends
    __syncthreads();
  }
}

// Latents of 32 PAIRS and more: pair_item, on 256 workgroups. us of 16 heads, tile_item and as many workgroups as items
// against pair_item: 512 + 64, 4 x 1,024 tokens 137, 114, 512 after 3,584 129, 108, 40 decode rows and 9 x 210 after 320
// 77, 74; 384 + 64: 90, 91; 87, 89; 55, 61; 256 + 32: 77, 73; 76, 74; 47, 50.
constexpr int PAIRS = 16;

template <int RT, int PT, bool XP = false>
constexpr int lds_bytes() {
  return std::max({XP ? 4 * X_STAGE : 0, RT >= PAIRS ? pair_lds_bytes<RT, PT>() : 2 * 32 * 32 * (RT + PT) * 2, NW * 32 * 32 * RT + 1024 * (RT + PT),
                   NW * 16 * MERGE_LD * 4 + 2 * NW * 16 * 4});
}

template <int RT, int PT, int CT, bool XP = false>
__global__ __launch_bounds__(64 * NW, 2) void mfma_kernel(const Args A) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int n = A.n_items[0];
  // Two passes over the workgroup's items, so that neither path's registers carry the other's.
  int y0 = blockIdx.y;  // this workgroup's place in the rounds of items
  if constexpr (XP) {  // as below, in rounds of all heads, so that an XCD's workgroups keep their heads
    const int G = gridDim.x * gridDim.y, b = blockIdx.y * gridDim.x + blockIdx.x, per = G / A.H, na = A.X.counts[0];
    if (b < per * A.H)
      for (int r = 0; r * per < na; ++r) {
        const int item = r * per + (r & 1 ? per - 1 - b / A.H : b / A.H);
        if (item >= na) continue;
        expanded_unit(A, A.X.att[item], b % A.H, smem);
        __syncthreads();
      }
    // the other items begin with the workgroups that had no unit
    y0 = (y0 + gridDim.y - min(na * A.H, G - 1) / gridDim.x) % gridDim.y;
  }
  if constexpr (RT >= PAIRS) {
    // Tiles are dealt in rounds over the workgroups, every second one from its end: a prompt's later items have more keys,
    // and with one workgroup a CU each gets as many keys in all (4,096 tokens, as many workgroups as items: 341 us, here
    // 318).
    for (int r = 0, b = y0; r * (int)gridDim.y < n; ++r, b = gridDim.y - 1 - b) {
      const int item = r * gridDim.y + b;
      if (item >= n) continue;
      const int4 it = A.items[item];
      if ((it.z & 0xff) <= A.dec_tokens || expanded<XP>(A, it.x)) continue;
      pair_item<RT, PT>(A, it, smem);
      __syncthreads();
    }
  } else {
    for (int item = blockIdx.y; item < n; item += gridDim.y) {
      const int4 it = A.items[item];
      if ((it.z & 0xff) <= A.dec_tokens || expanded<XP>(A, it.x)) continue;
      tile_item<RT, PT, CT>(A, it, smem);
      __syncthreads();
    }
  }
  for (int item = y0; item < n; item += gridDim.y) {
    const int4 it = A.items[item];
    if ((it.z & 0xff) > A.dec_tokens || expanded<XP>(A, it.x)) continue;
    split_item<RT, PT>(A, it, smem);
    __syncthreads();
  }
}

// merge_kernel and the next product in one launch, y[row, head h] = W_uv[h] (merged latent): a workgroup of 16 waves per (head, `per`
// columns, up to 16: tokens of the items in their order). The waves share the columns' dimensions, while the head's W_uv is on its
// way: a wave has 16 of its (at most 128) rows and half of their inputs. A chain of dependent reads bounds it (items, (max, sum) pairs, partitions),
// where two launches had each their own: 8 rows after 2,048 tokens, 16 heads of 512 and 128, a step's 8 layers 1,430 -> 1,399 us, 64 rows
// 2,241 -> 2,213, the launch 7.3 and 8.6. Partitions and inputs are added up in the order of the two launches: a request's bits do not
// depend on the step's form. (With partitions shared out over the waves, whose sums meet in LDS, the launch took 7.4 and 8.9; a workgroup for
// 16 items, whatever tokens they hold, 3 to 5 % more of a step of short prompts.)
constexpr int MH_WAVES = 16;

// Columns [d, d + VW) of the partitions of one token and head, added up in their order; all loads of a round are under way at once.
template <int VW>
__device__ __forceinline__ void merge_dims(const Args& A, int4 e, int RP, int d, float (&a)[8]) {
  typedef float vec __attribute__((ext_vector_type(VW > 4 ? 4 : VW)));
  constexpr int PIECES = VW > 4 ? 2 : 1, ROUND = VW == 1 ? 16 : VW == 2 ? 8 : 4;  // (few columns are of long splits)
  const int lane = threadIdx.x & 63, nparts = e.y >> 20, step = (e.y & 0xff) <= A.dec_tokens ? 1 : 8;
  const float2* ml = reinterpret_cast<const float2*>(A.part_ml);
  auto slot = [&](int p) { return (size_t)e.x + (size_t)p * step * A.NB * 16; };
  float gm = NEG_BIG, L = 0.f;
  for (int p0 = 0; p0 < nparts; p0 += 64) gm = fmaxf(gm, p0 + lane < nparts ? ml[slot(p0 + lane)].x : NEG_BIG);
  gm = wave_max(gm);
  for (int p0 = 0; p0 < nparts; p0 += 64) {
    float wt = 0.f;
    if (p0 + lane < nparts) {
      const float2 v = ml[slot(p0 + lane)];
      wt = exp2f(v.x - gm);
      L += wt * v.y;
    }
    const int np = min(64, nparts - p0);
#pragma unroll 1
    for (int q = 0; q < np; q += ROUND) {
      vec x[ROUND][PIECES];
#pragma unroll
      for (int p = 0; p < ROUND; ++p) {  // (behind the last: its values again)
        const vec* s = reinterpret_cast<const vec*>(A.part_o + slot(p0 + min(q + p, np - 1)) * RP + d);
#pragma unroll
        for (int i = 0; i < PIECES; ++i) x[p][i] = s[i];
      }
#pragma unroll
      for (int p = 0; p < ROUND; ++p) {
        const float wp = __shfl(wt, (q + p) & 63, 64);
#pragma unroll
        for (int j = 0; j < VW; ++j) a[j] = q + p < np ? fmaf(wp, x[p][j / 4][j % 4], a[j]) : a[j];
      }
    }
  }
  const float inv = 1.f / wave_sum(L);
#pragma unroll
  for (int j = 0; j < VW; ++j) a[j] *= inv;
}

template <int RT>
__global__ __launch_bounds__(64 * MH_WAVES) void merge_heads_kernel(const Args A, const bf16* __restrict__ uv, bf16* __restrict__ y, int ldy,
                                                                    int vp, int max_items, int per) {
  constexpr int RP = 32 * RT, LD = RP + 8, HALF = (RT + 1) / 2;
  __shared__ __attribute__((aligned(16))) bf16 xs[16][LD];
  __shared__ __attribute__((aligned(16))) float ps[8][256];
  __shared__ int4 cols[16];  // {the first partition's column, the item's z, sequence, token}
  __shared__ int sums[MH_WAVES];
  const int h = blockIdx.x, lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), tiles = vp / 16;
  const int g = lane >> 4, c16 = lane & 15, tile = wid & 7, k0 = wid >> 3 ? HALF : 0;
  bf16x8 w[HALF];
#pragma unroll
  for (int k = 0; k < HALF; ++k)
    w[k] = *reinterpret_cast<const bf16x8*>(uv + (((size_t)h * tiles + min(tile, tiles - 1)) * RT + min(k0 + k, RT - 1)) * 512 + lane * 8);
  const int lo = blockIdx.y * per;
  int total = 0;
  for (int b = 0; b < max_items && total < lo + per; b += 64 * MH_WAVES) {
    const int4 it = A.items[min(b + (int)threadIdx.x, max_items - 1)];  // (on its way with the list's length)
    const bool in = b + (int)threadIdx.x < A.n_items[0] && ((it.z >> 8) & 0xfff) == 0;
    const int nq = in ? it.z & 0xff : 0;
    int at = nq;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int v = __shfl_up(at, o, 64);
      if (lane >= o) at += v;
    }
    if (lane == 63) sums[wid] = at;
    __syncthreads();
    int before = total - nq;
#pragma unroll
    for (int q = 0; q < MH_WAVES; ++q) {
      if (q < wid) before += sums[q];
      total += sums[q];
    }
    at += before;  // this item's first column
    for (int t = max(0, lo - at); t < nq && at + t < lo + per; ++t)
      cols[at + t - lo] = int4{it.w * A.NB * 16 + t * A.H + h, it.z, it.x, it.y + t};
    __syncthreads();
  }
  const int m = min(per, total - lo);
  if (m <= 0) return;
  const int mine = min(c16, m - 1), row = A.q_start[cols[mine].z] + cols[mine].w;
  // a column's waves have 512 of its dimensions between them: 8 a lane where a wave has a column to itself, 1 where there are 8
  const int shift = m > 8 ? 0 : m > 4 ? 1 : m > 2 ? 2 : 3, c = wid >> shift;
  if (c < m) {
    const int4 e = cols[c];
    const int vw = 8 >> shift, d = ((wid & ((1 << shift) - 1)) * 64 + lane) * vw, at = min(d, RP - vw);
    float a[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    auto merged = [&](auto width) {
      constexpr int VW = decltype(width)::value;
      typedef bf16 vec __attribute__((ext_vector_type(VW)));
      vec v;
      if (e.y >> 20 <= 1) {
        v = *reinterpret_cast<const vec*>((const bf16*)A.out + ((size_t)(A.q_start[e.z] + e.w) * A.H + h) * RP + at);
      } else {
        merge_dims<VW>(A, e, RP, at, a);
#pragma unroll
        for (int j = 0; j < VW; ++j) v[j] = (bf16)a[j];
      }
      if (d < RP) *reinterpret_cast<vec*>(&xs[c][d]) = v;
    };
    if (shift == 0) merged(std::integral_constant<int, 8>{});
    else if (shift == 1) merged(std::integral_constant<int, 4>{});
    else if (shift == 2) merged(std::integral_constant<int, 2>{});
    else merged(std::integral_constant<int, 1>{});
  }
  __syncthreads();
  // (columns behind the last one hold anything: their products are not stored)
  f32x4* other = reinterpret_cast<f32x4*>(ps[tile]) + lane;
  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  auto products = [&]() {
#pragma unroll
    for (int k = 0; k < HALF; ++k)
      if (k0 + k < RT)
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[k], *reinterpret_cast<const bf16x8*>(&xs[c16][32 * (k0 + k) + 8 * g]), acc, 0, 0, 0);
  };
  if (wid < 8) {
    products();
    *other = acc;
  }
  __syncthreads();
  if (wid >= 8) {
    acc = *other;
    products();
    if (c16 >= m || tile >= tiles) return;
    bf16x4 o;
#pragma unroll
    for (int r = 0; r < 4; ++r) o[r] = (bf16)acc[r];
    *reinterpret_cast<bf16x4*>(y + (size_t)row * ldy + (size_t)h * vp + tile * 16 + 4 * g) = o;
  }
}

}  // namespace la
}  // namespace pa

#define PA_LA_RT(X) X(1) X(2) X(3) X(4) X(6) X(8) X(12) X(16)

// The padded latent width the MFMA kernels use for R (the smallest built size that holds it), or
// R rounded to 32 when none does (the simple kernel then runs); likewise the rotated part.
extern "C" int pa_latent_pad(int R) {
  const int need = (R + 31) / 32;
#define PA_X(N) if (need <= N) return N * 32;
  PA_LA_RT(PA_X)
#undef PA_X
  return need * 32;
}

extern "C" int pa_latent_attention(int fp32, void* out, float* part_o, float* part_ml, const void* q, const void* pages, const int* items, const int* n_items, int max_items,
                                   const int* q_start, const int* q_len, const int* ctx_len, const int* block_table,
                                   int max_blocks, int H, int Rp, int rp, int dec_tokens, int tile_tokens, int window,
                                   float scale_log2, int simple, const pa::la::Expand* expand, const void* uv, void* y, int ldy, int vp,
                                   int T, hipStream_t st) {
  // uv [H, vp / 16, RT, 64, 8] (optional): y [T, H vp] is written in place of out, see merge_heads_kernel
  if (max_items <= 0) return 0;
  const int D = Rp + rp, NB = (dec_tokens * H + 15) / 16;
  if (Rp % 32 || rp % 32 || H <= 0 || dec_tokens <= 0 || tile_tokens <= 0) return -1;
  pa::la::Args A{out, part_o, part_ml, q, pages, (const int4*)items, n_items, q_start, q_len, ctx_len,
                 block_table, max_blocks, H, NB, Rp, D, dec_tokens, window, scale_log2, expand ? *expand : pa::la::Expand{}};
  if (expand && (fp32 || simple || Rp != pa::la::X_RANK || rp != pa::la::X_ROT || H > 256)) return -1;
  const int RT = Rp / 32, PT = rp / 32;
  int per = 1;  // columns of a workgroup of merge_heads_kernel: as leave about one a CU
  while (per < 16 && (long long)T * H > 256ll * per) per *= 2;
  if (uv && (fp32 || simple || expand || PT > 2 || Rp > 512 || pa_latent_pad(Rp) != Rp || vp < 16 || vp > 128 || vp % 16 || ldy % 4 ||
             T <= 0)) return -1;
  if (!fp32 && !simple && PT <= 2) {
#define PA_LAX(R, P, ...)                                                                                     \
  do {                                                                                                        \
    constexpr int CT = 1;                                                                                     \
    constexpr int lds = pa::la::lds_bytes<R, P __VA_ARGS__>();                                                \
    static bool attr = false;                                                                                 \
    if (!attr) {                                                                                              \
      (void)hipFuncSetAttribute((const void*)pa::la::mfma_kernel<R, P, CT __VA_ARGS__>,                       \
                                hipFuncAttributeMaxDynamicSharedMemorySize, lds);                             \
      attr = true;                                                                                            \
    }                                                                                                         \
    const int cw = 16 * pa::la::NW * CT, gt = (tile_tokens * H + cw - 1) / cw, gx = NB > gt ? NB : gt;                       \
    /* items are strided over the grid: at least one workgroup per CU */                                      \
    const int gy = R >= pa::la::PAIRS || max_items < 256 ? 256 : (max_items < 4096 ? max_items : 4096);       \
    hipLaunchKernelGGL((pa::la::mfma_kernel<R, P, CT __VA_ARGS__>), dim3(gx, gy), dim3(64 * pa::la::NW), lds, st, A);     \
    if (uv) hipLaunchKernelGGL((pa::la::merge_heads_kernel<R>), dim3(H, (T + per - 1) / per), dim3(64 * pa::la::MH_WAVES), 0, st, A, \
                               (const pa::bf16*)uv, (pa::bf16*)y, ldy, vp, max_items, per);                    \
    else hipLaunchKernelGGL((pa::la::merge_kernel<R __VA_ARGS__>), dim3(16, std::min(gy, 256)), dim3(256), 0, st, A);      \
    return (int)hipGetLastError();                                                                            \
  } while (0)
#define PA_LA(R, P) PA_LAX(R, P, )
#define PA_COMMA ,
    if (expand) PA_LAX(pa::la::X_RANK / 32, pa::la::X_ROT / 32, PA_COMMA true);
    switch (RT) {
#define PA_X(N) case N: if (PT == 0) PA_LA(N, 0); else if (PT == 1) PA_LA(N, 1); else PA_LA(N, 2); break;
      PA_LA_RT(PA_X)
#undef PA_X
      default: break;
    }
#undef PA_LA
#undef PA_LAX
#undef PA_COMMA
  }
  if (Rp > 2048 || D * 4 + 2048 > 64 * 1024) return -2;
  const dim3 grid(H, max_items < 4096 ? max_items : 4096);
  const int lds = (D + 256 + 4) * 4;
  if (fp32) hipLaunchKernelGGL((pa::la::simple_kernel<float>), grid, dim3(256), lds, st, A);
  else hipLaunchKernelGGL((pa::la::simple_kernel<pa::bf16>), grid, dim3(256), lds, st, A);
  return (int)hipGetLastError();
}


// The plan of a step for requests with expanded keys: see expand_plan_kernel. X's work lists hold max_att and max_tiles
// entries, its workspace `room` blocks and `slots` partial results. skip [T]: 1 for the rows of expanded requests and of none.
extern "C" int pa_latent_plan(const pa::la::Expand* X, const int* q_start, const int* q_len, const int* ctx_len, int S, int T, int H,
                              int window, int room, int max_att, int max_tiles, int slots, int* skip, hipStream_t st) {
  hipLaunchKernelGGL(pa::la::expand_plan_kernel, dim3(1), dim3(1024), 0, st, *X, q_start, q_len, ctx_len, S, T, H, window, room,
                     max_att, max_tiles, slots, skip);
  return (int)hipGetLastError();
}

// wk, wv: [H, 8, 16, 64, 8], the heads' rows of W_uk and of W_uv
extern "C" int pa_latent_expand(const pa::la::Expand* X, const void* pages, const void* wk, const void* wv, const int* block_table, int max_blocks,
                                int H, int D, int max_tiles, hipStream_t st) {
  if (H <= 0 || D != pa::la::X_RANK + pa::la::X_ROT) return -1;
  constexpr int lds = pa::la::X_RING * pa::la::X_RANK * 32;
  static bool attr = false;
  if (!attr) {
    (void)hipFuncSetAttribute((const void*)pa::la::expand_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    attr = true;
  }
  const int shares = std::min(4 * max_tiles, std::max(1, 256 / H));  // one workgroup a CU
  hipLaunchKernelGGL(pa::la::expand_kernel, dim3(H * shares), dim3(512), lds, st, *X, (const pa::bf16*)pages, (const pa::bf16*)wk,
                     (const pa::bf16*)wv, block_table, max_blocks, H, D, shares);
  return (int)hipGetLastError();
}
