// Selection of the k best of a few hundred keys by a wave, and of a few thousand by a workgroup, without sorting: the
// k-th best key is found bit by bit from the counts of keys that reach a trial value (a ballot per key and bit).
#pragma once
#include "common.h"

namespace pa {

// Floats as unsigned integers in the same order; 0 lies below all of them and stands for "no entry".
__device__ __forceinline__ uint32_t ord_key(float x) {
  const uint32_t u = __float_as_uint(x);
  return (u >> 31) ? ~u : u | 0x80000000u;
}
__device__ __forceinline__ float key_value(uint32_t k) {
  return __uint_as_float((k >> 31) ? k & 0x7fffffffu : ~k);
}

// (by its bits: the compiler is told that there is nothing else)
__device__ __forceinline__ bool is_finite(float x) { return (__float_as_uint(x) & 0x7fffffffu) < 0x7f800000u; }

__device__ __forceinline__ uint32_t wave_umin(uint32_t v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = min(v, (uint32_t)__shfl_xor((int)v, o, 64));
  return v;
}

// entries of the lanes before this one that `p` holds for
__device__ __forceinline__ int rank_in(unsigned long long ballot) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(ballot >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)ballot, 0));
}

// The `want`-th largest of a wave's keys (N a lane; at least `want` of them are not 0, and those are v in the bits above `top`).
template <int N>
__device__ __forceinline__ uint32_t wave_select(const uint32_t (&key)[N], int want, uint32_t v = 0, int top = 31) {
  for (int b = top; b >= 0; --b) {
    const uint32_t t = v | (1u << b);
    int c = 0;
#pragma unroll
    for (int i = 0; i < N; ++i) c += __popcll(__ballot(key[i] >= t));
    if (c >= want) {
      v = t;
      if (c == want) break;
    }
  }
  uint32_t m = 0xffffffffu;
#pragma unroll
  for (int i = 0; i < N; ++i) m = key[i] >= v ? min(m, key[i]) : m;
  return wave_umin(m);
}

// A lower bound of it: the largest value of 32 - LOW leading bits that at least `want` keys reach.
template <int LOW, int N>
__device__ __forceinline__ uint32_t wave_select_floor(const uint32_t (&key)[N], int want) {
  uint32_t v = 0;
  for (int b = 31; b >= LOW; --b) {
    const uint32_t t = v | (1u << b);
    int c = 0;
#pragma unroll
    for (int i = 0; i < N; ++i) c += __popcll(__ballot(key[i] >= t));
    if (c >= want) v = t;
  }
  return v;
}

// wave_select over a workgroup of NW waves; every thread calls it. `red` holds 2 * NW integers in LDS.
template <int N, int NW>
__device__ __forceinline__ uint32_t block_select(const uint32_t (&key)[N], int want, int* red) {
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
  __syncthreads();  // (earlier readers of red)
  uint32_t v = 0;
  int flip = 0;
  for (int b = 31; b >= 0; --b) {
    const uint32_t t = v | (1u << b);
    int c = 0;
#pragma unroll
    for (int i = 0; i < N; ++i) c += __popcll(__ballot(key[i] >= t));
    if (lane == 0) red[flip * NW + wid] = c;
    __syncthreads();
    c = 0;
#pragma unroll
    for (int w = 0; w < NW; ++w) c += red[flip * NW + w];
    flip ^= 1;
    if (c >= want) {
      v = t;
      if (c == want) break;
    }
  }
  uint32_t m = 0xffffffffu;
#pragma unroll
  for (int i = 0; i < N; ++i) m = key[i] >= v ? min(m, key[i]) : m;
  m = wave_umin(m);
  __syncthreads();
  if (lane == 0) red[wid] = (int)m;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < NW; ++w) m = min(m, (uint32_t)red[w]);
  return m;
}

// wave_select behind the bits that all keys share: scores of a query have about ten.
template <int N>
__device__ __forceinline__ uint32_t wave_select_rest(const uint32_t (&key)[N], int want) {
  uint32_t lo = 0xffffffffu, hi = 0;
#pragma unroll
  for (int i = 0; i < N; ++i) {
    lo = key[i] ? min(lo, key[i]) : lo;
    hi = max(hi, key[i]);
  }
  lo = wave_umin(lo);
  hi = ~wave_umin(~hi);
  if (lo >= hi) return hi;
  const int top = 31 - __builtin_clz(lo ^ hi);
  return wave_select(key, want, hi & ~((2u << top) - 1), top);  // (2u << 31: 0)
}

// The `want`-th largest of n <= 1,024 keys in LDS (at least `want` of them are not 0), by the first wave: its ballots need no
// barriers, where block_select has one for every bit. Every thread of a workgroup calls it, the keys written before a
// barrier; `res`: a word in LDS.
__device__ __forceinline__ uint32_t lds_select(const uint32_t* keys, int n, int want, uint32_t* res) {
  if (n <= 64) {  // by its rank: where a bit has its ballot, count and branch to wait for, 2.0 us for 62 keys, so 1.5
    if (threadIdx.x < 64) {
      const uint32_t k = (int)threadIdx.x < n ? keys[threadIdx.x] : 0;
      int above = 0, upto = 0;
      for (int j0 = 0; j0 < n; j0 += 16)
#pragma unroll
        for (int j = 0; j < 16; ++j) {
          const uint32_t kj = __builtin_amdgcn_readlane((int)k, j0 + j);
          above += kj > k;
          upto += kj >= k;
        }
      if (above < want && upto >= want) *res = k;  // (lanes of equal keys write the same)
    }
  } else if (threadIdx.x < 64) {
    uint32_t key[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int e = i * 64 + threadIdx.x;
      key[i] = e < n ? keys[e] : 0;
    }
    const uint32_t v = n <= 256 ? wave_select_rest(reinterpret_cast<const uint32_t(&)[4]>(key), want) : wave_select_rest(key, want);
    if (threadIdx.x == 0) *res = v;
  }
  __syncthreads();
  return *res;
}

// The `K` best of (key, row) entries that gather() names, in order (key down, row up), to out_s / out_r, padded with
// (-inf, -1). Every thread of a workgroup of at least SEL threads calls it with its N entries; `kth`: the K-th best key
// (block_select), or 1 where there are at most K entries. More than SEL entries that tie with kth: any of them.
constexpr int SEL = 512;
struct Selection {
  uint32_t key[SEL];
  int row[SEL], n;
};
// The entries of s in order, behind a barrier
__device__ __forceinline__ void write_ranked(const Selection& s, int K, float* out_s, int* out_r) {
  const int n = min(s.n, SEL), t = threadIdx.x;
  if (t < n) {
    const uint32_t k = s.key[t];
    const int r = s.row[t];
    int rank = 0;
    for (int j = 0; j < n; ++j) rank += s.key[j] > k || (s.key[j] == k && s.row[j] < r);
    if (rank < K) { out_s[rank] = key_value(k); out_r[rank] = r; }
  }
  if (t < K && t >= n) { out_s[t] = -INFINITY; out_r[t] = -1; }
}
// The K <= 64 best of n <= 64 entries in LDS, by the first wave
__device__ __forceinline__ void write_best_few(const uint32_t* keys, const int* rows, int n, int K, float* out_s, int* out_r) {
  const int t = threadIdx.x;
  if (t >= 64) return;
  const uint32_t k = t < n ? keys[t] : 0;
  const int r = t < n ? rows[t] : -1;
  int rank = 0;
  for (int j0 = 0; j0 < n; j0 += 16)
#pragma unroll
    for (int j = 0; j < 16; ++j) {  // (behind the last: keys of 0)
      const uint32_t kj = __builtin_amdgcn_readlane((int)k, j0 + j);
      const int rj = __builtin_amdgcn_readlane(r, j0 + j);
      rank += (int)(kj > k) | ((int)(kj == k) & (int)(rj < r));
    }
  if (t < n && rank < K) { out_s[rank] = key_value(k); out_r[rank] = r; }
  if (t < K && t >= n) { out_s[t] = -INFINITY; out_r[t] = -1; }
}
template <int N>
__device__ __forceinline__ void write_best(const uint32_t (&key)[N], const int (&row)[N], uint32_t kth, int K, Selection& s,
                                           float* out_s, int* out_r) {
  __syncthreads();
  if (threadIdx.x == 0) s.n = 0;
  __syncthreads();
  auto take = [&](bool yes, uint32_t k, int r) {
    if (yes) {
      const int p = atomicAdd(&s.n, 1);
      if (p < SEL) { s.key[p] = k; s.row[p] = r; }
    }
  };
#pragma unroll
  for (int i = 0; i < N; ++i) take(key[i] > kth, key[i], row[i]);  // fewer than K
  __syncthreads();
#pragma unroll
  for (int i = 0; i < N; ++i) take(key[i] == kth, key[i], row[i]);
  __syncthreads();
  write_ranked(s, K, out_s, out_r);
}

}  // namespace pa
