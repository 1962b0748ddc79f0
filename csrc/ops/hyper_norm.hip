// The step between two sublayers of a decoder whose fp32 residual has several streams x_1 .. x_S
// (hyper-connections; S = 1 with unit weights is the plain residual sum):
//
//   y   <- sum_k w_k y_k + y2 + bias                   (K partial outputs per token, weights optional)
//   x_t <- sum_s mix[s][t] x_s + post[t] y              or, at the start, x_t <- E[id]
//   out <- norm(sum_s pre[s] x_s) * w_next              (the next sublayer's input)
//
// in one launch: one workgroup per row; the streams are read and written once, all from the old ones, and
// the next input waits in LDS for its norm. All arithmetic is fp32; y, E and out are T (bf16 or fp32).
// out's columns D .. ldo are set to zero (projections read K padded to whole MFMA chunks). `rows`
// (optional): out row i is row rows[i]'s, and x is left as it was.
//
// Also here: the soft cap of logits, z <- cap * tanh(z / cap).
#include "common.h"

namespace pa {
namespace hn {

constexpr int MAX_S = 8;

struct Args {
  float* x;             // [T, S, D]
  const void* y;        // [T, K, ldy]
  const float* y_w;     // [T, K] or null
  const void* y2;       // [T, ldy2] or null
  const float* bias;    // [D] or null
  const float *mix, *post, *pre;  // [S, S] from x to, [S], [S]
  const void* emb;
  const int* ids;
  const float* w_next;
  void* out;
  const int* rows;
  const int* live;      // by row: below 0 from the first row without a token on (with rows: not looked at)
  int K, ldy, ldy2, vocab, ldo, D;
  float eps;
  const float* sums;    // [T, K, ldy] in place of y, or null
};

// LIVE: with `live` (bf16 rows of whole 4s, the others do all rows). SUMS: y may be sums; launches without are apart (304 rows, 4
// streams of 2,048: 8.8 us with the test, 8.6 without; and 9.1 where `sums` lay among the other arguments, not behind them).
template <typename T, int VEC, int S, int NW, bool LIVE = false, bool SUMS = true>
__global__ __launch_bounds__(64 * NW) void hyper_norm_kernel(const Args A) {
  constexpr int NT = 64 * NW;
  extern __shared__ __attribute__((aligned(16))) float row[];
  __shared__ float red[NW];
  if (LIVE && A.live[blockIdx.x] < 0) return;
  const int t = A.rows ? A.rows[blockIdx.x] : blockIdx.x, D = A.D;
  float* xr = A.x + (size_t)t * S * D;
  const bool add = A.y || (SUMS && A.sums);
  float mix[S][S], post[S], pre[S];
#pragma unroll
  for (int s = 0; s < S; ++s) {
    pre[s] = A.pre ? A.pre[s] : 0.f;
    post[s] = add ? A.post[s] : 0.f;
#pragma unroll
    for (int r = 0; r < S; ++r) mix[s][r] = add ? A.mix[s * S + r] : 0.f;
  }
  const T* yr = (const T*)A.y + (size_t)t * A.K * A.ldy;
  const float* sr = A.sums + (size_t)t * A.K * A.ldy;
  const float* yw = A.y_w ? A.y_w + (size_t)t * A.K : nullptr;
  const T* er = A.emb ? (const T*)A.emb + (size_t)min(max(A.ids[t], 0), A.vocab - 1) * D : nullptr;
  float ss = 0.f;
  for (int i = threadIdx.x * VEC; i < D; i += NT * VEC) {
    float x[S][VEC], u[VEC];
    T a[VEC];
#pragma unroll
    for (int j = 0; j < VEC; ++j) u[j] = 0.f;
    if (er) {
      __builtin_memcpy(a, __builtin_assume_aligned(er + i, sizeof(T) * VEC), sizeof(T) * VEC);
#pragma unroll
      for (int s = 0; s < S; ++s)
#pragma unroll
        for (int j = 0; j < VEC; ++j) x[s][j] = (float)a[j];
    } else {
#pragma unroll
      for (int s = 0; s < S; ++s)
        __builtin_memcpy(x[s], __builtin_assume_aligned(xr + (size_t)s * D + i, 4 * VEC), 4 * VEC);
    }
    if (add) {
      float y[VEC];
#pragma unroll
      for (int j = 0; j < VEC; ++j) y[j] = A.bias ? A.bias[i + j] : 0.f;
      if (A.y2) {
        __builtin_memcpy(a, __builtin_assume_aligned((const T*)A.y2 + (size_t)t * A.ldy2 + i, sizeof(T) * VEC), sizeof(T) * VEC);
#pragma unroll
        for (int j = 0; j < VEC; ++j) y[j] += (float)a[j];
      }
      if (SUMS && A.sums) {
#pragma unroll 8
        for (int k = 0; k < A.K; ++k) {
          float f[VEC];
          __builtin_memcpy(f, __builtin_assume_aligned(sr + (size_t)k * A.ldy + i, 4 * VEC), 4 * VEC);
#pragma unroll
          for (int j = 0; j < VEC; ++j) y[j] += f[j];
        }
      }
#pragma unroll 4
      for (int k = 0; (!SUMS || A.y) && k < A.K; ++k) {
        __builtin_memcpy(a, __builtin_assume_aligned(yr + (size_t)k * A.ldy + i, sizeof(T) * VEC), sizeof(T) * VEC);
        const float w = yw ? yw[k] : 1.f;
#pragma unroll
        for (int j = 0; j < VEC; ++j) y[j] = fmaf(w, (float)a[j], y[j]);
      }
#pragma unroll
      for (int j = 0; j < VEC; ++j) {
        float z[S];
#pragma unroll
        for (int r = 0; r < S; ++r) {
          z[r] = post[r] * y[j];
#pragma unroll
          for (int s = 0; s < S; ++s) z[r] = fmaf(mix[s][r], x[s][j], z[r]);
        }
#pragma unroll
        for (int r = 0; r < S; ++r) x[r][j] = z[r];
      }
    }
    if ((add || er) && !A.rows) {
#pragma unroll
      for (int s = 0; s < S; ++s)
        __builtin_memcpy(__builtin_assume_aligned(xr + (size_t)s * D + i, 4 * VEC), x[s], 4 * VEC);
    }
#pragma unroll
    for (int s = 0; s < S; ++s)
#pragma unroll
      for (int j = 0; j < VEC; ++j) u[j] = fmaf(pre[s], x[s][j], u[j]);
#pragma unroll
    for (int j = 0; j < VEC; ++j) {
      row[i + j] = u[j];
      ss += u[j] * u[j];
    }
  }
  if (!A.w_next) return;
  const float inv = 1.f / sqrtf(block_sum<NW>(ss, red) / (float)D + A.eps);
  T* o = (T*)A.out + (size_t)blockIdx.x * A.ldo;
  for (int i = threadIdx.x * VEC; i < D; i += NT * VEC) {
    T a[VEC];
#pragma unroll
    for (int j = 0; j < VEC; ++j) a[j] = (T)(row[i + j] * inv * A.w_next[i + j]);
    __builtin_memcpy(__builtin_assume_aligned(o + i, sizeof(T) * VEC), a, sizeof(T) * VEC);
  }
  for (int i = D + threadIdx.x; i < A.ldo; i += NT) o[i] = (T)0.f;
}

template <typename T, int VEC>
__global__ __launch_bounds__(256) void softcap_kernel(T* __restrict__ x, int ld, int cols, float cap) {
  T* r = x + (size_t)blockIdx.y * ld;
  for (int i = (blockIdx.x * 256 + threadIdx.x) * VEC; i < cols; i += gridDim.x * 256 * VEC) {
    T a[VEC];  // (columns behind cols, up to a whole vector of the row, are padding)
    __builtin_memcpy(a, __builtin_assume_aligned(r + i, sizeof(T) * VEC), sizeof(T) * VEC);
#pragma unroll
    for (int j = 0; j < VEC; ++j)
      if (VEC == 1 || i + j < cols) a[j] = (T)(cap * tanhf((float)a[j] / cap));
    __builtin_memcpy(__builtin_assume_aligned(r + i, sizeof(T) * VEC), a, sizeof(T) * VEC);
  }
}

}  // namespace hn
}  // namespace pa

extern "C" int pa_hyper_norm(int fp32, float* x, int S, const void* y, const float* sums, int K, int ldy, const float* y_w,
                             const void* y2, int ldy2, const float* bias, const float* mix, const float* post, const float* pre, const void* emb,
                             const int* ids, int vocab, const float* w_next, void* out, int ldo, const int* rows, const int* live,
                             int n, int D, float eps, hipStream_t st) {
  using namespace pa::hn;
  if (n <= 0) return 0;
  if (D <= 0 || D * 4 > 96 * 1024 || S < 1 || S > MAX_S) return -1;
  // Rows without a token stay as they are in launches that look for them (a step of mudepel's 8 layers, 4 streams of 2,048
  // columns: 3,658 tokens in 4,096 rows 2 % of its 5,840 us, 2,101 in 3,072 3 % of 4,640)
  if (rows || n <= pa::LIVE_MIN_ROWS) live = nullptr;
  const Args A{x, y, y_w, y2, bias, mix, post, pre, emb, ids, w_next, out, rows, live, K, ldy, ldy2, vocab, ldo, D, eps, sums};
  // fewer rows than CUs: twice the waves to a row, all of it in one pass up to 2,048 columns (64 rows, 4 streams of 2,048:
  // 6.8 -> 5.7 us)
  const bool few = n <= 256 && D > 1024;
  const bool vec = D % 4 == 0 && ((!y && !sums) || ldy % 4 == 0) && (!y2 || ldy2 % 4 == 0) && (!out || ldo % 4 == 0);
#define PA_HN(T, V, N, W, ...)                                                                                  \
  do {                                                                                                          \
    static bool attr = false;                                                                                   \
    if (!attr) {                                                                                                \
      (void)hipFuncSetAttribute((const void*)hyper_norm_kernel<T, V, N, W __VA_OPT__(,) __VA_ARGS__>,           \
                                hipFuncAttributeMaxDynamicSharedMemorySize, 96 * 1024);                         \
      attr = true;                                                                                              \
    }                                                                                                           \
    hipLaunchKernelGGL((hyper_norm_kernel<T, V, N, W __VA_OPT__(,) __VA_ARGS__>), dim3(n), dim3(64 * W),        \
                       (size_t)D * 4, st, A);                                                                   \
  } while (0)
#define PA_HN_S(N)                                                             \
  case N:                                                                      \
    if (fp32) { if (vec) PA_HN(float, 4, N, 4); else PA_HN(float, 1, N, 4); }  \
    else if (!vec) PA_HN(pa::bf16, 1, N, 4);                                   \
    else if (few && sums) PA_HN(pa::bf16, 4, N, 8);                            \
    else if (few) PA_HN(pa::bf16, 4, N, 8, false, false);                      \
    else if (live && sums) PA_HN(pa::bf16, 4, N, 4, true);                     \
    else if (live) PA_HN(pa::bf16, 4, N, 4, true, false);                      \
    else if (sums) PA_HN(pa::bf16, 4, N, 4);                                   \
    else PA_HN(pa::bf16, 4, N, 4, false, false);                               \
    break
  switch (S) {
    PA_HN_S(1); PA_HN_S(2); PA_HN_S(3); PA_HN_S(4); PA_HN_S(5); PA_HN_S(6); PA_HN_S(7); PA_HN_S(8);
  }
#undef PA_HN_S
#undef PA_HN
  return (int)hipGetLastError();
}

extern "C" int pa_softcap(int fp32, void* x, int ld, int rows, int cols, float cap, hipStream_t st) {
  if (rows <= 0 || cols <= 0) return 0;
  const bool vec = ld % 8 == 0;  // (a whole vector then never leaves the row)
  const dim3 grid((cols + 2047) / 2048, rows);
  if (fp32) {
    if (vec) hipLaunchKernelGGL((pa::hn::softcap_kernel<float, 8>), grid, dim3(256), 0, st, (float*)x, ld, cols, cap);
    else hipLaunchKernelGGL((pa::hn::softcap_kernel<float, 1>), grid, dim3(256), 0, st, (float*)x, ld, cols, cap);
  } else {
    if (vec) hipLaunchKernelGGL((pa::hn::softcap_kernel<pa::bf16, 8>), grid, dim3(256), 0, st, (pa::bf16*)x, ld, cols, cap);
    else hipLaunchKernelGGL((pa::hn::softcap_kernel<pa::bf16, 1>), grid, dim3(256), 0, st, (pa::bf16*)x, ld, cols, cap);
  }
  return (int)hipGetLastError();
}
