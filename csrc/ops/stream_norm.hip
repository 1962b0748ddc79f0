// The step between two sublayers of hyper_norm.hip without its streams. mix and post are weights, so every stream is a sum of the
// embedding row and the outputs of the sublayers so far with coefficients that are known when the model is loaded (models/streams.py):
//
//   x_s = sum_t coef[t][s] term_t     terms: fp32 rows and biases, bf16 rows (the first may be E[id]), at last y (or sums)
//   out <- norm(sum_s pre[s] x_s) * w_next, and x (optional) <- all of them, y_kept <- y's sum
//
// Steps of many rows are bound by these bytes: 4 streams of 2,048 are 64 KB a row to read and write, a term of bf16 4 KB. A lane
// has the columns and adds in the order that hyper_norm_kernel has, so that streams without mixing come to the same bits.
// 3,658 of 4,096 rows, 4 streams of 2,048, 16 sublayers: 45 us a sublayer with the streams, 34 of sums of 1 to 17 terms (4.7 TB/s).
#include "common.h"

#include <type_traits>

namespace pa {
namespace sn {

constexpr int MAX_S = 8, MAX_TERMS = 63;

struct SumArgs {
  const void* term[MAX_TERMS];  // the first nf are fp32
  int ld[MAX_TERMS];    // 0: the same row for all
  int nf, n;
  const int* ids;       // term nf's row of a row, or null: its own
  int vocab;
  const float* coef;    // [n + (y or sums)][S]
  const float* pre;     // [S]
  float* x;             // [T, S, D] or null
  const bf16* y;        // [T, K, ldy] with weights y_w [T, K] or null, or sums alike, or neither
  const float *sums, *y_w;
  float* y_kept;        // [T, D] or null
  int K, ldy;
  const float* w_next;
  bf16* out;
  const int *rows, *live;
  int ldo, D;
  float eps;
};

// A lane's columns of a pass are 4 from i on and 4 from i + STEP on (behind a row's end: its last ones, which then count for nothing).
constexpr int NW_SUM = 4, STEP = 256 * NW_SUM;

template <typename T>
struct Quad {
  typedef T vec __attribute__((ext_vector_type(4)));
  vec v[2];
  __device__ __forceinline__ void load(uint64_t row, int a, int b) {
    typedef __attribute__((address_space(1))) const vec global;
    v[0] = *(global*)(row + a * sizeof(T));
    v[1] = *(global*)(row + b * sizeof(T));
  }
  __device__ __forceinline__ float operator[](int j) const { return (float)v[j >> 2][j & 3]; }
};

// Where the terms lie and their coefficients are in the lanes, one a lane, and come from there: read for each group of terms from the
// arguments they were a chain of scalar loads (3 rows 17 us, so 9). Groups of 4 terms: a kernel that loads all before it uses the
// first has two waves a SIMD, which wait for each other (60 us for 34).
template <int S, bool FRESH>
__global__ __launch_bounds__(64 * NW_SUM, S <= 4 && !FRESH ? 6 : 1) void stream_norm_kernel(const SumArgs A) {
  extern __shared__ __attribute__((aligned(16))) float row[];
  __shared__ float red[NW_SUM];
  if (A.live && A.live[blockIdx.x] < 0) return;
  const size_t t = A.rows ? A.rows[blockIdx.x] : blockIdx.x;
  const int D = A.D, lane = threadIdx.x & 63;
  uint64_t place = 0;
  float coef[S];
#pragma unroll
  for (int s = 0; s < S; ++s) coef[s] = lane < A.n + FRESH ? A.coef[lane * S + s] : 0.f;
  if (lane < A.n) {
    const size_t r = A.ids && lane == A.nf ? (size_t)min(max(A.ids[t], 0), A.vocab - 1) : t;
    place = (uint64_t)A.term[lane] + r * A.ld[lane] * (lane < A.nf ? 4 : 2);
  }
  auto at = [&](int k) {
    return (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)place, k) |
           (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(place >> 32), k) << 32;
  };
  auto factor = [&](int k, int s) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(coef[s]), k)); };
  float ss = 0.f;
  for (int i0 = 0; i0 < D; i0 += 2 * STEP) {
    const int i = i0 + threadIdx.x * 4;
    const bool first = i < D, second = i + STEP < D;
    const int ia = min(i, D - 4), ib = min(i + STEP, D - 4);
    float x[S][8], u[8];
#pragma unroll
    for (int s = 0; s < S; ++s)
#pragma unroll
      for (int j = 0; j < 8; ++j) x[s][j] = 0.f;
    auto add = [&](auto n, auto type, int k) {
      constexpr int N = decltype(n)::value;
      using T = decltype(type);
      Quad<T> v[N];
#pragma unroll
      for (int q = 0; q < N; ++q) v[q].load(at(k + q), ia, ib);
#pragma unroll
      for (int q = 0; q < N; ++q)
#pragma unroll
        for (int s = 0; s < S; ++s) {
          const float c = factor(k + q, s);
#pragma unroll
          for (int j = 0; j < 8; ++j) x[s][j] = fmaf(c, v[q][j], x[s][j]);
        }
    };
    int k = 0;
    for (; k < A.nf; ++k) add(std::integral_constant<int, 1>{}, 0.f, k);
    for (; k + 4 <= A.n; k += 4) add(std::integral_constant<int, 4>{}, bf16{}, k);
    for (; k < A.n; ++k) add(std::integral_constant<int, 1>{}, bf16{}, k);
    if constexpr (FRESH) {
      float y[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) y[j] = 0.f;
      auto partial = [&](auto type, const void* base) {
        using T = decltype(type);
#pragma unroll 4
        for (int q = 0; q < A.K; ++q) {
          Quad<T> v;
          v.load((uint64_t)base + (t * A.K + q) * A.ldy * sizeof(T), ia, ib);
          const float w = A.y_w ? A.y_w[t * A.K + q] : 1.f;
#pragma unroll
          for (int j = 0; j < 8; ++j) y[j] = fmaf(w, v[j], y[j]);
        }
      };
      if (A.sums) partial(0.f, A.sums);
      else partial(bf16{}, A.y);
      float* kept = A.y_kept + t * D + i;
      if (A.y_kept && first) __builtin_memcpy(__builtin_assume_aligned(kept, 16), y, 16);
      if (A.y_kept && second) __builtin_memcpy(__builtin_assume_aligned(kept + STEP, 16), y + 4, 16);
#pragma unroll
      for (int s = 0; s < S; ++s) {
        const float c = factor(A.n, s);
#pragma unroll
        for (int j = 0; j < 8; ++j) x[s][j] = fmaf(c, y[j], x[s][j]);
      }
    }
    if (A.x)
#pragma unroll
      for (int s = 0; s < S; ++s) {
        float* xs = A.x + (t * S + s) * D + i;
        if (first) __builtin_memcpy(__builtin_assume_aligned(xs, 16), x[s], 16);
        if (second) __builtin_memcpy(__builtin_assume_aligned(xs + STEP, 16), x[s] + 4, 16);
      }
#pragma unroll
    for (int j = 0; j < 8; ++j) u[j] = 0.f;
#pragma unroll
    for (int s = 0; s < S; ++s)
#pragma unroll
      for (int j = 0; j < 8; ++j) u[j] = fmaf(A.pre[s], x[s][j], u[j]);
    // (squares in the order that the compiler gave hyper_norm_kernel)
    auto write = [&](const float* v, float* to) {
      __builtin_memcpy(__builtin_assume_aligned(to, 16), v, 16);
#pragma unroll
      for (int j = 0; j < 4; ++j) ss = fmaf(v[(0x0213 >> 4 * j) & 3], v[(0x0213 >> 4 * j) & 3], ss);
    };
    if (first) write(u, row + i);
    if (second) write(u + 4, row + i + STEP);
  }
  const float inv = 1.f / sqrtf(block_sum<NW_SUM>(ss, red) / (float)D + A.eps);
  bf16* o = A.out + (size_t)blockIdx.x * A.ldo;
  for (int i = threadIdx.x * 4; i < D; i += STEP) {
    bf16x4 a;
#pragma unroll
    for (int j = 0; j < 4; ++j) a[j] = (bf16)(row[i + j] * inv * A.w_next[i + j]);
    *reinterpret_cast<bf16x4*>(o + i) = a;
  }
  for (int i = D + threadIdx.x; i < A.ldo; i += 64 * NW_SUM) o[i] = (bf16)0.f;
}

}  // namespace sn
}  // namespace pa

// term, ld: host arrays of n_terms, the first nf fp32. D and all rows in whole 4s, fp32 rows 16-byte and bf16 rows 8-byte aligned.
extern "C" int pa_stream_norm(const void* const* term, const int* ld, int nf, int n_terms, const int* ids, int vocab,
                              const float* coef, const float* pre, int S, float* x, const void* y, const float* sums, int K, int ldy,
                              const float* y_w, float* y_kept, const float* w_next, void* out, int ldo, const int* rows,
                              const int* live, int n, int D, float eps, hipStream_t st) {
  using namespace pa::sn;
  if (n <= 0) return 0;
  if (D <= 0 || D % 4 || ldo % 4 || D * 4 > 96 * 1024 || n_terms < 0 || n_terms > MAX_TERMS || S < 2 || S > MAX_S ||
      n_terms + (y || sums) < 1 || (y && sums) || nf < 0 || nf > n_terms || (ids && nf == n_terms)) return -1;
  SumArgs A{};
  for (int i = 0; i < n_terms; ++i) { A.term[i] = term[i]; A.ld[i] = ld[i]; }
  A.nf = nf;
  A.n = n_terms;
  A.ids = ids;
  A.vocab = vocab;
  A.coef = coef;
  A.pre = pre;
  A.x = x;
  A.y = (const pa::bf16*)y;
  A.sums = sums;
  A.K = K;
  A.ldy = ldy;
  A.y_w = y_w;
  A.y_kept = y_kept;
  A.w_next = w_next;
  A.out = (pa::bf16*)out;
  A.ldo = ldo;
  A.rows = rows;
  A.live = rows || n <= pa::LIVE_MIN_ROWS ? nullptr : live;
  A.D = D;
  A.eps = eps;
#define PA_SN(N, F)                                                                                                              \
  do {                                                                                                                           \
    static bool attr = false;                                                                                                    \
    if (!attr) {                                                                                                                 \
      (void)hipFuncSetAttribute((const void*)stream_norm_kernel<N, F>, hipFuncAttributeMaxDynamicSharedMemorySize, 96 * 1024);   \
      attr = true;                                                                                                               \
    }                                                                                                                            \
    hipLaunchKernelGGL((stream_norm_kernel<N, F>), dim3(n), dim3(64 * NW_SUM), (size_t)D * 4, st, A);                            \
  } while (0)
#define PA_SN_S(N) case N: if (y || sums) PA_SN(N, true); else PA_SN(N, false); break
  switch (S) {
    PA_SN_S(2); PA_SN_S(3); PA_SN_S(4); PA_SN_S(5); PA_SN_S(6); PA_SN_S(7); PA_SN_S(8);
  }
#undef PA_SN_S
#undef PA_SN
  return (int)hipGetLastError();
}
