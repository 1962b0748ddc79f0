// RMSNorm and fused residual-add + RMSNorm for Llama blocks.
//
// y = x * rsqrt(mean(x^2) + eps) * w        (bf16 in/out, fp32 math)
// fused: r = r + d (stored back to r in bf16), y = rmsnorm(r) * w
//
// One workgroup per row. A row of D = BS*8*NV elements is held in registers
// (NV 16-byte vectors per thread) so HBM is touched exactly once for read and
// once for write; the only cross-wave traffic is the 4-float LDS reduction.
// `rows` (optional, not fused): out row i is the norm of x's row rows[i], held in 0 .. nx - 1, so that a step's sampled rows need
// no gather before it. Of a few rows it takes the time of any launch (4.7 us for 64 rows of 4096), with the gather 9.4.
#include "common.h"

namespace pa {

template <int BS, int NV, bool FUSED>
__global__ __launch_bounds__(BS) void rmsnorm_kernel(bf16* __restrict__ out,
                                                     bf16* __restrict__ resid,
                                                     const bf16* __restrict__ x,
                                                     const bf16* __restrict__ w,
                                                     const int* __restrict__ rows, int nx,
                                                     int D, float eps) {
  __shared__ float red[BS / 64];
  const int row = blockIdx.x;
  const int from = !FUSED && rows ? min(max(rows[row], 0), nx - 1) : row;
  const bf16x8* xr = reinterpret_cast<const bf16x8*>(x + (size_t)from * D);
  bf16x8* rr = reinterpret_cast<bf16x8*>(resid + (size_t)row * D);
  float v[NV][8];
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int idx = threadIdx.x + i * BS;
    bf16x8 a = xr[idx];
    if (FUSED) {
      bf16x8 b = rr[idx];
      bf16x8 s;
#pragma unroll
      for (int j = 0; j < 8; ++j) s[j] = f2bf(bf2f(a[j]) + bf2f(b[j]));
      rr[idx] = s;
      a = s;
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      v[i][j] = bf2f(a[j]);
      ss += v[i][j] * v[i][j];
    }
  }
  const float tot = block_sum<BS / 64>(ss, red);
  const float inv = rsqrtf(tot / (float)D + eps);
  const bf16x8* wr = reinterpret_cast<const bf16x8*>(w);
  bf16x8* orow = reinterpret_cast<bf16x8*>(out + (size_t)row * D);
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int idx = threadIdx.x + i * BS;
    bf16x8 ww = wr[idx];
    bf16x8 o;
#pragma unroll
    for (int j = 0; j < 8; ++j) o[j] = f2bf(bf2f(f2bf(v[i][j] * inv)) * bf2f(ww[j]));
    orow[idx] = o;
  }
}

// Generic fallback for row lengths that are a multiple of 8 but not of the
// register-resident shapes (used by small test models): two passes, the second
// re-reads the row from L1/L2.
template <bool FUSED>
__global__ __launch_bounds__(256) void rmsnorm_generic_kernel(bf16* __restrict__ out,
                                                              bf16* __restrict__ resid,
                                                              const bf16* __restrict__ x,
                                                              const bf16* __restrict__ w,
                                                              const int* __restrict__ rows, int nx,
                                                              int D, float eps) {
  __shared__ float red[4];
  const int row = blockIdx.x;
  const int from = !FUSED && rows ? min(max(rows[row], 0), nx - 1) : row;
  const bf16x8* xr = reinterpret_cast<const bf16x8*>(x + (size_t)from * D);
  bf16x8* rr = reinterpret_cast<bf16x8*>(resid + (size_t)row * D);
  const int nvec = D / 8;
  float ss = 0.f;
  for (int idx = threadIdx.x; idx < nvec; idx += 256) {
    bf16x8 a = xr[idx];
    if (FUSED) {
      bf16x8 b = rr[idx];
#pragma unroll
      for (int j = 0; j < 8; ++j) a[j] = f2bf(bf2f(a[j]) + bf2f(b[j]));
      rr[idx] = a;
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) ss += bf2f(a[j]) * bf2f(a[j]);
  }
  __syncthreads();
  const float tot = block_sum<4>(ss, red);
  const float inv = rsqrtf(tot / (float)D + eps);
  const bf16x8* src = FUSED ? reinterpret_cast<const bf16x8*>(rr) : xr;
  const bf16x8* wr = reinterpret_cast<const bf16x8*>(w);
  bf16x8* orow = reinterpret_cast<bf16x8*>(out + (size_t)row * D);
  for (int idx = threadIdx.x; idx < nvec; idx += 256) {
    bf16x8 a = src[idx], ww = wr[idx], o;
#pragma unroll
    for (int j = 0; j < 8; ++j) o[j] = f2bf(bf2f(f2bf(bf2f(a[j]) * inv)) * bf2f(ww[j]));
    orow[idx] = o;
  }
}

template <bool FUSED>
static int launch_rmsnorm(bf16* out, bf16* resid, const bf16* x, const bf16* w, const int* rows, int nx, int T, int D,
                          float eps, hipStream_t st) {
  if (T <= 0) return 0;
  if (D % 8 != 0 || (rows && nx < 1)) return -1;
  dim3 g(T);
#define PA_RMS(BS, NV)                                                                 \
  hipLaunchKernelGGL((rmsnorm_kernel<BS, NV, FUSED>), g, dim3(BS), 0, st, out, resid, x, w, rows, nx, D, \
                     eps)
  if (D == 8192) PA_RMS(256, 4);
  else if (D == 4096) PA_RMS(256, 2);
  else if (D == 2048) PA_RMS(256, 1);
  else if (D == 1024) PA_RMS(128, 1);
  else if (D == 512) PA_RMS(64, 1);
  else hipLaunchKernelGGL((rmsnorm_generic_kernel<FUSED>), g, dim3(256), 0, st, out, resid, x, w, rows, nx, D, eps);
#undef PA_RMS
  return (int)hipGetLastError();
}

// The first launch of a step: out row t is emb's row ids[t] (held in 0 .. V - 1), ss[t] the sum of its squares in the order of
// row_sumsq_kernel (the same bits), and ss_zero[t] the clear of the statistics that the first residual epilogue adds to. A wave a
// row, 8 loads of a lane in flight: any launch's time up to a few hundred rows, where a gather, the sums and the clear took one
// each (64 rows of 4096: 4.7 + 4.6 + 4.6 us before, 4.9 now).
__global__ __launch_bounds__(256) void embed_rows_kernel(bf16* __restrict__ out, const bf16* __restrict__ emb,
                                                         const int* __restrict__ ids, float* __restrict__ ss,
                                                         float* __restrict__ ss_zero, int T, int V, int D, int64_t lde) {
  const int lane = threadIdx.x & 63, t = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (t >= T) return;
  const int id = min(max(ids[t], 0), V - 1), n = D / 8;
  const bf16x8* src = reinterpret_cast<const bf16x8*>(emb + (size_t)id * lde);
  bf16x8* dst = reinterpret_cast<bf16x8*>(out + (size_t)t * D);
  float acc = 0.f;
  for (int i0 = lane; i0 < n; i0 += 512) {
    bf16x8 v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (i0 + j * 64 < n) v[j] = src[i0 + j * 64];
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (i0 + j * 64 < n) {
        dst[i0 + j * 64] = v[j];
#pragma unroll
        for (int e = 0; e < 8; ++e) acc = fmaf((float)v[j][e], (float)v[j][e], acc);
      }
  }
  if (ss) {
    acc = wave_sum(acc);
    if (lane == 0) ss[t] = acc;
  }
  if (ss_zero && lane == 0) ss_zero[t] = 0.f;
}

}  // namespace pa

extern "C" int pa_rmsnorm(void* out, const void* x, const void* w, const int* rows, int nx, int T, int D, float eps,
                          hipStream_t st) {
  return pa::launch_rmsnorm<false>((pa::bf16*)out, nullptr, (const pa::bf16*)x,
                                   (const pa::bf16*)w, rows, nx, T, D, eps, st);
}

extern "C" int pa_embed_rows(void* out, const void* emb, const int* ids, float* ss, float* ss_zero, int T, int V, int D,
                             long long lde, hipStream_t st) {
  if (T <= 0) return 0;
  if (D < 8 || D % 8 || lde % 8 || V < 1) return 1;
  hipLaunchKernelGGL(pa::embed_rows_kernel, dim3((T + 3) / 4), dim3(256), 0, st, (pa::bf16*)out, (const pa::bf16*)emb, ids, ss,
                     ss_zero, T, V, D, (int64_t)lde);
  return hipGetLastError() == hipSuccess ? 0 : -2;
}

extern "C" int pa_fused_add_rmsnorm(void* out, void* resid, const void* x, const void* w, int T,
                                    int D, float eps, hipStream_t st) {
  return pa::launch_rmsnorm<true>((pa::bf16*)out, (pa::bf16*)resid, (const pa::bf16*)x,
                                  (const pa::bf16*)w, nullptr, 0, T, D, eps, st);
}
