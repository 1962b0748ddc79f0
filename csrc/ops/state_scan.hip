// State-space recurrence (Mamba-2) for decode rows and prompt portions of a ragged step, with a causal
// convolution ahead of it. Per head h (group g = h / (H / G)):
//
//   u = silu(conv(x | B | C)),   dt = softplus(dt_raw + bias)
//   S <- exp(-a dt) S + dt B x^T,   y = S^T C + D x
//
// State of a sequence (its slot): S fp32 [H, V, N], N innermost, and the convolution's inputs in a ring:
// the input of position p in row p % RING. A sequence whose portion starts at position 0 starts from
// zeros whatever its slot holds, so a slot is handed on without being cleared.
//
// Projection rows [z: H V | x: H V | B: G N | C: G N | dt: H], V padded to 16 and N to 32 per head and
// group; xBC channels Cc = H V + 2 G N in that order.
//
// Short portions (at most `scan_min` tokens, decode rows among them): step_kernel, convolution included,
// token after token; the ring has room for their inputs beside the taps they read.
// Longer ones (bf16), in chunks of 64 tokens (l = running sum of -a dt over the chunk, L = its end; held in log2):
//   convolution   u for all their rows, in step_kernel's launch (bf16, 4 taps) or ahead of it (conv_kernel)
//   scan_kernel   y_i = exp(l_i) C_i . S + sum_{j <= i} exp(l_i - l_j) dt_j (C_i . B_j) x_j + D x_i,
//                 S <- exp(L) S + sum_j exp(L - l_j) dt_j B_j x_j^T, chunk after chunk
//   or the same in three launches, each over all chunks: chunk_state_kernel, state_pass_kernel, chunk_out_kernel
// The MFMA operands are bf16. B, C and x are bf16 values; everything that carries a decay, a step size or
// the state goes in as a pair of bf16 (value and remainder), 16 bits of mantissa: the recurrence keeps
// the accuracy of fp32 to that order, and chunked and stepped portions agree.
// fp32 models: conv_kernel and step_kernel for long portions too.
#include "common.h"

#include <algorithm>

namespace pa {
namespace ss {

constexpr int LC = 64;        // tokens of a chunk
constexpr int LD = LC + 8;    // LDS row of a chunk's tokens, in elements
constexpr int MAX_SHORT = 8;  // tokens of a short portion at most

struct Args {
  const void* proj;        // [T, ldp]
  void* u;                 // [T, Cc] convolved rows of long portions
  void* y;                 // [T, ldy] (columns h * V + v)
  float* state;            // [slots, H, V, N]
  void* ring;              // [slots, RING, Cc]
  const void* conv_w;      // [taps, Cc] fp32, oldest first
  const float *conv_b, *dt_bias, *a, *d;
  const int *q_start, *q_len, *ctx_len, *state_slot;
  const int4* items;
  const int* n_items;
  int ldp, ldy, H, G, V, N, Cc, taps, RING, scan_min, long_too;
  int vsplit;    // workgroups of step_kernel a head: 1, 2, 4 or 8
  float* work;   // [items, H, V, N]: every chunk's state
  float* total;  // [items, H]: a chunk's summed log2 decay
  int* form;     // null, or 1 where the step's long portions go through the three launches, else 0 (pick_form)
  float chain, fixed;
  int per_group;  // heads
  int conv_x, conv_y, conv_rows;  // the convolution's workgroups; the rows of step_kernel's that they are, 0: none
};

// (a base that is the same for a wave and an offset of 32 bits: one register a load in flight instead of two)
template <typename T>
__device__ __forceinline__ T& at_byte(const void* p, uint32_t off) { return *(T*)((char*)p + off); }
template <typename T>
__device__ __forceinline__ float ld(const void* p, size_t i) { return (float)((const T*)p)[i]; }
__device__ __forceinline__ float silu(float x) { return x / (1.f + __expf(-x)); }
__device__ __forceinline__ float softplus(float x) { return fmaxf(x, 0.f) + log1pf(expf(-fabsf(x))); }

// value and remainder
__device__ __forceinline__ void split(float x, bf16& hi, bf16& lo) {
  hi = (bf16)x;
  lo = (bf16)(x - (float)hi);
}

// ---- convolution of long portions: 8 channels x 16 tokens a thread ---------------------------------
// Which form the step's long portions take (one wave): the chain of the longest one's chunks, or all chunks' work.
__device__ __forceinline__ void pick_form(const Args& A) {
  const int n_items = A.n_items[0], lane = threadIdx.x;
  int most = 0;
  for (int i = lane; i < n_items; i += 64) {
    const int4 it = A.items[i];
    if (it.y == 0) most = max(most, (A.q_len[it.x] + LC - 1) / LC);
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) most = max(most, __shfl_xor(most, o, 64));
  if (lane == 0) A.form[0] = A.chain * most > A.fixed + n_items;
}

// workgroup (x, y) of conv_x, conv_y
template <typename T, int TAPS>
__device__ __forceinline__ void convolve(const Args& A, int x, int y) {
  if (A.form && x == A.conv_x - 1) {  // (a column of workgroups past the channels)
    if (y == 0 && threadIdx.x < 64) pick_form(A);
    return;
  }
  const int c8 = (x * 64 + (threadIdx.x & 63)) * 8, sub = threadIdx.x >> 6, n_items = A.n_items[0];
  if (c8 >= A.Cc || y >= n_items) return;
  const int inner = A.H * A.V;
  const float* W = (const float*)A.conv_w;
  float w[TAPS][8], b[8];
#pragma unroll
  for (int k = 0; k < TAPS; ++k)
#pragma unroll
    for (int j = 0; j < 8; ++j) w[k][j] = W[(size_t)k * A.Cc + c8 + j];
#pragma unroll
  for (int j = 0; j < 8; ++j) b[j] = A.conv_b[c8 + j];
  for (int item = y; item < n_items; item += A.conv_y) {
    const int4 it = A.items[item];
    const int s = it.x, t0 = it.y + sub * 16, t1 = min(it.y + it.z, t0 + 16);
    if (t0 >= t1) continue;
    const int q0 = A.q_start[s], p0 = A.ctx_len[s] - A.q_len[s];
    const T* ring = (const T*)A.ring + (size_t)A.state_slot[s] * A.RING * A.Cc + c8;
    auto load = [&](int t, float (&v)[8]) {  // input of the portion's token t (negative: before it)
      T a[8];
      if (t >= 0) {
        __builtin_memcpy(a, __builtin_assume_aligned((const T*)A.proj + (size_t)(q0 + t) * A.ldp + inner + c8, sizeof(T) * 8), sizeof(T) * 8);
      } else if (p0 + t >= 0) {
        __builtin_memcpy(a, __builtin_assume_aligned(ring + (size_t)((p0 + t) % A.RING) * A.Cc, sizeof(T) * 8), sizeof(T) * 8);
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) a[j] = (T)0.f;
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = (float)a[j];
    };
    float x[TAPS][8];
#pragma unroll
    for (int k = 0; k < TAPS - 1; ++k) load(t0 - (TAPS - 1) + k, x[k + 1]);
    T* out = (T*)A.u + (size_t)q0 * A.Cc + c8;
#pragma unroll 4
    for (int t = t0; t < t1; ++t) {
#pragma unroll
      for (int k = 0; k + 1 < TAPS; ++k)
#pragma unroll
        for (int j = 0; j < 8; ++j) x[k][j] = x[k + 1][j];
      load(t, x[TAPS - 1]);
      T o[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        float v = b[j];
#pragma unroll
        for (int k = 0; k < TAPS; ++k) v = fmaf(w[k][j], x[k][j], v);
        o[j] = (T)silu(v);
      }
      __builtin_memcpy(__builtin_assume_aligned(out + (size_t)t * A.Cc, sizeof(T) * 8), o, sizeof(T) * 8);
    }
  }
}

template <typename T, int TAPS>
__global__ __launch_bounds__(256) void conv_kernel(const Args A) { convolve<T, TAPS>(A, blockIdx.x, blockIdx.y); }

// Channels [c0, c1) of the last `rows` positions of a long portion go to the ring: nobody reads it any
// more in this step (the convolution was in an earlier launch).
template <typename T>
__device__ __forceinline__ void store_ring(const Args& A, int s, int c0, int c1) {
  const int q0 = A.q_start[s], n = A.q_len[s], p0 = A.ctx_len[s] - n, inner = A.H * A.V, rows = min(A.taps - 1, n);
  T* ring = (T*)A.ring + (size_t)A.state_slot[s] * A.RING * A.Cc;
  for (int e = threadIdx.x; e < rows * (c1 - c0); e += blockDim.x) {
    const int i = e / (c1 - c0), c = c0 + e - i * (c1 - c0), t = n - rows + i;
    ring[(size_t)((p0 + t) % A.RING) * A.Cc + c] = ((const T*)A.proj)[(size_t)(q0 + t) * A.ldp + inner + c];
  }
}

// ---- token by token: a workgroup per (sequence, head, part of V) -------------------------------------
constexpr int REGS = 8;  // state vectors of a thread that stay in registers over the portion

// TN: N / 4 as a constant (8 .. 64) where the state fits the registers of the workgroup; 0: any sizes. CONV: the first conv_rows
// rows of workgroups are the long portions' convolution, which no short portion waits for: a launch of its own took 4.6 us of every layer of a
// decoding step, which has none. 4 such layers, 64 decoding rows 1,089 -> 1,079 us a step; 3,658 tokens of prompts, convolution and
// steps 30 -> 27 us a layer, though under this bound the convolution spills 9 registers. (4 taps; with 8 it wants twice the bound's.)
template <typename T, int TAPS, int TN, bool CONV>
__global__ __launch_bounds__(256, 5) void step_kernel(const Args A) {
  extern __shared__ __attribute__((aligned(16))) float sm[];
  if constexpr (CONV)
    if ((int)blockIdx.y < A.conv_rows) {
      const int w = blockIdx.y * gridDim.x + blockIdx.x, y = w / A.conv_x;
      if (y < A.conv_y) convolve<T, TAPS>(A, w - y * A.conv_x, y);
      return;
    }
  const int vlog = __builtin_ctz(A.vsplit), h = blockIdx.x >> vlog, vpart = blockIdx.x & (A.vsplit - 1), s = blockIdx.y - (CONV ? A.conv_rows : 0);
  const int n = A.q_len[s];
  if (n <= 0) return;
  const int slot = A.state_slot[s], q0 = A.q_start[s], p0 = A.ctx_len[s] - n;
  if (slot < 0) return;
  const bool conv = n <= A.scan_min;  // short: the convolution is done here
  if (!conv && !A.long_too) return;
  const int V = A.V, N = TN ? 4 * TN : A.N, g = (uint32_t)h / (uint32_t)A.per_group, inner = A.H * V;
  float *sB = sm, *sC = sm + N, *sx = sm + 2 * N, *sdt = sm + 2 * N + V;  // one token
  float* S = A.state + ((size_t)slot * A.H + h) * V * N;
  T* ring = (T*)A.ring + (size_t)slot * A.RING * A.Cc;
  const float* W = (const float*)A.conv_w;
  // lanes along N, 4 values each (a power of two of them, whole groups inside a wave), the rest along V
  int tn = TN ? TN : 1;
  if constexpr (TN == 0)
    while (tn < 64 && (N >> 2) % (2 * tn) == 0) tn *= 2;
  const int ln = threadIdx.x % tn, lv = threadIdx.x / tn, nv = 256 / tn;
  const int v0 = vpart * (V >> vlog), v1 = v0 + (V >> vlog);
  const float a = A.a[h], dd = A.d[h], bias = A.dt_bias[h];
  // The state in registers over the portion: a lane's vectors are of rows v0 + lv + k nv. Read and written once a step, past
  // the caches' usual place, which is left to the weights and keys. Bound by these bytes: 64 rows, 64 heads of 64 x 128 take
  // 48 us, 5.5 TB/s, where nothing but the update of the same bytes takes 43 (4 workgroups a CU or 5: the
  // same, but those of rows without a sequence, which are gone at once, start faster: 16,384 of them 6.7 us, 5.1 with 5. Five are
  // what the launch bound asks for, 96 registers; the kernel has 82 to 93. Without the two asm statements below it would have
  // 90 to 99, and under the bound spill up to two of them).
  f32x4 st[TN ? REGS : 1];
  // The first token's inputs of a short portion are asked for ahead of the state: its wait then leaves the state's loads in
  // flight, and a thread's second channel waits with the first (64 -> 51 us). That token is apart from the others' loop,
  // whose addresses would take its registers.
  constexpr int EC = TN ? (8 * TN + REGS * 256 / TN + 255) / 256 : 1;  // channels of a thread
  const int n_ch = 2 * N + v1 - v0;
  auto channel = [&](int e) {
    return e < N ? inner + g * N + e : e < 2 * N ? inner + A.G * N + g * N + e - N : h * V + v0 + e - 2 * N;
  };
  float x0[EC][TAPS], w0[EC][TAPS], b0[EC], dt0 = 0.f;
  const bool ahead = TN > 0 && conv;
  if (ahead) {
    const T* row = (const T*)A.proj + (size_t)q0 * A.ldp + inner;
    const int at = (uint32_t)p0 % (uint32_t)A.RING;
#pragma unroll
    for (int j = 0; j < EC; ++j) {
      const int c = channel(min((int)threadIdx.x + j * 256, n_ch - 1));
#pragma unroll
      for (int k = 0; k < TAPS; ++k) {
        const int i = k - (TAPS - 1);  // positions before the first hold no input: row 0 is read for them and not used
        const int r = p0 + i < 0 ? 0 : at + i + (at + i < 0 ? A.RING : 0);
        x0[j][k] = (float)at_byte<T>(k == TAPS - 1 ? row : ring + (size_t)r * A.Cc, c * sizeof(T));
        w0[j][k] = at_byte<float>(W + (size_t)k * A.Cc, c * 4);
      }
      b0[j] = at_byte<float>(A.conv_b, c * 4);
    }
    dt0 = (float)row[A.Cc + h];
  }
  if constexpr (TN > 0) {
    // (rows beyond the part's last: its last again)
#pragma unroll
    for (int k = 0; k < REGS; ++k) st[k] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (p0 > 0) {
#pragma unroll
      for (int k = 0; k < REGS; ++k)
        if (k * nv < v1 - v0)
          st[k] = __builtin_nontemporal_load(&at_byte<f32x4>(S, 4u * (min(v0 + lv + k * nv, v1 - 1) * N + 4 * ln)));
    }
  }
  auto token = [&](int t, auto first) {
    const T* row = (const T*)A.proj + (size_t)(q0 + t) * A.ldp;
    __syncthreads();
    auto put = [&](int e, float v) {
      if (e < 2 * N) sm[e] = v;
      else sx[v0 + e - 2 * N] = v;
    };
    // the owner of a channel keeps its input (rows that no token of this portion reads)
    auto keep = [&](int e, int c) {
      if (e >= 2 * N || (h == g * A.per_group && vpart == 0)) ring[(size_t)((uint32_t)(p0 + t) % (uint32_t)A.RING) * A.Cc + c] = row[inner + c];
    };
    if constexpr (first) {
#pragma unroll
      for (int j = 0; j < EC; ++j) {
        const int e = threadIdx.x + j * 256;
        float v = b0[j];
#pragma unroll
        for (int k = 0; k < TAPS; ++k) v = fmaf(w0[j][k], p0 + k < TAPS - 1 ? 0.f : x0[j][k], v);
        if (e < n_ch) {
          put(e, (float)(T)silu(v));
          keep(e, channel(e));
        }
      }
    } else {
      int first_e = threadIdx.x;
      asm volatile("" : "+v"(first_e));  // (addresses are made anew for every token: kept, they are a workgroup a CU fewer)
      for (int e = first_e; e < n_ch; e += 256) {
        const int c = channel(e);
        float v;
        if (conv) {
          v = A.conv_b[c];
          float x[TAPS];
#pragma unroll
          for (int k = 0; k < TAPS; ++k) {
            const int i = t - (TAPS - 1) + k;
            x[k] = 0.f;
            if (i >= 0) x[k] = (float)((const T*)A.proj)[(size_t)(q0 + i) * A.ldp + inner + c];
            else if (p0 + i >= 0) x[k] = (float)ring[(size_t)((p0 + i) % A.RING) * A.Cc + c];
          }
#pragma unroll
          for (int k = 0; k < TAPS; ++k) v = fmaf(W[(size_t)k * A.Cc + c], x[k], v);
          v = (float)(T)silu(v);
          keep(e, c);
        } else {
          v = (float)((const T*)A.u)[(size_t)(q0 + t) * A.Cc + c];
        }
        put(e, v);
      }
    }
    if (threadIdx.x == 255) {  // (a thread of the last wave, which has the fewest channels)
      const float dt = softplus((first ? dt0 : (float)row[inner + A.Cc + h]) + bias);
      sdt[0] = dt;
      sdt[1] = expf(-a * dt);
    }
    __syncthreads();
    const float dt = sdt[0], decay = sdt[1];
    // one vector's step; returns its part of S^T C
    auto step = [&](f32x4& w, int i, float u) {
      const f32x4 b = *reinterpret_cast<const f32x4*>(sB + i), c = *reinterpret_cast<const f32x4*>(sC + i);
      float acc = 0.f;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        w[j] = w[j] * decay + u * b[j];
        acc = fmaf(w[j], c[j], acc);
      }
      return acc;
    };
    if constexpr (TN > 0) {
      // Rows beyond the part's last are steps of no use, so that nothing branches. The sums over a row's lanes halve the rows
      // that a lane holds in their first three rounds: the same sums in the same order, with 9 shuffles for 40 where 32 lanes
      // share a row (51 -> 48 us).
      float acc[REGS];
      int top = v0 + lv;
      if constexpr (!first) asm volatile("" : "+v"(top));
#pragma unroll
      for (int k = 0; k < REGS; ++k) acc[k] = step(st[k], 4 * ln, dt * sx[min(top + k * nv, v1 - 1)]);
      int k = 0;
#pragma unroll
      for (int left = REGS / 2, o = TN / 2; left > 0; left /= 2, o /= 2) {
        const bool upper = ln & o;
#pragma unroll
        for (int i = 0; i < left; ++i) {
          const float other = __shfl_xor(upper ? acc[i] : acc[i + left], o, 64);
          acc[i] = (upper ? acc[i + left] : acc[i]) + other;
        }
        k += upper ? left : 0;
      }
#pragma unroll
      for (int o = TN / 16; o > 0; o /= 2) acc[0] += __shfl_xor(acc[0], o, 64);
      const int v = top + k * nv;
      if (ln % (TN / 8) == 0 && v < v1) ((T*)A.y)[(size_t)(q0 + t) * A.ldy + h * V + v] = (T)(acc[0] + dd * sx[v]);
    } else {
      const bool fresh = p0 + t == 0;
      for (int v = v0 + lv; v < v1; v += nv) {
        const float x = sx[v];
        float acc = 0.f;
        for (int i = ln * 4; i < N; i += tn * 4) {
          f32x4* p = reinterpret_cast<f32x4*>(S + (size_t)v * N + i);
          f32x4 w = fresh ? f32x4{0.f, 0.f, 0.f, 0.f} : *p;
          acc += step(w, i, dt * x);
          *p = w;
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1)
          if (tn > o) acc += __shfl_xor(acc, o, 64);
        if (ln == 0) ((T*)A.y)[(size_t)(q0 + t) * A.ldy + h * V + v] = (T)(acc + dd * x);
      }
    }
  };
  int t = 0;
  if (ahead) token(t++, std::true_type{});
  for (; t < n; ++t) token(t, std::false_type{});
  if constexpr (TN > 0) {
#pragma unroll
    for (int k = 0; k < REGS; ++k)
      if (v0 + lv + k * nv < v1) __builtin_nontemporal_store(st[k], &at_byte<f32x4>(S, 4u * ((v0 + lv + k * nv) * N + 4 * ln)));
  }
  if (!conv && vpart == 0) {
    const int per = (A.Cc + A.H - 1) / A.H;
    store_ring<T>(A, s, min(A.Cc, h * per), min(A.Cc, (h + 1) * per));
  }
}

// ---- long portions: a workgroup per (portion, head, part of V), chunk after chunk --------------------
// The state stays in the accumulators of the workgroup from a portion's first chunk to its last, so only u is read and y
// written, and the next chunk's rows are on their way while one is computed. Bound by a chunk's chain, 2.8 us with one
// workgroup a CU: about 900 instructions a wave with two barriers, and 280 KB through LDS.
// 64 heads of 64 x 128, three launches with every chunk's state through memory before -> here: 3 prompts of 1,219 tokens
// 184 -> 79 us, 8 of 450 193 -> 81, one of 3,600 204 -> 163, one of 300 37 -> 21.
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) bf16x4 lds_bf16x4;

// (restrict: without alias information the compiler waits at it for loads it does not depend on)
__device__ __forceinline__ bf16x4 tr_read(const char* __restrict__ p) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)p);
}
__device__ __forceinline__ void lds_barrier() {  // global loads stay in flight across it
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// dt and the running log2 decay of a chunk's tokens (wave 0, from their raw step sizes), rows past the end neutral
__device__ __forceinline__ void chunk_steps(float raw, float a, int n, float* dt, float* l) {
  if (threadIdx.x < 64) {
    const int j = threadIdx.x;
    const float d = j < n ? softplus(raw) : 0.f;
    float x = -a * d;
    // running sum over the lanes by data-parallel moves: rows of 16, then their ends to the rows behind
#define PA_ADD(CTRL, ROWS) x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, ROWS, 0xf, false))
    PA_ADD(0x111, 0xf);  // row_shr:1, 2, 4, 8
    PA_ADD(0x112, 0xf);
    PA_ADD(0x114, 0xf);
    PA_ADD(0x118, 0xf);
    PA_ADD(0x142, 0xa);  // row_bcast:15 to rows 1 and 3
    PA_ADD(0x143, 0xc);  // row_bcast:31 to rows 2 and 3
#undef PA_ADD
    dt[j] = d;
    l[j] = x * 1.4426950408889634f;
  }
}

// Rows of a chunk lie in LDS by units of 8 columns, [columns / 8][64 rows][8], a row's worth of padding behind each: a
// row-operand's fragment is a plain 16-byte read, a column operand's a transposed one. NK: N / 32, rounded up to
// a built size (columns past N are zeros); VT: 16-column blocks of V.
constexpr int UNIT = (LC + 1) * 16;
constexpr int VT = 2;  // 16-column blocks of V a workgroup (3 prompts of 1,219 tokens: 79 us; with 1 106, with 4 118)
template <int NK>
struct ScanLds {
  static constexpr int B = 4 * NK * UNIT, X = 2 * VT * UNIT, BUF = B + X + 2 * LC * 4;
  static constexpr int NL = 32 * NK + 8, S = 16 * VT * NL * 2;  // the state, [V][NL], value and remainder
  static constexpr int BYTES = 2 * BUF + 2 * X + 2 * S;
};

template <int NK>
__global__ __launch_bounds__(256, 2) void scan_kernel(const Args A) {
  using L = ScanLds<NK>;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  static_assert(NK * VT % 2 == 0, "every wave keeps as many blocks");
  if (A.form && A.form[0]) return;
  constexpr int PAIRS = NK * VT / 2;  // 16 x 16 blocks of the state a wave keeps
  // heads of a group, which share B and C, on one XCD
  const int parts = gridDim.x / A.H, per = gridDim.x >> 3;
  const int b = gridDim.x % 8 ? (int)blockIdx.x : (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
  const int h = b / parts, v0 = (b % parts) * 16 * VT, V = A.V, N = A.N, g = h / (A.H / A.G), inner = A.H * V;
  const int lane = threadIdx.x & 63, wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lg = lane >> 4, c = lane & 15;
  const int i = 16 * wid + c;  // this lane's token of a chunk
  const int toff = ((c & 3) >> 1) * UNIT + (4 * lg + (c >> 2)) * 16 + (c & 1) * 8;
  char* xw = smem + 2 * L::BUF;  // weighted x, value and remainder
  bf16 *sh = (bf16*)(xw + 2 * L::X), *sl = sh + L::S / 2;
  const int bu = threadIdx.x % (4 * NK), bj = threadIdx.x / (4 * NK);   // this thread's units of B: bj + k (64 / NK)
  const int xu = threadIdx.x % (2 * VT), xj = threadIdx.x / (2 * VT);   // and of x
  const bool bin = 8 * bu < N, xin = v0 + 8 * xu < V;  // (the others' columns are loaded from elsewhere in the row, and dropped
  // when they are used: a select behind the load would wait for it)
  const int bcol = inner + g * N + (bin ? 8 * bu : 0), xcol = h * V + (xin ? v0 + 8 * xu : 0);
  const bf16x8 zero = {};
  const float a = A.a[h], bias = A.dt_bias[h], dd = A.d[h];

  auto portion = [&](int s) {
    const int n = A.q_len[s], q0 = A.q_start[s], chunks = (n + LC - 1) / LC;
    float* S = A.state + ((size_t)A.state_slot[s] * A.H + h) * V * N;
    bf16x8 bv[NK], xv, cf[NK];
    bf16 raw;  // the step size of a token of the chunk after
    auto load_raw = [&](int ch) {
      const int j = min(min(ch, chunks - 1) * LC + lane, n - 1);
      raw = ((const bf16*)A.proj)[(size_t)(q0 + j) * A.ldp + inner + A.Cc + h];
    };
    // (a uniform base and 32-bit offsets: rows of a chunk span less than 2^31 bytes)
    auto at = [](const bf16* base, int e) { return *reinterpret_cast<const bf16x8*>((const char*)base + (uint32_t)(2 * e)); };
    auto load = [&](int ch, bf16x8 (&cn)[NK]) {
      const int m = min(LC, n - ch * LC);
      const bf16* u = (const bf16*)A.u + (size_t)(q0 + ch * LC) * A.Cc;
      load_raw(ch + 1);
#pragma unroll
      for (int k = 0; k < NK; ++k) bv[k] = at(u, min(bj + k * (LC / NK), m - 1) * A.Cc + bcol);
      xv = at(u, min(xj, m - 1) * A.Cc + xcol);
      const int row = min(i, m - 1) * A.Cc + inner + A.G * N + g * N + 8 * lg;
#pragma unroll
      for (int k = 0; k < NK; ++k) cn[k] = at(u, row + (32 * k < N ? 32 * k : 0));  // (past N: meets zeros)
    };
    load_raw(0);
    chunk_steps((float)raw + bias, a, min(LC, n), (float*)(smem + L::B + L::X), (float*)(smem + L::B + L::X) + LC);
    load(0, cf);
    f32x4 st[PAIRS];  // S[v0 + 16 vt + c][16 nt + 4 lg ..]
    auto block = [&](int q, int& nt, int& vt) {
      const int p = wid + 4 * q;
      nt = p % (2 * NK);
      vt = p / (2 * NK);
    };
    auto held = [&](int nt, int vt) { return 16 * nt < N && v0 + 16 * vt < V; };
    auto put_state = [&] {
#pragma unroll
      for (int q = 0; q < PAIRS; ++q) {
        int nt, vt;
        block(q, nt, vt);
        bf16x4 hi, lo;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          bf16 x, y;
          split(st[q][r], x, y);
          hi[r] = x;
          lo[r] = y;
        }
        *reinterpret_cast<bf16x4*>(sh + (16 * vt + c) * L::NL + 16 * nt + 4 * lg) = hi;
        *reinterpret_cast<bf16x4*>(sl + (16 * vt + c) * L::NL + 16 * nt + 4 * lg) = lo;
      }
    };
#pragma unroll
    for (int q = 0; q < PAIRS; ++q) {
      int nt, vt;
      st[q] = f32x4{0.f, 0.f, 0.f, 0.f};
      block(q, nt, vt);
      if (held(nt, vt) && A.ctx_len[s] > n)
        st[q] = *reinterpret_cast<const f32x4*>(S + (size_t)(v0 + 16 * vt + c) * N + 16 * nt + 4 * lg);
    }
    put_state();
    // (A chunk's outputs are stored a chunk later: right behind them, the waits for the loads would be for the stores too,
    // as not every lane makes them.)
    bf16x4 out[VT];
    auto store = [&](int ch) {
      if (ch * LC + i >= n) return;
#pragma unroll
      for (int vt = 0; vt < VT; ++vt)
        if (v0 + 16 * vt < V)
          *reinterpret_cast<bf16x4*>((bf16*)A.y + (size_t)(q0 + ch * LC + i) * A.ldy + h * V + v0 + 16 * vt + 4 * lg) = out[vt];
    };
    for (int ch = 0; ch < chunks; ++ch) {
      char *sb = smem + (ch & 1) * L::BUF, *sx = sb + L::B;
      float *dt = (float*)(sx + L::X), *l = dt + LC;
#pragma unroll
      for (int k = 0; k < NK; ++k) *reinterpret_cast<bf16x8*>(sb + bu * UNIT + (bj + k * (LC / NK)) * 16) = bin ? bv[k] : zero;
      *reinterpret_cast<bf16x8*>(sx + xu * UNIT + xj * 16) = xin ? xv : zero;
      lds_barrier();  // the chunk is whole, and the state
      const float end = l[LC - 1];
      {
        const float w = dt[xj] * __builtin_amdgcn_exp2f(end - l[xj]);  // (0 past the end)
        bf16x8 hi, lo;
#pragma unroll
        for (int r = 0; r < 8; ++r) {
          bf16 x, y;
          split(xin ? w * (float)xv[r] : 0.f, x, y);
          hi[r] = x;
          lo[r] = y;
        }
        *reinterpret_cast<bf16x8*>(xw + xu * UNIT + xj * 16) = hi;
        *reinterpret_cast<bf16x8*>(xw + L::X + xu * UNIT + xj * 16) = lo;
      }
      bf16x8 cn[NK];
      if (ch + 1 < chunks) {
        float* next = (float*)(smem + ((ch + 1) & 1) * L::BUF + L::B + L::X);
        chunk_steps((float)raw + bias, a, min(LC, n - (ch + 1) * LC), next, next + LC);
        load(ch + 1, cn);
      }
      if (ch) store(ch - 1);
      // y: from the state before the chunk, then M[i][j] = exp(l_i - l_j) dt_j (C_i . B_j), j <= i, times x_j
      const float li = l[i], ei = __builtin_amdgcn_exp2f(li);
      f32x4 acc[VT];
#pragma unroll
      for (int vt = 0; vt < VT; ++vt) {
        acc[vt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int k = 0; k < NK; ++k) {
          const int at = (16 * vt + c) * L::NL + 32 * k + 8 * lg;
          acc[vt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*reinterpret_cast<const bf16x8*>(sh + at), cf[k], acc[vt], 0, 0, 0);
          acc[vt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*reinterpret_cast<const bf16x8*>(sl + at), cf[k], acc[vt], 0, 0, 0);
        }
        acc[vt] *= ei;
      }
#pragma unroll
      for (int jt = 0; jt < 4; ++jt) {  // (all four without a branch: tiles above the diagonal are zeros)
        f32x4 cb = {0.f, 0.f, 0.f, 0.f};  // C_i . B_j of j = 16 jt + 4 lg ..
#pragma unroll
        for (int k = 0; k < NK; ++k)
          cb = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*reinterpret_cast<const bf16x8*>(sb + (4 * k + lg) * UNIT + (16 * jt + c) * 16), cf[k], cb, 0, 0, 0);
        const f32x4 lj = *reinterpret_cast<const f32x4*>(l + 16 * jt + 4 * lg), dj = *reinterpret_cast<const f32x4*>(dt + 16 * jt + 4 * lg);
        bf16x4 hi, lo;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          bf16 x, y;
          split(16 * jt + 4 * lg + r <= i ? cb[r] * (__builtin_amdgcn_exp2f(li - lj[r]) * dj[r]) : 0.f, x, y);
          hi[r] = x;
          lo[r] = y;
        }
#pragma unroll
        for (int vt = 0; vt < VT; ++vt) {
          const s16x4 x = __builtin_bit_cast(s16x4, tr_read(sx + 2 * vt * UNIT + jt * 256 + toff));
          acc[vt] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(x, __builtin_bit_cast(s16x4, hi), acc[vt], 0, 0, 0);
          acc[vt] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(x, __builtin_bit_cast(s16x4, lo), acc[vt], 0, 0, 0);
        }
      }
#pragma unroll
      for (int vt = 0; vt < VT; ++vt) {
        const bf16x4 x = *reinterpret_cast<const bf16x4*>(sx + (2 * vt + (lg >> 1)) * UNIT + i * 16 + (lg & 1) * 8);
#pragma unroll
        for (int r = 0; r < 4; ++r) out[vt][r] = (bf16)(acc[vt][r] + dd * (float)x[r]);
      }
      lds_barrier();  // the weighted x is whole, and nobody reads the state any more
      // S <- exp(L) S + sum_j exp(L - l_j) dt_j B_j x_j^T
      const float decay = __builtin_amdgcn_exp2f(end);
#pragma unroll
      for (int q = 0; q < PAIRS; ++q) {
        int nt, vt;
        block(q, nt, vt);
        st[q] *= decay;
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          auto pair = [&](const char* p) {  // rows 32 k ..: 16 and 16
            const bf16x4 x = tr_read(p + 512 * k + toff), y = tr_read(p + 512 * k + 256 + toff);
            return bf16x8{x[0], x[1], x[2], x[3], y[0], y[1], y[2], y[3]};
          };
          const bf16x8 bt = pair(sb + 2 * nt * UNIT);
          st[q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bt, pair(xw + 2 * vt * UNIT), st[q], 0, 0, 0);
          st[q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bt, pair(xw + L::X + 2 * vt * UNIT), st[q], 0, 0, 0);
        }
      }
      put_state();
      if (ch + 1 < chunks) {
#pragma unroll
        for (int k = 0; k < NK; ++k) cf[k] = cn[k];
      }
    }
    store(chunks - 1);
#pragma unroll
    for (int q = 0; q < PAIRS; ++q) {
      int nt, vt;
      block(q, nt, vt);
      if (held(nt, vt))
        *reinterpret_cast<f32x4*>(S + (size_t)(v0 + 16 * vt + c) * N + 16 * nt + 4 * lg) = st[q];
    }
    if (b % parts == 0) {  // this head's share of the channels
      const int share = (A.Cc + A.H - 1) / A.H;
      store_ring<bf16>(A, s, min(A.Cc, h * share), min(A.Cc, (h + 1) * share));
    }
    lds_barrier();  // (the next portion's state goes where this one's was)
  };
  // portions, by their first items, are dealt over the grid's rows
  const int n_items = A.n_items[0];
  int seen = 0;
  for (int base = 0; base < n_items; base += 64) {
    const int4 it = A.items[min(base + lane, n_items - 1)];
    for (unsigned long long first = __ballot(base + lane < n_items && it.y == 0); first; first &= first - 1)
      if (seen++ % gridDim.y == blockIdx.y) portion(__builtin_amdgcn_readlane(it.x, __ffsll(first) - 1));
  }
}

// ---- the same in three launches: every chunk on its own -----------------------------------------------
// For states wider than scan_kernel is built for, and for few heads, whose portions leave it few workgroups that each walk
// all chunks in turn. Two of the three launches run all chunks at once, and every chunk's state goes through memory.
// A token's step size before softplus (wave 0), rows past the end whatever the last one has
__device__ __forceinline__ float load_step(const Args& A, int h, int row0, int n) {
  if (threadIdx.x >= 64) return 0.f;
  return (float)((const bf16*)A.proj)[(size_t)(row0 + min((int)threadIdx.x, n - 1)) * A.ldp + A.H * A.V + A.Cc + h] + A.dt_bias[h];
}
// 8 columns of one of a chunk's rows (unit e of D / 8 columns x 64 rows); rows past the end repeat the
// last one, and meet weights of 0
__device__ __forceinline__ bf16x8 load_cols(const bf16* u, int ld, int e, int D, int n) {
  return *reinterpret_cast<const bf16x8*>(u + (size_t)min(e & (LC - 1), n - 1) * ld + min((e >> 6) * 8, D - 8));
}
constexpr int XB = 2, BB = 4, SB = 8;  // units of x, B and the state that a thread loads ahead

// U_c = sum_j exp(L - l_j) dt_j B_j x_j^T of every chunk
__global__ __launch_bounds__(256) void chunk_state_kernel(const Args A) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  if (A.form && !A.form[0]) return;
  const int h = blockIdx.x, n_items = A.n_items[0];
  const int V = A.V, N = A.N, g = h / (A.H / A.G), inner = A.H * V;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, lg = lane >> 4, c = lane & 15;
  float *dt = (float*)smem, *l = dt + LC;
  bf16* bt = (bf16*)(smem + 2 * LC * 4);  // [N][LD]: B transposed
  bf16 *xh = bt + N * LD, *xl = xh + V * LD;  // [V][LD]: weighted x transposed, value and remainder
  for (int item = blockIdx.y; item < n_items; item += gridDim.y) {
    const int4 it = A.items[item];
    const int n = it.z, row0 = A.q_start[it.x] + it.y;
    const bf16 *ux = (const bf16*)A.u + (size_t)row0 * A.Cc + h * V, *ub = (const bf16*)A.u + (size_t)row0 * A.Cc + inner + g * N;
    const float raw = load_step(A, h, row0, n);
    bf16x8 xv[XB], bv[BB];
#pragma unroll
    for (int i = 0; i < BB; ++i) bv[i] = load_cols(ub, A.Cc, threadIdx.x + 256 * i, N, n);
#pragma unroll
    for (int i = 0; i < XB; ++i) xv[i] = load_cols(ux, A.Cc, threadIdx.x + 256 * i, V, n);
    __syncthreads();
    chunk_steps(raw, A.a[h], n, dt, l);
    auto put_b = [&](int e, const bf16x8& b) {
      const int j = e & (LC - 1), i = (e >> 6) * 8;
      if (i >= N) return;
#pragma unroll
      for (int k = 0; k < 8; ++k) bt[(i + k) * LD + j] = b[k];
    };
#pragma unroll
    for (int i = 0; i < BB; ++i) put_b(threadIdx.x + 256 * i, bv[i]);
    for (int e = threadIdx.x + 256 * BB; e < (N >> 3) * LC; e += 256) put_b(e, load_cols(ub, A.Cc, e, N, n));
    __syncthreads();
    const float end = l[LC - 1];
    auto put_x = [&](int e, const bf16x8& x) {
      const int j = e & (LC - 1), i = (e >> 6) * 8;
      if (i >= V) return;
      const float w = j < n ? dt[j] * __builtin_amdgcn_exp2f(end - l[j]) : 0.f;
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        bf16 hi, lo;
        split(w * (float)x[k], hi, lo);
        xh[(i + k) * LD + j] = hi;
        xl[(i + k) * LD + j] = lo;
      }
    };
#pragma unroll
    for (int i = 0; i < XB; ++i) put_x(threadIdx.x + 256 * i, xv[i]);
    for (int e = threadIdx.x + 256 * XB; e < (V >> 3) * LC; e += 256) put_x(e, load_cols(ux, A.Cc, e, V, n));
    __syncthreads();
    float* out = A.work + ((size_t)item * A.H + h) * V * N;
    const int tn = N >> 4, tv = V >> 4;
    for (int t = wid; t < tn * tv; t += 4) {
      const int n0 = (t % tn) * 16, v0 = (t / tn) * 16;
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const bf16x8 b = *reinterpret_cast<const bf16x8*>(bt + (n0 + c) * LD + 32 * k + 8 * lg);
        const bf16x8 x0 = *reinterpret_cast<const bf16x8*>(xh + (v0 + c) * LD + 32 * k + 8 * lg);
        const bf16x8 x1 = *reinterpret_cast<const bf16x8*>(xl + (v0 + c) * LD + 32 * k + 8 * lg);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b, x0, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b, x1, acc, 0, 0, 0);
      }
      *reinterpret_cast<f32x4*>(out + (size_t)(v0 + c) * N + n0 + 4 * lg) = acc;
    }
    if (threadIdx.x == 0) A.total[(size_t)item * A.H + h] = end;
  }
}

// The state before every chunk, in place of U_c, and the last one to the slot: 4 values a thread, chunk after chunk; the
// next 8 chunks are on their way while 8 are written
__global__ __launch_bounds__(256) void state_pass_kernel(const Args A) {
  const int h = blockIdx.z, VN = A.V * A.N, e = (blockIdx.x * 256 + threadIdx.x) * 4, n_items = A.n_items[0];
  if (e >= VN || (A.form && !A.form[0])) return;
  const size_t step = (size_t)A.H * VN;
  for (int item = blockIdx.y; item < n_items; item += gridDim.y) {
    const int4 it = A.items[item];
    if (it.y != 0) continue;  // a portion's first item takes all of them
    const int s = it.x, n = A.q_len[s], chunks = (n + LC - 1) / LC;
    float* S = A.state + ((size_t)A.state_slot[s] * A.H + h) * VN + e;
    f32x4 st = {0.f, 0.f, 0.f, 0.f};
    if (A.ctx_len[s] > n) st = *reinterpret_cast<const f32x4*>(S);
    float* w = A.work + ((size_t)item * A.H + h) * VN + e;
    const float* tot = A.total + (size_t)item * A.H + h;
    f32x4 u[8], un[8];
    float d[8], dn[8];
    auto load = [&](int c0, f32x4 (&uu)[8], float (&ddd)[8]) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int k = min(c0 + i, chunks - 1);
        uu[i] = *reinterpret_cast<const f32x4*>(w + k * step);
        ddd[i] = tot[(size_t)k * A.H];
      }
    };
    load(0, u, d);
    for (int c0 = 0; c0 < chunks; c0 += 8) {
      if (c0 + 8 < chunks) load(c0 + 8, un, dn);
#pragma unroll
      for (int i = 0; i < 8; ++i)
        if (c0 + i < chunks) {
          *reinterpret_cast<f32x4*>(w + (c0 + i) * step) = st;
          const float f = __builtin_amdgcn_exp2f(d[i]);
#pragma unroll
          for (int j = 0; j < 4; ++j) st[j] = st[j] * f + u[i][j];
        }
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        u[i] = un[i];
        d[i] = dn[i];
      }
    }
    *reinterpret_cast<f32x4*>(S) = st;
  }
}

// Outputs of every chunk. STAGED: the incoming state is split into LDS once; otherwise every wave reads it from memory.
// NK: N / 32 as a constant, for which C stays in registers and B's loads go out together; 0: any N.
template <bool STAGED, int NK>
__global__ __launch_bounds__(256) void chunk_out_kernel(const Args A) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  if (A.form && !A.form[0]) return;
  const int h = blockIdx.x, n_items = A.n_items[0];
  const int V = A.V, N = NK ? 32 * NK : A.N, g = h / (A.H / A.G), inner = A.H * V, NL = N + 8;
  const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, lg = lane >> 4, c = lane & 15;
  float *dt = (float*)smem, *l = dt + LC;
  bf16 *mh = (bf16*)(smem + 2 * LC * 4), *ml = mh + LC * LD;  // [i][LD], value and remainder
  bf16* xt = ml + LC * LD;                                    // [V][LD]
  bf16 *sh = xt + V * LD, *sl = sh + V * NL;                  // [V][NL], value and remainder
  for (int item = blockIdx.y; item < n_items; item += gridDim.y) {
    const int4 it = A.items[item];
    const int n = it.z, row0 = A.q_start[it.x] + it.y;
    const bf16* u = (const bf16*)A.u + (size_t)row0 * A.Cc;
    const float* S = A.work + ((size_t)item * A.H + h) * V * N;
    // (rows past the end repeat the last one; their results are dropped)
    const int i = 16 * wid + c, ri = min(i, n - 1);
    const bf16* cr = u + (size_t)ri * A.Cc + inner + A.G * N + g * N + 8 * lg;
    const bf16* ux = u + h * V;
    const float raw = load_step(A, h, row0, n);
    bf16x8 cf[NK ? NK : 1], xv[XB];
    f32x4 cb[4];  // C_i . B_j
    f32x4 sv[STAGED ? SB : 1];
#pragma unroll
    for (int k = 0; k < XB; ++k) xv[k] = load_cols(ux, A.Cc, threadIdx.x + 256 * k, V, n);
    auto load_state = [&](int e) { return *reinterpret_cast<const f32x4*>(S + min(e, V * N - 4)); };
    if constexpr (STAGED) {
#pragma unroll
      for (int k = 0; k < SB; ++k) sv[k] = load_state(1024 * k + threadIdx.x * 4);
    }
    if constexpr (NK > 0) {
#pragma unroll
      for (int k = 0; k < NK; ++k) cf[k] = *reinterpret_cast<const bf16x8*>(cr + 32 * k);
#pragma unroll
      for (int jt = 0; jt < 4; ++jt) {
        cb[jt] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (jt <= wid) {
          const bf16* br = u + (size_t)min(16 * jt + c, n - 1) * A.Cc + inner + g * N + 8 * lg;
          bf16x8 bf[NK ? NK : 1];
#pragma unroll
          for (int k = 0; k < NK; ++k) bf[k] = *reinterpret_cast<const bf16x8*>(br + 32 * k);
#pragma unroll
          for (int k = 0; k < NK; ++k) cb[jt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf[k], cf[k], cb[jt], 0, 0, 0);
        }
      }
    }
    __syncthreads();
    chunk_steps(raw, A.a[h], n, dt, l);
    auto put_x = [&](int e, const bf16x8& x) {
      const int j = e & (LC - 1), i = (e >> 6) * 8;
      if (i >= V) return;
#pragma unroll
      for (int k = 0; k < 8; ++k) xt[(i + k) * LD + j] = x[k];
    };
#pragma unroll
    for (int k = 0; k < XB; ++k) put_x(threadIdx.x + 256 * k, xv[k]);
    for (int e = threadIdx.x + 256 * XB; e < (V >> 3) * LC; e += 256) put_x(e, load_cols(ux, A.Cc, e, V, n));
    if constexpr (STAGED) {
      auto put_state = [&](int e, const f32x4& v) {
        if (e >= V * N) return;
        const int r = e / N, k0 = e - r * N;
        bf16x4 hi, lo;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          bf16 a, b;
          split(v[k], a, b);
          hi[k] = a;
          lo[k] = b;
        }
        *reinterpret_cast<bf16x4*>(sh + r * NL + k0) = hi;
        *reinterpret_cast<bf16x4*>(sl + r * NL + k0) = lo;
      };
#pragma unroll
      for (int k = 0; k < SB; ++k) put_state(1024 * k + threadIdx.x * 4, sv[k]);
      for (int e = 1024 * SB + threadIdx.x * 4; e < V * N; e += 1024) put_state(e, load_state(e));
    }
    __syncthreads();
    // M[i][j] = exp(l_i - l_j) dt_j (C_i . B_j), a lane's row i, its columns j = 16 jt + 4 lg ..
    const float li = l[i];
#pragma unroll
    for (int jt = 0; jt < 4; ++jt) {
      bf16x4 hi = {(bf16)0.f, (bf16)0.f, (bf16)0.f, (bf16)0.f}, lo = hi;
      if (jt <= wid) {
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
        if constexpr (NK > 0) {
          acc = cb[jt];
        } else {
          const bf16* br = u + (size_t)min(16 * jt + c, n - 1) * A.Cc + inner + g * N + 8 * lg;
          for (int k = 0; k < N; k += 32)
            acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*reinterpret_cast<const bf16x8*>(br + k),
                                                          *reinterpret_cast<const bf16x8*>(cr + k), acc, 0, 0, 0);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int j = 16 * jt + 4 * lg + r;
          bf16 a, b;
          split(j <= i ? acc[r] * (__builtin_amdgcn_exp2f(li - l[j]) * dt[j]) : 0.f, a, b);
          hi[r] = a;
          lo[r] = b;
        }
      }
      *reinterpret_cast<bf16x4*>(mh + i * LD + 16 * jt + 4 * lg) = hi;
      *reinterpret_cast<bf16x4*>(ml + i * LD + 16 * jt + 4 * lg) = lo;
    }
    __syncthreads();
    bf16x8 m0[2], m1[2];
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      m0[k] = *reinterpret_cast<const bf16x8*>(mh + i * LD + 32 * k + 8 * lg);
      m1[k] = *reinterpret_cast<const bf16x8*>(ml + i * LD + 32 * k + 8 * lg);
    }
    const float ei = __builtin_amdgcn_exp2f(li), dd = A.d[h];
    for (int v0 = 0; v0 < V; v0 += 16) {
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
      auto from_state = [&](int k) {
        bf16x8 s0, s1;
        if (STAGED) {
          s0 = *reinterpret_cast<const bf16x8*>(sh + (v0 + c) * NL + k + 8 * lg);
          s1 = *reinterpret_cast<const bf16x8*>(sl + (v0 + c) * NL + k + 8 * lg);
        } else {
          const float* p = S + (size_t)(v0 + c) * N + k + 8 * lg;
#pragma unroll
          for (int q = 0; q < 8; ++q) {
            bf16 a, b;
            split(p[q], a, b);
            s0[q] = a;
            s1[q] = b;
          }
        }
        const bf16x8 cv = NK ? cf[NK ? k / 32 : 0] : *reinterpret_cast<const bf16x8*>(cr + k);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(s0, cv, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(s1, cv, acc, 0, 0, 0);
      };
      if constexpr (NK > 0) {
#pragma unroll
        for (int k = 0; k < NK; ++k) from_state(32 * k);
      } else {
        for (int k = 0; k < N; k += 32) from_state(k);
      }
      acc *= ei;
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const bf16x8 x = *reinterpret_cast<const bf16x8*>(xt + (v0 + c) * LD + 32 * k + 8 * lg);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, m0[k], acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, m1[k], acc, 0, 0, 0);
      }
      if (i < n) {
        bf16x4 o;
#pragma unroll
        for (int r = 0; r < 4; ++r) o[r] = (bf16)(acc[r] + dd * (float)xt[(v0 + 4 * lg + r) * LD + i]);
        *reinterpret_cast<bf16x4*>((bf16*)A.y + (size_t)(row0 + i) * A.ldy + h * V + v0 + 4 * lg) = o;
      }
    }
    if (it.y == 0) {  // the portion's first chunk: this head's share of the channels
      const int per = (A.Cc + A.H - 1) / A.H;
      store_ring<bf16>(A, it.x, min(A.Cc, h * per), min(A.Cc, (h + 1) * per));
    }
  }
}

}  // namespace ss
}  // namespace pa

// max_items: room of the scan items; 0 when no portion of this launch can be longer than scan_min. work [max_items, H, V, N]
// and total [max_items * H + 1]: null where chunks need not go through memory; they must be there for bf16 and N above 256.
// With N up to 256 the step's portions then choose: three launches if chain * (the longest one's chunks) > fixed + all chunks.
extern "C" int pa_state_scan(int fp32, const void* proj, int ldp, void* u, void* y, int ldy, float* state, void* ring,
                             float* work, float* total, float chain, float fixed, const float* conv_w, const float* conv_b,
                             const float* dt_bias, const float* a, const float* d, const int* q_start, const int* q_len,
                             const int* ctx_len, const int* state_slot, const int* items, const int* n_items,
                             int max_items, int seqs, int H, int G, int V, int N, int taps, int ring_rows,
                             int scan_min, hipStream_t st) {
  using namespace pa::ss;
  if (seqs <= 0) return 0;
  if (V % 16 || N % 32 || H % G || scan_min > MAX_SHORT || ring_rows < taps - 1 + scan_min || (taps != 4 && taps != 8)) return -1;  // (shorter ones are padded)
  Args A{proj, u, y, state, ring, conv_w, conv_b, dt_bias, a, d, q_start, q_len, ctx_len, state_slot,
         (const int4*)items, n_items, ldp, ldy, H, G, V, N, H * V + 2 * G * N, taps, ring_rows, scan_min, fp32, 1,
         work, total, nullptr, chain, fixed, H / G, 0, 0, 0};
  if (A.Cc % 8 || ldp % 8) return -1;
  // the three launches: (bf16) states that scan_kernel is not built for, or a choice
  const int lds_s = 2 * LC * 4 + (N + 2 * V) * LD * 2;
  const int lds_o = 2 * LC * 4 + (2 * LC + V) * LD * 2, staged = lds_o + 2 * V * (N + 8) * 2;
  constexpr int MAX_LDS = 160 * 1024;
  const bool fits = lds_s <= MAX_LDS && lds_o <= MAX_LDS, wide = N > 256, three = !fp32 && max_items > 0 && work && fits;
  if (!fp32 && wide && !three) {
    if (max_items > 0 && fits) return -1;  // (no workspace)
    A.long_too = 1;
  }
  if (three && !wide) A.form = (int*)(total + (size_t)max_items * H);
  // few sequences: a head's V over more workgroups
  while (A.vsplit < 8 && H * seqs * A.vsplit < 512 && V % (A.vsplit * 2) == 0) A.vsplit *= 2;
  const bool apart = taps != 4 || A.long_too;  // (its readers are in step_kernel, or too many registers)
  if (max_items > 0) {
    A.conv_x = (A.Cc / 8 + 63) / 64 + (A.form ? 1 : 0);
    A.conv_y = std::min(max_items, 4096);
    if (!apart) A.conv_rows = (A.conv_x * A.conv_y + H * A.vsplit - 1) / (H * A.vsplit);
  }
  if (max_items > 0 && apart) {
    const dim3 grid(A.conv_x, A.conv_y);
#define PA_CONV(T)                                                                                        \
  do {                                                                                                    \
    if (taps == 4) hipLaunchKernelGGL((conv_kernel<T, 4>), grid, dim3(256), 0, st, A);                    \
    else hipLaunchKernelGGL((conv_kernel<T, 8>), grid, dim3(256), 0, st, A);                              \
  } while (0)
    if (fp32) PA_CONV(float); else PA_CONV(pa::bf16);
#undef PA_CONV
  }
  const int step_lds = (2 * N + V + 2) * 4;
  if (step_lds > 64 * 1024) return -2;
  const dim3 sgrid(H * A.vsplit, A.conv_rows + seqs);
  const int tn = V / A.vsplit <= REGS * 1024 / N ? N / 4 : 0;
#define PA_STEP_N(T, K)                                                                                   \
  do {                                                                                                    \
    if (taps == 4) hipLaunchKernelGGL((step_kernel<T, 4, K, sizeof(T) == 2>), sgrid, dim3(256), step_lds, st, A); \
    else hipLaunchKernelGGL((step_kernel<T, 8, K, false>), sgrid, dim3(256), step_lds, st, A);            \
  } while (0)
#define PA_STEP(T)                                                                                        \
  do {                                                                                                    \
    if (tn == 8) PA_STEP_N(T, 8);                                                                         \
    else if (tn == 16) PA_STEP_N(T, 16);                                                                  \
    else if (tn == 32) PA_STEP_N(T, 32);                                                                  \
    else if (tn == 64) PA_STEP_N(T, 64);                                                                  \
    else PA_STEP_N(T, 0);                                                                                 \
  } while (0)
  if (fp32) PA_STEP(float); else PA_STEP(pa::bf16);
#undef PA_STEP
#undef PA_STEP_N
  if (A.long_too || max_items <= 0) return (int)hipGetLastError();
  if (three) {
    static bool attr = false;
    if (!attr) {
      (void)hipFuncSetAttribute((const void*)chunk_state_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, MAX_LDS);
      attr = true;
    }
    const dim3 grid(H, std::min(max_items, 4096));
    hipLaunchKernelGGL(chunk_state_kernel, grid, dim3(256), lds_s, st, A);
    hipLaunchKernelGGL(state_pass_kernel, dim3((V * N / 4 + 255) / 256, std::min(max_items, 16), H), dim3(256), 0, st, A);
    const bool in_lds = staged <= 80 * 1024;
    const int lds = in_lds ? staged : lds_o;
#define PA_OUT(S, K)                                                                                                       \
  do {                                                                                                                     \
    static bool set = false;                                                                                               \
    if (!set) {                                                                                                            \
      (void)hipFuncSetAttribute((const void*)chunk_out_kernel<S, K>, hipFuncAttributeMaxDynamicSharedMemorySize, MAX_LDS); \
      set = true;                                                                                                          \
    }                                                                                                                      \
    hipLaunchKernelGGL((chunk_out_kernel<S, K>), grid, dim3(256), lds, st, A);                                             \
  } while (0)
    if (!in_lds) PA_OUT(false, 0);
    else if (N == 32) PA_OUT(true, 1);
    else if (N == 64) PA_OUT(true, 2);
    else if (N == 128) PA_OUT(true, 4);
    else PA_OUT(true, 0);
#undef PA_OUT
    if (wide) return (int)hipGetLastError();
  }
  // portions loop over the grid's rows
#define PA_SCAN(K)                                                                                                        \
  do {                                                                                                                    \
    constexpr int lds = ScanLds<K>::BYTES;                                                                            \
    static bool set = false;                                                                                              \
    if (!set) {                                                                                                           \
      (void)hipFuncSetAttribute((const void*)scan_kernel<K>, hipFuncAttributeMaxDynamicSharedMemorySize, lds);        \
      set = true;                                                                                                         \
    }                                                                                                                     \
    hipLaunchKernelGGL((scan_kernel<K>), dim3(H * ((V + 31) / 32), std::min(max_items, 32)), dim3(256), lds, st, A); \
  } while (0)
  if (N <= 32) PA_SCAN(1);
  else if (N <= 64) PA_SCAN(2);
  else if (N <= 128) PA_SCAN(4);
  else PA_SCAN(8);
#undef PA_SCAN
  return (int)hipGetLastError();
}
