// softmax, log_softmax, softmax_causal and layer_norm of rows that are long
// (over 2048 columns) or not 16-byte aligned (odd lengths): the row is read
// once, kept in registers and written once.  rows.hip holds the same ops for
// short aligned rows and for rows past the registers' reach.
//
// Bound by HBM.  log_softmax of 2047 x 50257 fp32 (rows of 201 KB at odd
// addresses): 330 -> 177 us, 4.6 TB/s of the 4.8 that a large copy reaches;
// the two-pass block it replaces read the row twice with 4-byte loads.
// layer_norm of the same rows: 414 -> 287 us (13 vectors a thread leave some
// spills beside gamma and beta).
#include "device.hpp"

#include <algorithm>
#include <type_traits>

namespace agpu {
namespace k {
using namespace dev;

namespace {

// ── rows held as 16-byte vectors, any alignment ────────────────────────────
// W wavefronts own a row and keep it in registers as 16-byte vectors: one
// HBM read and one write, bound by HBM.  Vector i of thread t starts at
// column V (64 W i + t), V = 16 / sizeof(T); a vector that would reach past
// the row is loaded from the row's last V columns instead (so every load is
// unconditional and in bounds; needs cols >= V), and its first `skip`
// elements, which belong to other threads, hold `fill`.  The loads need only
// the elements' own alignment: global memory takes 16-byte accesses at any
// element boundary, so rows of odd length keep wide loads.
template <typename T, int W, int NV>
struct RegRow {
  static constexpr int V = 16 / (int)sizeof(T);
  struct Vec { T e[V]; };
  Vec v[NV];
  static __device__ __forceinline__ int at(int i, int t) { return (i * 64 * W + t) * V; }
  static __device__ __forceinline__ int from(int i, int t, int cols) { return min(at(i, t), cols - V); }
  __device__ __forceinline__ void load(const T* __restrict__ row, int t, int cols) {
#pragma unroll
    for (int i = 0; i < NV; ++i) __builtin_memcpy(&v[i], row + from(i, t, cols), 16);
  }
  // Makes the values and the thread index opaque: what was computed from
  // them before is computed again, not kept in registers (16-bit elements as
  // floats would take twice the row's registers, columns one more a vector).
  __device__ __forceinline__ void forget(int& t) {
    asm volatile("" : "+v"(t));
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      uint32_t u[4];
      __builtin_memcpy(u, &v[i], 16);
      asm volatile("" : "+v"(u[0]), "+v"(u[1]), "+v"(u[2]), "+v"(u[3]));
      __builtin_memcpy(&v[i], u, 16);
    }
  }
  // Elements of other threads' columns, and columns at or past `valid`.
  __device__ __forceinline__ void mask(int t, int cols, int valid, float fill) {
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int c = at(i, t);
      if (c + V > valid) {
        const int b = min(c, cols - V);
#pragma unroll
        for (int j = 0; j < V; ++j)
          if (b + j < c || b + j >= valid) v[i].e[j] = from_f<T>(fill);
      }
    }
  }
  __device__ __forceinline__ void store(T* __restrict__ row, int t, int cols) const {
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int c = at(i, t);
      if (c + V <= cols) {
        __builtin_memcpy(row + c, &v[i], 16);
      } else {
        const int b = cols - V;
#pragma unroll
        for (int j = 0; j < V; ++j)
          if (b + j >= c) row[b + j] = v[i].e[j];
      }
    }
  }
};

// Reductions over the W wavefronts of a row (W = 1: several rows a block, no
// barrier; else one row a block).
template <int W>
__device__ __forceinline__ float row_sum(float v, float* sh) {
  v = wave_sum(v);
  if constexpr (W > 1) {
    __syncthreads();
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
    __syncthreads();
    v = 0.f;
#pragma unroll
    for (int w = 0; w < W; ++w) v += sh[w];
  }
  return v;
}
template <int W>
__device__ __forceinline__ float row_max(float v, float* sh) {
  v = wave_max(v);
  if constexpr (W > 1) {
    __syncthreads();
    if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
    __syncthreads();
    v = sh[0];
#pragma unroll
    for (int w = 1; w < W; ++w) v = fmaxf(v, sh[w]);
  }
  return v;
}

// LOG: log_softmax.  causal_rows > 0: row r sees its first
// r % causal_rows + 1 columns.
template <typename T, int W, int NV, bool LOG>
__global__ void __launch_bounds__(W == 1 ? 256 : 64 * W) softmax_reg(const T* __restrict__ x, int64_t ldx,
                                                                     T* __restrict__ y, int64_t ldy, int rows,
                                                                     int cols, int causal_rows) {
  __shared__ float sh[W];
  constexpr int V = RegRow<T, W, NV>::V;
  int t = W == 1 ? threadIdx.x & 63 : threadIdx.x;
  const unsigned row = W == 1 ? blockIdx.x * 4 + (threadIdx.x >> 6) : blockIdx.x;
  if (W == 1 && row >= (unsigned)rows) return;
  const int valid = !LOG && causal_rows > 0 ? min((int)(row % (unsigned)causal_rows) + 1, cols) : cols;
  RegRow<T, W, NV> r;
  r.load(x + (int64_t)row * ldx, t, cols);
  r.mask(t, cols, valid, -INFINITY);
  float mx = -INFINITY;
#pragma unroll
  for (int i = 0; i < NV; ++i)
#pragma unroll
    for (int j = 0; j < V; ++j) mx = fmaxf(mx, to_f(r.v[i].e[j]));
  mx = row_max<W>(mx, sh);
  // as in softmax_wave: the hardware exp2 of the difference for 16-bit rows,
  // expf for fp32
  constexpr float kLog2e = 1.4426950408889634f;
  float one = 1.f;
  asm("" : "+s"(one));  // v - mx as an fma, which takes an fp16 v as it is (v_fma_mix)
  auto ex = [&](float v) {
    if constexpr (sizeof(T) == 2) return __builtin_amdgcn_exp2f(fmaf(v, one, -mx) * kLog2e);
    else return expf(v - mx);
  };
  r.forget(t);
  float sum = 0.f;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    __builtin_amdgcn_sched_barrier(0);  // one vector's exponentials at a time: fewer live registers
#pragma unroll
    for (int j = 0; j < V; ++j) {
      const float e = ex(to_f(r.v[i].e[j]));
      sum += e;
      if constexpr (sizeof(T) == 4)
        if (!LOG) r.v[i].e[j] = e;
    }
  }
  r.forget(t);
  sum = row_sum<W>(sum, sh);
  if constexpr (LOG) {
    const float ls = logf(sum);
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < V; ++j) r.v[i].e[j] = from_f<T>(to_f(r.v[i].e[j]) - mx - ls);
    }
  } else {
    // one division per row; the fp32 quotient is corrected by its remainder,
    // 16-bit rows take the division into the exponent
    const float inv = 1.f / sum, ls2 = -__log2f(sum);
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < V; ++j) {
        if constexpr (sizeof(T) == 4) {
          const float e = r.v[i].e[j], q = e * inv;
          r.v[i].e[j] = fmaf(fmaf(-q, sum, e), inv, q);
        } else {
          r.v[i].e[j] = from_f<T>(__builtin_amdgcn_exp2f(fmaf(fmaf(to_f(r.v[i].e[j]), one, -mx), kLog2e, ls2)));
        }
      }
    }
  }
  r.store(y + (int64_t)row * ldy, t, cols);
}

template <typename T, int W, int NV>
__global__ void __launch_bounds__(W == 1 ? 256 : 64 * W) layer_norm_reg(const T* __restrict__ x, int64_t ldx,
                                                                        const T* __restrict__ g,
                                                                        const T* __restrict__ b, T* __restrict__ y,
                                                                        T* __restrict__ mean_out,
                                                                        T* __restrict__ rstd_out, int64_t rows,
                                                                        int cols, float eps) {
  __shared__ float sh[W];
  typedef RegRow<T, W, NV> R;
  constexpr int V = R::V;
  int t = W == 1 ? threadIdx.x & 63 : threadIdx.x;
  const int64_t row = W == 1 ? (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6) : (int64_t)blockIdx.x;
  if (W == 1 && row >= rows) return;
  R r;
  r.load(x + (int64_t)row * ldx, t, cols);
  r.mask(t, cols, cols, 0.f);
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < NV; ++i)
#pragma unroll
    for (int j = 0; j < V; ++j) s += to_f(r.v[i].e[j]);
  const float mean = row_sum<W>(s, sh) / (float)cols;
  r.forget(t);
  float q = 0.f;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    __builtin_amdgcn_sched_barrier(0);
    const int c = R::at(i, t), f = R::from(i, t, cols);
#pragma unroll
    for (int j = 0; j < V; ++j) {
      const float d = f + j >= c ? to_f(r.v[i].e[j]) - mean : 0.f;
      q += d * d;
    }
  }
  const float inv = 1.f / sqrtf(row_sum<W>(q, sh) / (float)cols + eps);
  if (mean_out && t == 0) {
    mean_out[row] = from_f<T>(mean);
    rstd_out[row] = from_f<T>(inv);
  }
  r.forget(t);
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");  // one vector's gamma and beta at a time
    const int f = R::from(i, t, cols);
    typename R::Vec gv, bv;
    __builtin_memcpy(&gv, g + f, 16);
    __builtin_memcpy(&bv, b + f, 16);
#pragma unroll
    for (int j = 0; j < V; ++j)
      r.v[i].e[j] = from_f<T>(to_f(gv.e[j]) * (to_f(r.v[i].e[j]) - mean) * inv + to_f(bv.e[j]));
  }
  r.store(y + row * cols, t, cols);
}

// How many wavefronts own a row (W) and how many vectors a thread holds (NV),
// by the row's bytes: one wavefront up to 4 KB, so that short rows need no
// barrier and fill the chip; four to 32 KB (one with 8 vectors a lane took longer
// from 4 to 8 KB: layer_norm of fp16 16 x 2049 7.4 -> 4.6 us, 2048 x 3000 10.9 ->
// 9.4, softmax 300 x 4096 5.4 -> 4.3; of 8192 rows most gain, fp32 8192 x 1025
// loses, 16.7 -> 18.8); 16
// beyond, which keeps a thread's share within the 128 registers that a
// 1024-thread block leaves it.
constexpr int64_t kRegRowMax32 = 212992;  // fp32: 13 vectors of 16 wavefronts
constexpr int64_t kRegRowMax16 = 131072;  // 16-bit: 8

template <typename T, typename F>
void by_row_bytes(int64_t bytes, F f) {
  auto go = [&](auto w, auto nv) { f(w, nv); };
#define AGPU_ROW(W, NV) go(std::integral_constant<int, W>{}, std::integral_constant<int, NV>{})
  if (bytes <= 1024) AGPU_ROW(1, 1);
  else if (bytes <= 2048) AGPU_ROW(1, 2);
  else if (bytes <= 4096) AGPU_ROW(1, 4);
  else if (bytes <= 8192) AGPU_ROW(4, 2);
  else if (bytes <= 16384) AGPU_ROW(4, 4);
  else if (bytes <= 32768) AGPU_ROW(4, 8);
  else if (bytes <= 65536) AGPU_ROW(16, 4);
  else if (bytes <= 131072) AGPU_ROW(16, 8);
  else if constexpr (sizeof(T) == 4) AGPU_ROW(16, 13);
#undef AGPU_ROW
}

dim3 row_blocks(int w, int64_t rows) { return dim3((unsigned)(w == 1 ? (rows + 3) / 4 : rows)); }

}  // namespace

bool reg_row_ok(DType dt, int64_t rows, int64_t cols) {
  if (!dtype_is_float(dt) || dt == DType::F64 || rows > 0x7fffffffLL) return false;
  const int64_t es = (int64_t)dtype_size(dt), bytes = cols * es;
  return bytes >= 16 && bytes <= (es == 4 ? kRegRowMax32 : kRegRowMax16);
}

void softmax_reg_rows(int op, DType dt, const void* x, int64_t ldx, void* y, int64_t ldy, int64_t rows, int64_t cols,
                      int64_t causal_rows, hipStream_t s) {
  const int causal = op == kSoftmaxCausal ? (int)std::min<int64_t>(causal_rows, rows) : 0;
  AGPU_FLOAT_SWITCH(dt, by_row_bytes<T>(cols * (int64_t)sizeof(T), [&](auto w, auto nv) {
                      const dim3 grid = row_blocks(w.value, rows), block(w.value == 1 ? 256 : 64 * w.value);
                      if (op == kLogSoftmax)
                        hipLaunchKernelGGL((softmax_reg<T, w.value, nv.value, true>), grid, block, 0, s, (const T*)x,
                                           ldx, (T*)y, ldy, (int)rows, (int)cols, 0);
                      else
                        hipLaunchKernelGGL((softmax_reg<T, w.value, nv.value, false>), grid, block, 0, s,
                                           (const T*)x, ldx, (T*)y, ldy, (int)rows, (int)cols, causal);
                    }));
}

void layer_norm_reg_rows(DType dt, const void* x, int64_t ldx, const void* gamma, const void* beta, void* y,
                         void* mean, void* rstd, int64_t rows, int64_t cols, float eps, hipStream_t s) {
  AGPU_FLOAT_SWITCH(dt, by_row_bytes<T>(cols * (int64_t)sizeof(T), [&](auto w, auto nv) {
                      hipLaunchKernelGGL((layer_norm_reg<T, w.value, nv.value>), row_blocks(w.value, rows),
                                         dim3(w.value == 1 ? 256 : 64 * w.value), 0, s, (const T*)x, ldx,
                                         (const T*)gamma, (const T*)beta, (T*)y, (T*)mean, (T*)rstd, rows,
                                         (int)cols, eps);
                    }));
}

}  // namespace k
}  // namespace agpu
