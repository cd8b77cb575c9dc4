// Reductions (sum over one dim, whole-tensor sum / squared-error sum, MSE
// backward) and index kernels (embedding, index_select, gather).
//
// Reference semantics:
//   sum_dim output shape, keepdim                 crates/core/src/eager.rs:827-855
//   mean_all -> one element                       crates/core/src/eager.rs:710-769
//   mse_loss = mean((a-b)^2), grad = (a-b)*2/n*g  backend_cpp/applegpu_backend.cpp:801-867
//   embedding out[i,:] = W[idx[i],:]              crates/core/src/kernel_templates.rs:1119-1143
//   gather / index_select                         crates/core/src/kernel_templates.rs:870-975
// The reference's mean_all chains thread-per-row mean kernels; here a
// two-stage tree reduction with a fixed order (deterministic, no atomics).
#include "device.hpp"

namespace agpu {
namespace k {
using namespace dev;

namespace {

// [outer, red, inner] -> [outer, inner]; inner == 1 uses a wavefront per row.
template <typename T>
__global__ void __launch_bounds__(256) sum_last(const T* __restrict__ x, T* __restrict__ y, int64_t rows,
                                                int64_t red, float scale) {
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;
  const T* xr = x + row * red;
  float s = 0.f;
  for (int64_t c = lane; c < red; c += 64) s += to_f(xr[c]);
  s = wave_sum(s);
  if (lane == 0) y[row] = from_f<T>(s * scale);
}

// Column sums: a 1024-thread block covers 64 columns x 16 row slices (each
// thread's loads are independent, so they are all in flight), then the 16
// partial sums meet in LDS and are added in slice order.  acc != 0 adds the
// scaled sum to y instead of storing it (y += scale * sum: the bias update
// of an SGD step fused with its gradient).
template <typename T>
__global__ void __launch_bounds__(1024) sum_cols(const T* __restrict__ x, T* __restrict__ y, int64_t outer,
                                                 int64_t red, int64_t inner, float scale, int acc) {
  __shared__ float sh[16][64];
  const int lane = threadIdx.x & 63, slice = threadIdx.x >> 6;
  const int64_t col = (int64_t)blockIdx.x * 64 + lane;
  const int64_t o = blockIdx.y;
  float s = 0.f;
  if (col < inner) {
    const T* base = x + o * red * inner + col;
#pragma unroll 8
    for (int64_t r = slice; r < red; r += 16) s += to_f(base[r * inner]);
  }
  sh[slice][lane] = s;
  __syncthreads();
  if (slice == 0 && col < inner) {
    float t = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) t += sh[i][lane];
    float v = t * scale;
    if (acc) v += to_f(y[o * inner + col]);
    y[o * inner + col] = from_f<T>(v);
  }
}

template <typename T>
__global__ void __launch_bounds__(256) sum_int_dim(const T* __restrict__ x, T* __restrict__ y, int64_t outer,
                                                   int64_t red, int64_t inner) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= outer * inner) return;
  int64_t o = i / inner, c = i % inner;
  long long s = 0;
  for (int64_t r = 0; r < red; ++r) s += (long long)x[(o * red + r) * inner + c];
  y[i] = (T)s;
}

constexpr int kPartials = 512;

// Stage 1: each block writes one fp32 partial.
template <typename T>
__global__ void __launch_bounds__(256) reduce_stage1(int kind, const T* __restrict__ a, const T* __restrict__ b,
                                                     int64_t n, float* __restrict__ part) {
  __shared__ float sh[4];
  float s = 0.f;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
    float v = to_f(a[i]);
    if (kind == 1) {
      v -= to_f(b[i]);
      v *= v;
    }
    s += v;
  }
  s = wave_sum(s);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) part[blockIdx.x] = sh[0] + sh[1] + sh[2] + sh[3];
}

template <typename T>
__global__ void __launch_bounds__(256) reduce_stage2(const float* __restrict__ part, int nparts, float scale,
                                                     T* __restrict__ out) {
  __shared__ float sh[4];
  float s = 0.f;
  for (int i = threadIdx.x; i < nparts; i += 256) s += part[i];
  s = wave_sum(s);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) out[0] = from_f<T>((sh[0] + sh[1] + sh[2] + sh[3]) * scale);
}

template <typename T>
__global__ void __launch_bounds__(256) mse_bwd_kernel(const T* __restrict__ a, const T* __restrict__ b,
                                                      const T* __restrict__ g, T* __restrict__ dx, int64_t n,
                                                      float two_over_n) {
  const float gs = to_f(g[0]);
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256)
    dx[i] = from_f<T>((to_f(a[i]) - to_f(b[i])) * two_over_n * gs);
}

// MSE loss and its gradient (upstream gradient 1) in one single-block
// launch, for the small outputs of a training step: loss = sum((a-b)^2) / n
// (the 1024 per-thread partial sums are reduced in a fixed order) and
// grad = (a - b) * 2/n, the expressions of reduce_stage1/2 and
// mse_bwd_kernel.
constexpr int kMseFusedMax = 1 << 16;
template <typename T>
__global__ void __launch_bounds__(1024) mse_fused_kernel(const T* __restrict__ a, const T* __restrict__ b,
                                                         T* __restrict__ loss, T* __restrict__ grad, int64_t n,
                                                         float inv_n, float two_over_n) {
  __shared__ float sh[16];
  float s = 0.f;
  for (int64_t i = threadIdx.x; i < n; i += 1024) {
    const float d = to_f(a[i]) - to_f(b[i]);
    s += d * d;
    grad[i] = from_f<T>(d * two_over_n * 1.f);
  }
  s = wave_sum(s);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    float t = 0.f;
#pragma unroll
    for (int i = 0; i < 16; ++i) t += sh[i];
    loss[0] = from_f<T>(t * inv_n);
  }
}

// Rows with an index outside [0, vocab) come out as zeros.
template <typename T, typename I>
__global__ void __launch_bounds__(256) embedding_kernel(const T* __restrict__ w, int64_t vocab, int64_t dim,
                                                        const I* __restrict__ idx, int64_t n,
                                                        T* __restrict__ out) {
  const int64_t row = blockIdx.y;
  for (int64_t r = row; r < n; r += gridDim.y) {
    const int64_t id = (int64_t)idx[r];
    const bool ok = id >= 0 && id < vocab;
    for (int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x; c < dim; c += (int64_t)gridDim.x * 256)
      out[r * dim + c] = ok ? w[id * dim + c] : T(0);
  }
}

// The same with whole rows of 16-byte vectors, `rv` to a row: one vector a
// thread, whatever the element type (4096 rows of 768 fp32: 8.4 -> 5.7 us).
template <typename I>
__global__ void __launch_bounds__(256) embedding_vec_kernel(const uint4* __restrict__ w, int64_t vocab, unsigned rv,
                                                            const I* __restrict__ idx, unsigned total,
                                                            uint4* __restrict__ out) {
  const unsigned t = blockIdx.x * 256 + threadIdx.x;
  if (t >= total) return;
  const unsigned r = t / rv, c = t - r * rv;
  const int64_t id = (int64_t)idx[r];
  const bool ok = id >= 0 && id < vocab;
  const uint4 v = w[(ok ? id : 0) * rv + c];
  out[t] = ok ? v : make_uint4(0, 0, 0, 0);
}

// ── embedding backward ────────────────────────────────────────────────────
// dw[w, :] = sum of dy[i, :] over the tokens i with idx[i] == w, added in
// token order; rows no token names are zero (filled first).  One 256-thread
// block per token: the first token naming w collects every token naming w,
// in ascending order, into an LDS list (wavefront ballots keep the order)
// and writes the row, so each row has one writer and one summation order.
// The reference scatters with float atomics (kernel_templates.rs:1867-1913),
// whose order varies from run to run.  Tokens whose index is outside
// [0, nw) add nothing.
//
// Bound by the table's write (4 nw dim bytes) and, in a text, by its most
// frequent word, whose rows one block sums in order: it keeps kEbRows rows'
// loads in flight (with one, 262 rows of 768 took 200 us of latency).  4096
// tokens of a text over 50257 x 768 fp32: 208 -> 18 us, beside 20 us for the
// fill (154 MB).
constexpr int kEbList = 2048;  // tokens gathered per round
constexpr int kEbScan = 4;     // tokens per thread and step of a scan over the indices
constexpr int kEbRows = 16;    // rows in flight

template <typename T>
__global__ void __launch_bounds__(256) fill_zero_kernel(T* __restrict__ p, int64_t n, int64_t nv) {
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x, step = (int64_t)gridDim.x * 256;
  for (int64_t i = t; i < nv; i += step) ((uint4*)p)[i] = make_uint4(0, 0, 0, 0);
  for (int64_t i = nv * (16 / (int64_t)sizeof(T)) + t; i < n; i += step) p[i] = T(0);
}

// C columns per thread, read as one vector: C > 1 needs rows of whole vectors
// at addresses that C elements divide.
template <typename T, typename I, int C>
__global__ void __launch_bounds__(256) embedding_bwd_kernel(const T* __restrict__ dy, const I* __restrict__ idx,
                                                            T* __restrict__ dw, int64_t n, int64_t dim,
                                                            int64_t nw) {
  struct alignas(C * sizeof(T)) Vec { T e[C]; };
  __shared__ int list[kEbList];
  __shared__ int wave_cnt[4];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int64_t i = blockIdx.x;
  const int64_t w = (int64_t)idx[i];
  if (w < 0 || w >= nw) return;  // uniform over the block
  int dup = 0;
  for (int64_t j = tid; j < i; j += 256 * kEbScan) {
#pragma unroll
    for (int k = 0; k < kEbScan; ++k) {
      const int64_t jk = j + 256 * k;
      dup |= (int64_t)idx[jk < i ? jk : j] == w;  // past the end: the first one again
    }
  }
  if (__syncthreads_or(dup)) return;  // an earlier token's block writes row w

  const uint64_t below = lane == 0 ? 0ull : (~0ull >> (64 - lane));
  for (int64_t c0 = 0; c0 < dim; c0 += 256 * C) {
    const int64_t c = c0 + (int64_t)tid * C;
    const bool live = c < dim;
    float acc[C];
#pragma unroll
    for (int k = 0; k < C; ++k) acc[k] = 0.f;
    auto add = [&](const Vec& v) {
#pragma unroll
      for (int k = 0; k < C; ++k) acc[k] += to_f(v.e[k]);
    };
    int64_t t0 = i;
    while (t0 < n) {
      // gather the next round of matching tokens (ascending) into the list:
      // a step looks at 256 kEbScan tokens, wave by wave, kEbScan ballots each
      int cnt = 0;
      while (t0 < n && cnt <= kEbList - 256 * kEbScan) {
        bool m[kEbScan];
        uint64_t mask[kEbScan];
        int mine = 0;
#pragma unroll
        for (int k = 0; k < kEbScan; ++k) {
          const int64_t j = t0 + (wv * kEbScan + k) * 64 + lane;
          m[k] = (int64_t)idx[j < n ? j : n - 1] == w && j < n;
        }
#pragma unroll
        for (int k = 0; k < kEbScan; ++k) {
          mask[k] = __ballot(m[k]);
          mine += __popcll(mask[k]);
        }
        if (lane == 0) wave_cnt[wv] = mine;
        __syncthreads();
        int off = cnt;
        for (int x = 0; x < wv; ++x) off += wave_cnt[x];
#pragma unroll
        for (int k = 0; k < kEbScan; ++k) {
          if (m[k]) list[off + __popcll(mask[k] & below)] = (int)(t0 + (wv * kEbScan + k) * 64 + lane);
          off += __popcll(mask[k]);
        }
        cnt += wave_cnt[0] + wave_cnt[1] + wave_cnt[2] + wave_cnt[3];
        __syncthreads();
        t0 += 256 * kEbScan;
      }
      if (live) {
        const T* col = dy + c;
        int e = 0;
        for (; e + kEbRows <= cnt; e += kEbRows) {
          Vec v[kEbRows];
#pragma unroll
          for (int k = 0; k < kEbRows; ++k) v[k] = *(const Vec*)(col + list[e + k] * dim);
#pragma unroll
          for (int k = 0; k < kEbRows; ++k) add(v[k]);
        }
        for (; e + 4 <= cnt; e += 4) {
          Vec v[4];
#pragma unroll
          for (int k = 0; k < 4; ++k) v[k] = *(const Vec*)(col + list[e + k] * dim);
#pragma unroll
          for (int k = 0; k < 4; ++k) add(v[k]);
        }
        for (; e < cnt; ++e) add(*(const Vec*)(col + list[e] * dim));
      }
      __syncthreads();  // the list is refilled next round
    }
    if (live) {
      Vec o;
#pragma unroll
      for (int k = 0; k < C; ++k) o.e[k] = from_f<T>(acc[k]);
      *(Vec*)(dw + w * dim + c) = o;
    }
  }
}

template <typename T, typename I>
__global__ void __launch_bounds__(256) index_select_kernel(const T* __restrict__ x, int64_t outer, int64_t size,
                                                           int64_t inner, const I* __restrict__ idx, int64_t m,
                                                           T* __restrict__ out) {
  const int64_t n = outer * m * inner;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
    int64_t c = i % inner, j = (i / inner) % m, o = i / (inner * m);
    int64_t id = (int64_t)idx[j];
    out[i] = (id >= 0 && id < size) ? x[(o * size + id) * inner + c] : T(0);
  }
}

template <typename T, typename I>
__global__ void __launch_bounds__(256) gather_kernel(const T* __restrict__ x, int64_t outer, int64_t size,
                                                     int64_t inner, const I* __restrict__ idx, int64_t m,
                                                     T* __restrict__ out) {
  const int64_t n = outer * m * inner;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
    int64_t c = i % inner, o = i / (inner * m);
    int64_t id = (int64_t)idx[i];
    out[i] = (id >= 0 && id < size) ? x[(o * size + id) * inner + c] : T(0);
  }
}

unsigned grid_for(int64_t n) {
  int64_t b = (n + 255) / 256;
  if (b > 65536) b = 65536;
  return (unsigned)(b < 1 ? 1 : b);
}

}  // namespace

void sum_dim(DType dt, const void* x, void* y, int64_t outer, int64_t red, int64_t inner, float scale,
             hipStream_t s) {
  if (outer * inner == 0) return;
  if (!dtype_is_float(dt)) {
    AGPU_ALL_SWITCH(dt, hipLaunchKernelGGL((sum_int_dim<T>), dim3(grid_for(outer * inner)), dim3(256), 0, s,
                                           (const T*)x, (T*)y, outer, red, inner));
  } else if (inner == 1) {
    AGPU_FLOAT_SWITCH(dt, hipLaunchKernelGGL((sum_last<T>), dim3((unsigned)((outer + 3) / 4)), dim3(256), 0, s,
                                             (const T*)x, (T*)y, outer, red, scale));
  } else {
    if (outer > 65535) fail("sum_dim: outer extent %lld too large", (long long)outer);
    dim3 grid((unsigned)((inner + 63) / 64), (unsigned)outer);
    AGPU_FLOAT_SWITCH(dt, hipLaunchKernelGGL((sum_cols<T>), grid, dim3(1024), 0, s, (const T*)x, (T*)y, outer,
                                             red, inner, scale, 0));
  }
  check_launch("sum_dim");
}

size_t reduce_all_ws_bytes() { return kPartials * sizeof(float); }

void reduce_all(int kind, DType dt, const void* a, const void* b, int64_t n, float scale, void* out, void* ws,
                hipStream_t s) {
  int64_t blocks = (n + 255) / 256;
  if (blocks > kPartials) blocks = kPartials;
  if (blocks < 1) blocks = 1;
  AGPU_FLOAT_SWITCH(dt, {
    hipLaunchKernelGGL((reduce_stage1<T>), dim3((unsigned)blocks), dim3(256), 0, s, kind, (const T*)a,
                       (const T*)b, n, (float*)ws);
    hipLaunchKernelGGL((reduce_stage2<T>), dim3(1), dim3(256), 0, s, (const float*)ws, (int)blocks, scale,
                       (T*)out);
  });
  check_launch("reduce_all");
}

void mse_backward(DType dt, const void* a, const void* b, const void* g, void* dx, int64_t n, hipStream_t s) {
  if (n == 0) return;
  float two_over_n = 2.f / (float)n;
  AGPU_FLOAT_SWITCH(dt, hipLaunchKernelGGL((mse_bwd_kernel<T>), dim3(grid_for(n)), dim3(256), 0, s, (const T*)a,
                                           (const T*)b, (const T*)g, (T*)dx, n, two_over_n));
  check_launch("mse_backward");
}

void sum_rows_axpy(DType dt, const void* x, void* y, int64_t rows, int64_t cols, float alpha, hipStream_t s) {
  if (cols == 0) return;
  dim3 grid((unsigned)((cols + 63) / 64), 1);
  AGPU_FLOAT_SWITCH(dt, hipLaunchKernelGGL((sum_cols<T>), grid, dim3(1024), 0, s, (const T*)x, (T*)y, (int64_t)1,
                                           rows, cols, alpha, 1));
  check_launch("sum_rows_axpy");
}

bool mse_fused_ok(int64_t n) { return n > 0 && n <= kMseFusedMax; }

void mse_loss_grad(DType dt, const void* a, const void* b, void* loss, void* grad, int64_t n, hipStream_t s) {
  if (!mse_fused_ok(n)) fail("mse_loss_grad: %lld elements (one block handles at most %d)", (long long)n,
                             kMseFusedMax);
  AGPU_FLOAT_SWITCH(dt, hipLaunchKernelGGL((mse_fused_kernel<T>), dim3(1), dim3(1024), 0, s, (const T*)a,
                                           (const T*)b, (T*)loss, (T*)grad, n, 1.f / (float)n, 2.f / (float)n));
  check_launch("mse_loss_grad");
}

void embedding(DType dt, const void* w, int64_t vocab, int64_t dim, DType idx_dt, const void* idx, int64_t n,
               void* out, hipStream_t s) {
  if (n == 0 || dim == 0) return;
  const int64_t row = dim * (int64_t)dtype_size(dt), vecs = n * (row / 16);
  if (row % 16 == 0 && (uintptr_t)w % 16 == 0 && (uintptr_t)out % 16 == 0 && vocab > 0 && vecs < (1LL << 31)) {
    AGPU_INT_SWITCH(idx_dt, hipLaunchKernelGGL((embedding_vec_kernel<I>), dim3((unsigned)((vecs + 255) / 256)),
                                               dim3(256), 0, s, (const uint4*)w, vocab, (unsigned)(row / 16),
                                               (const I*)idx, (unsigned)vecs, (uint4*)out));
    check_launch("embedding");
    return;
  }
  dim3 grid((unsigned)((dim + 255) / 256), (unsigned)(n < 65535 ? n : 65535));
  AGPU_ALL_SWITCH(dt, {
    typedef T TV;
    AGPU_INT_SWITCH(idx_dt, hipLaunchKernelGGL((embedding_kernel<TV, I>), grid, dim3(256), 0, s, (const TV*)w,
                                               vocab, dim, (const I*)idx, n, (TV*)out));
  });
  check_launch("embedding");
}

void embedding_backward(DType dt, const void* dy, DType idx_dt, const void* idx, int64_t n, int64_t dim,
                        int64_t nw, void* dw, hipStream_t s) {
  if (nw == 0 || dim == 0) return;
  if (n > 0x7fffffffLL) fail("embedding_backward: %lld tokens exceed the grid", (long long)n);
  AGPU_FLOAT_SWITCH(dt, {
    typedef T TV;
    const int64_t total = nw * dim;
    const int64_t nv = (uintptr_t)dw % 16 == 0 ? total / (16 / (int64_t)sizeof(TV)) : 0;
    hipLaunchKernelGGL((fill_zero_kernel<TV>), dim3(grid_for(nv ? nv : total)), dim3(256), 0, s, (TV*)dw, total, nv);
    // four columns a thread where every row starts at a whole vector
    const bool vec = dim % 4 == 0 && (uintptr_t)dy % (4 * sizeof(TV)) == 0 && (uintptr_t)dw % (4 * sizeof(TV)) == 0;
    if (n > 0)
      AGPU_INT_SWITCH(idx_dt, {
        if (vec)
          hipLaunchKernelGGL((embedding_bwd_kernel<TV, I, 4>), dim3((unsigned)n), dim3(256), 0, s, (const TV*)dy,
                             (const I*)idx, (TV*)dw, n, dim, nw);
        else
          hipLaunchKernelGGL((embedding_bwd_kernel<TV, I, 1>), dim3((unsigned)n), dim3(256), 0, s, (const TV*)dy,
                             (const I*)idx, (TV*)dw, n, dim, nw);
      });
  });
  check_launch("embedding_backward");
}

void index_select(DType dt, const void* x, int64_t outer, int64_t size, int64_t inner, DType idx_dt,
                  const void* idx, int64_t m, void* out, hipStream_t s) {
  int64_t n = outer * m * inner;
  if (n == 0) return;
  AGPU_ALL_SWITCH(dt, {
    typedef T TV;
    AGPU_INT_SWITCH(idx_dt, hipLaunchKernelGGL((index_select_kernel<TV, I>), dim3(grid_for(n)), dim3(256), 0, s,
                                               (const TV*)x, outer, size, inner, (const I*)idx, m, (TV*)out));
  });
  check_launch("index_select");
}

void gather(DType dt, const void* x, int64_t outer, int64_t size, int64_t inner, DType idx_dt, const void* idx,
            int64_t m, void* out, hipStream_t s) {
  int64_t n = outer * m * inner;
  if (n == 0) return;
  AGPU_ALL_SWITCH(dt, {
    typedef T TV;
    AGPU_INT_SWITCH(idx_dt, hipLaunchKernelGGL((gather_kernel<TV, I>), dim3(grid_for(n)), dim3(256), 0, s,
                                               (const TV*)x, outer, size, inner, (const I*)idx, m, (TV*)out));
  });
  check_launch("gather");
}

}  // namespace k
}  // namespace agpu
