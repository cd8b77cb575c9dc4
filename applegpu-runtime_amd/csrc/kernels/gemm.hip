// Batched GEMM C(m,n) = epilogue(sum_k A(m,k) B(k,n)) for gfx950: planning,
// launch, and the kernels outside the bf16-MFMA family of gemm_kernels.hpp.
//
// Reference semantics: row-major batched matmul with fp32 accumulate
// (crates/core/src/kernel_templates.rs:987-1072, crates/core/src/eager.rs:403-479),
// transposed operands read in place (crates/core/src/eager.rs:485-560), and
// Linear = x W^T + b (backend_cpp/applegpu_backend.cpp:584-620).
//
// fp32, fp16 and bf16 GEMMs run gemm_mf (gemm_kernels.hpp): bf16/fp16 MFMA
// 32x32x16 tiles, with fp32 operands split into bf16 hi + lo (three MFMAs per
// product: hi*hi + hi*lo + lo*hi, fp32 accumulate).  gfx950 has no xf32
// MFMA; the native fp32 alternative, v_mfma_f32_32x32x2_f32, is kept below
// (gemm_f32_mfma) and selected with GemmTune::f32_mode = kF32Native.
// Problems with too few tiles for the CU count split K across blocks into an
// fp32 workspace that splitk_reduce sums in a fixed order (deterministic)
// while applying the epilogue.  Block ids are remapped so that consecutive
// tiles land on the same XCD (blocks are dealt round-robin over the 8 XCDs,
// each with its own L2), then grouped 8 tile-rows at a time for L2 reuse of B.
#include "gemm_kernels.hpp"

#include <cstdio>
#include <cstdlib>
#include <cstring>

namespace agpu {
namespace k {
using namespace dev;

namespace {

// ── fp32 MFMA kernel ──────────────────────────────────────────────────────
// Loads a ROWSxBK (KCONT: k contiguous) or BKxROWS (!KCONT) fp32 tile slice
// owned by this thread into registers.
template <int ROWS, bool KCONT>
struct TileF32 {
  static constexpr int BK = 16;
  static constexpr int FPT = ROWS * BK / 256;  // floats per thread
  float v[FPT];

  __device__ __forceinline__ void load(const float* __restrict__ base, int64_t s_row, int64_t s_k, int64_t r0,
                                       int64_t rmax, int64_t k, int64_t kmax, bool vec) {
    const int t = threadIdx.x;
    if constexpr (KCONT) {
      constexpr int TPR = BK / FPT;
      const int r = t / TPR, kk = (t % TPR) * FPT;
      const int64_t gr = r0 + r, gk = k + kk;
      const float* src = base + gr * s_row + gk;
      if (vec && gr < rmax && gk + FPT <= kmax) {
#pragma unroll
        for (int i = 0; i < FPT; i += 4) *(float4*)&v[i] = *(const float4*)(src + i);
      } else {
#pragma unroll
        for (int i = 0; i < FPT; ++i) v[i] = (gr < rmax && gk + i < kmax) ? src[i] : 0.f;
      }
    } else {
      constexpr int TPK = ROWS / FPT;
      const int kk = t / TPK, r = (t % TPK) * FPT;
      const int64_t gr = r0 + r, gk = k + kk;
      const float* src = base + gk * s_k + gr;
      if (vec && gk < kmax && gr + FPT <= rmax) {
#pragma unroll
        for (int i = 0; i < FPT; i += 4) *(float4*)&v[i] = *(const float4*)(src + i);
      } else {
#pragma unroll
        for (int i = 0; i < FPT; ++i) v[i] = (gk < kmax && gr + i < rmax) ? src[i] : 0.f;
      }
    }
  }

  // LDS tile is [BK][ROWS] (rows contiguous).
  __device__ __forceinline__ void store(float* __restrict__ lds) const {
    const int t = threadIdx.x;
    if constexpr (KCONT) {
      constexpr int TPR = BK / FPT;
      const int r = t / TPR, kk = (t % TPR) * FPT;
#pragma unroll
      for (int i = 0; i < FPT; ++i) lds[(kk + i) * ROWS + r] = v[i];
    } else {
      constexpr int TPK = ROWS / FPT;
      const int kk = t / TPK, r = (t % TPK) * FPT;
#pragma unroll
      for (int i = 0; i < FPT; i += 4) *(float4*)&lds[kk * ROWS + r + i] = *(const float4*)&v[i];
    }
  }
};

template <int BM, int BN, bool AK, bool BKC>
__global__ void __launch_bounds__(256) gemm_f32_mfma(GArgs p) {
  constexpr int BK = 16;
  constexpr int TM = BM / 64, TN = BN / 64;  // 32x32 blocks per wave
  __shared__ __attribute__((aligned(16))) float As[2][BK * BM];
  __shared__ __attribute__((aligned(16))) float Bs[2][BK * BN];

  int tm, tn;
  tile_coords(p, tm, tn);
  const int64_t z = blockIdx.y;
  const int64_t b = z / p.splits;
  const int split = (int)(z % p.splits);
  const int64_t m0 = (int64_t)tm * BM, n0 = (int64_t)tn * BN;
  const int64_t kbeg = (int64_t)split * p.k_per_split;
  int64_t kend = kbeg + p.k_per_split;
  if (kend > p.K) kend = p.K;

  const float* A = (const float*)p.A + b * p.a_sb;
  const float* B = (const float*)p.B + b * p.b_sb;
  // For A, "rows" are m; for B, "rows" are n.
  const int64_t a_srow = p.a_sm, a_sk = p.a_sk;
  const int64_t b_srow = p.b_sn, b_sk = p.b_sk;

  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = (wave >> 1) * (BM / 2), wn = (wave & 1) * (BN / 2);

  f32x16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

  TileF32<BM, AK> ta;
  TileF32<BN, BKC> tb;
  const int64_t nk = (kend - kbeg + BK - 1) / BK;
  if (nk > 0) {
    ta.load(A, a_srow, a_sk, m0, p.M, kbeg, kend, p.vec_a);
    tb.load(B, b_srow, b_sk, n0, p.N, kbeg, kend, p.vec_b);
    ta.store(As[0]);
    tb.store(Bs[0]);
  }
  __syncthreads();

  for (int64_t kt = 0; kt < nk; ++kt) {
    const int buf = (int)(kt & 1);
    const bool more = kt + 1 < nk;
    if (more) {
      const int64_t kn = kbeg + (kt + 1) * BK;
      ta.load(A, a_srow, a_sk, m0, p.M, kn, kend, p.vec_a);
      tb.load(B, b_srow, b_sk, n0, p.N, kn, kend, p.vec_b);
    }
    const float* as = As[buf];
    const float* bs = Bs[buf];
#pragma unroll
    for (int kk = 0; kk < BK; kk += 2) {
      const int krow = kk + (lane >> 5);
      float av[TM], bv[TN];
#pragma unroll
      for (int i = 0; i < TM; ++i) av[i] = as[krow * BM + wm + i * 32 + (lane & 31)];
#pragma unroll
      for (int j = 0; j < TN; ++j) bv[j] = bs[krow * BN + wn + j * 32 + (lane & 31)];
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(av[i], bv[j], acc[i][j], 0, 0, 0);
    }
    if (more) {
      ta.store(As[buf ^ 1]);
      tb.store(Bs[buf ^ 1]);
    }
    __syncthreads();
  }

  // Output layout of a 32x32 block: lane l, register r ->
  //   row = 8*(r/4) + 4*(l/32) + r%4, col = l%32.
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int64_t col = n0 + wn + j * 32 + (lane & 31);
      if (col >= p.N) continue;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int64_t row = m0 + wm + i * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
        if (row >= p.M) continue;
        if (p.splits > 1)
          p.ws[((int64_t)split * p.batch + b) * p.M * p.N + row * p.N + col] = acc[i][j][r];
        else
          epilogue_store<float>(p, b, row, col, acc[i][j][r]);
      }
    }
}

// Split-K reduction in split order, then the epilogue.  Four outputs per
// thread; every split's partial is loaded before the first add, so the
// loads overlap instead of costing one memory latency per split.
template <typename T>
__global__ void __launch_bounds__(256) splitk_reduce(GArgs p) {
  constexpr int kMaxSplits = 8;
  const int64_t total = p.batch * p.M * p.N;
  const bool vec = (total & 3) == 0;
  for (int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4; i < total; i += (int64_t)gridDim.x * 1024) {
    float part[kMaxSplits][4];
    const int ns = p.splits < kMaxSplits ? p.splits : kMaxSplits;
#pragma unroll
    for (int sp = 0; sp < kMaxSplits; ++sp) {
      if (sp >= ns) break;
      const float* src = p.ws + (int64_t)sp * total + i;
      if (vec) {
        const float4 v = *(const float4*)src;
        part[sp][0] = v.x; part[sp][1] = v.y; part[sp][2] = v.z; part[sp][3] = v.w;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) part[sp][e] = i + e < total ? src[e] : 0.f;
      }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (i + e >= total) break;
      float s = 0.f;
#pragma unroll
      for (int sp = 0; sp < kMaxSplits; ++sp) {
        if (sp >= ns) break;
        s += part[sp][e];
      }
      for (int sp = kMaxSplits; sp < p.splits; ++sp) s += p.ws[(int64_t)sp * total + i + e];
      const int64_t ie = i + e;
      const int64_t col = ie % p.N, row = (ie / p.N) % p.M, b = ie / (p.M * p.N);
      epilogue_store<T>(p, b, row, col, s);
    }
  }
}

// Split-K reduction that also layer-normalises each output row (one batch,
// N <= 256*NV, N % 4 == 0): one wavefront per row sums the partials in split order and
// applies the epilogue as splitk_reduce does, stores C, then computes
// Y = layer_norm(C) from the stored values with layer_norm_wave's element
// mapping (element (64 i + lane) * 4 + j), two-pass statistics and
// reduction order, so Y equals what a separate layer_norm of C would give.
// GPT-2 runs it for the projection and fc2 GEMMs, whose outputs (residual
// stream) feed ln_2 / the next layer's ln_1 (models/gpt2.py:84-178).
// 4 consecutive elements as floats (16-byte or 8-byte load; 16-byte aligned
// for fp32, 8-byte for 16-bit types).
template <typename T>
__device__ __forceinline__ void ld4f(const T* src, float (&o)[4]) {
  if constexpr (sizeof(T) == 4) {
    const float4 v = *(const float4*)src;
    o[0] = v.x; o[1] = v.y; o[2] = v.z; o[3] = v.w;
  } else {
    T t[4];
    *(uint2*)t = *(const uint2*)src;
#pragma unroll
    for (int j = 0; j < 4; ++j) o[j] = to_f(t[j]);
  }
}
template <typename T>
__device__ __forceinline__ void st4(T* dst, const float (&v)[4]) {
  if constexpr (sizeof(T) == 4) {
    *(float4*)dst = make_float4(v[0], v[1], v[2], v[3]);
  } else {
    T t[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) t[j] = from_f<T>(v[j]);
    *(uint2*)dst = *(const uint2*)t;
  }
}

template <typename T, int NV, int MS>  // MS: partials loaded up front; more are added afterwards
__global__ void __launch_bounds__(256) splitk_reduce_ln(GArgs p) {
  if (prefetch_block(p.pf)) return;
  const int lane = threadIdx.x & 63;
  // one wavefront per row; a block holds blockDim.x / 64 rows
  const int64_t row = (int64_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  if (row >= p.M) return;  // whole wavefront; no barriers below
  const int64_t N = p.N, total = p.M * p.N;
  const int ns = p.splits;
  // Every load first, from clamped legal addresses (chunks past N read
  // chunk 0 and are discarded), so that they are all in flight together;
  // gamma and beta, needed last, go out last (a wavefront's loads complete
  // in issue order).  Absent epilogue operands are not loaded (the tests
  // are uniform across the wavefront).
  float part[NV][MS][4], bias[NV][4] = {}, res[NV][4] = {}, msk[NV][4] = {}, gam[NV][4], bet[NV][4];
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int64_t c = ((int64_t)i * 64 + lane) * 4;
    const int64_t cc = c < N ? c : 0;
#pragma unroll
    for (int sp = 0; sp < MS; ++sp) {
      const float4 w = *(const float4*)(p.ws + (int64_t)(sp < ns ? sp : 0) * total + row * N + cc);
      part[i][sp][0] = w.x; part[i][sp][1] = w.y; part[i][sp][2] = w.z; part[i][sp][3] = w.w;
    }
    if (p.bias) ld4f<T>((const T*)p.bias + cc, bias[i]);
    if (p.res) ld4f<T>((const T*)p.res + row * p.r_sm + cc, res[i]);
    if (p.mask) ld4f<T>((const T*)p.mask + row * p.k_sm + cc, msk[i]);
  }
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int64_t c = ((int64_t)i * 64 + lane) * 4;
    const int64_t cc = c < N ? c : 0;
    ld4f<T>((const T*)p.pln_g + cc, gam[i]);
    ld4f<T>((const T*)p.pln_b + cc, bet[i]);
  }
  float v[NV][4];
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int64_t c = ((int64_t)i * 64 + lane) * 4;
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int sp = 0; sp < MS; ++sp)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[j] += sp < ns ? part[i][sp][j] : 0.f;
    for (int sp = MS; sp < ns; ++sp)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[j] += c < N ? p.ws[(int64_t)sp * total + row * N + c + j] : 0.f;
    float o[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      // epilogue_store's arithmetic
      float x = p.alpha * acc[j];
      if (p.bias) x += bias[i][j];
      if (p.act == kActRelu) x = fmaxf(x, 0.f);
      else if (p.act == kActGelu) x = gelu_tanh(x);
      else if (p.act == kActGeluExact) x = 0.5f * x * (1.f + erff(x * 0.70710678118654752f));
      if (p.res) x += res[i][j];
      if (p.mask) x = msk[i][j] > 0.f ? x : 0.f;
      o[j] = to_f(from_f<T>(x));  // the value as stored
    }
    if (c < N) st4<T>((T*)p.C + row * p.c_sm + c, o);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      v[i][j] = c < N ? o[j] : 0.f;
      s += v[i][j];
    }
  }
  const float mean = wave_sum(s) / (float)N;
  float q = 0.f;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int64_t c = ((int64_t)i * 64 + lane) * 4;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float d = c < N ? v[i][j] - mean : 0.f;
      q += d * d;
    }
  }
  const float var = wave_sum(q) / (float)N;
  const float inv = 1.f / sqrtf(var + p.pln_eps);
  T* y = (T*)p.pln_y + row * N;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int64_t c = ((int64_t)i * 64 + lane) * 4;
    float o[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) o[j] = gam[i][j] * (v[i][j] - mean) * inv + bet[i][j];
    if (c < N && p.pln_y) st4<T>(y + c, o);
    if constexpr (sizeof(T) == 4)
      if (c < N && p.pln_ypk) x3_store4(p.pln_ypk, N / 16, row, c, o);
  }
}

// splitk_reduce_ln for more than 8 splits: one 4-wavefront block per row.
// Wave w sums splits [w q, (w + 1) q) in order (q = ceil(splits / 4), all
// its loads issued first), the four sums meet in LDS and wave 0 adds them in
// wave order, then finishes as splitk_reduce_ln does (epilogue, store,
// layer_norm of the stored row).  The order is fixed, so repeated launches
// give identical bits.
template <typename T, int NV, int MQ>  // MQ: splits per wave loaded up front
__global__ void __launch_bounds__(256) splitk_reduce_ln_mw(GArgs p) {
  __shared__ float sum_w[3][NV * 256];
  if (prefetch_block(p.pf)) return;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int64_t row = blockIdx.x;
  const int64_t N = p.N, total = p.M * p.N;
  const int ns = p.splits;
  const int q = (ns + 3) / 4;
  const int s0 = w * q, s1 = s0 + q < ns ? s0 + q : ns;
  float part[NV][MQ][4];
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int64_t c = ((int64_t)i * 64 + lane) * 4;
    const int64_t cc = c < N ? c : 0;
#pragma unroll
    for (int j = 0; j < MQ; ++j) {
      const int sp = s0 + j < s1 ? s0 + j : 0;
      const float4 v = *(const float4*)(p.ws + (int64_t)sp * total + row * N + cc);
      part[i][j][0] = v.x; part[i][j][1] = v.y; part[i][j][2] = v.z; part[i][j][3] = v.w;
    }
  }
  float bias[NV][4] = {}, res[NV][4] = {}, msk[NV][4] = {}, gam[NV][4], bet[NV][4];
  if (w == 0) {
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int64_t c = ((int64_t)i * 64 + lane) * 4;
      const int64_t cc = c < N ? c : 0;
      if (p.bias) ld4f<T>((const T*)p.bias + cc, bias[i]);
      if (p.res) ld4f<T>((const T*)p.res + row * p.r_sm + cc, res[i]);
      if (p.mask) ld4f<T>((const T*)p.mask + row * p.k_sm + cc, msk[i]);
      ld4f<T>((const T*)p.pln_g + cc, gam[i]);
      ld4f<T>((const T*)p.pln_b + cc, bet[i]);
    }
  }
  float acc[NV][4];
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int64_t c = ((int64_t)i * 64 + lane) * 4;
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[i][e] = 0.f;
#pragma unroll
    for (int j = 0; j < MQ; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[i][e] += s0 + j < s1 ? part[i][j][e] : 0.f;
    for (int sp = s0 + MQ; sp < s1; ++sp)
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[i][e] += c < N ? p.ws[(int64_t)sp * total + row * N + c + e] : 0.f;
    if (w > 0) {
#pragma unroll
      for (int e = 0; e < 4; ++e) sum_w[w - 1][(i * 64 + lane) * 4 + e] = acc[i][e];
    }
  }
  __syncthreads();
  if (w > 0) return;
  float v[NV][4];
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int64_t c = ((int64_t)i * 64 + lane) * 4;
    float o[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float a = acc[i][e];
#pragma unroll
      for (int x = 0; x < 3; ++x) a += sum_w[x][(i * 64 + lane) * 4 + e];
      float y = p.alpha * a;
      if (p.bias) y += bias[i][e];
      if (p.act == kActRelu) y = fmaxf(y, 0.f);
      else if (p.act == kActGelu) y = gelu_tanh(y);
      else if (p.act == kActGeluExact) y = 0.5f * y * (1.f + erff(y * 0.70710678118654752f));
      if (p.res) y += res[i][e];
      if (p.mask) y = msk[i][e] > 0.f ? y : 0.f;
      o[e] = to_f(from_f<T>(y));  // the value as stored
    }
    if (c < N) st4<T>((T*)p.C + row * p.c_sm + c, o);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      v[i][e] = c < N ? o[e] : 0.f;
      s += v[i][e];
    }
  }
  const float mean = wave_sum(s) / (float)N;
  float qq = 0.f;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int64_t c = ((int64_t)i * 64 + lane) * 4;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float d = c < N ? v[i][e] - mean : 0.f;
      qq += d * d;
    }
  }
  const float var = wave_sum(qq) / (float)N;
  const float inv = 1.f / sqrtf(var + p.pln_eps);
  T* y = (T*)p.pln_y + row * N;
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const int64_t c = ((int64_t)i * 64 + lane) * 4;
    float o[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = gam[i][e] * (v[i][e] - mean) * inv + bet[i][e];
    if (c < N && p.pln_y) st4<T>(y + c, o);
    if constexpr (sizeof(T) == 4)
      if (c < N && p.pln_ypk) x3_store4(p.pln_ypk, N / 16, row, c, o);
  }
}

template <typename T, int NV>
void launch_reduce_ln_nv(const GArgs& p0, dim3 grid, dim3 block, hipStream_t s) {
  GArgs p = p0;
  if (p.splits > 8) {
    // one 4-wave block per row
    p.pf = make_prefetch((int)p.M, 256);
    const dim3 g2((unsigned)(p.M + p.pf.blocks)), b2(256);
    if (p.splits <= 16) hipLaunchKernelGGL((splitk_reduce_ln_mw<T, NV, 4>), g2, b2, 0, s, p);
    else hipLaunchKernelGGL((splitk_reduce_ln_mw<T, NV, 8>), g2, b2, 0, s, p);
    return;
  }
  p.pf = make_prefetch((int)grid.x, (int)block.x);
  grid.x += p.pf.blocks;
  if (p.splits <= 2) hipLaunchKernelGGL((splitk_reduce_ln<T, NV, 2>), grid, block, 0, s, p);
  else if (p.splits <= 4) hipLaunchKernelGGL((splitk_reduce_ln<T, NV, 4>), grid, block, 0, s, p);
  else hipLaunchKernelGGL((splitk_reduce_ln<T, NV, 8>), grid, block, 0, s, p);
}

template <typename T>
void launch_reduce_ln(const GArgs& p, hipStream_t s) {
  // Up to 1024 rows, one row per block: the rows then spread over as many
  // CUs as there are rows (GPT-2's 128 rows: 128 CUs, not 32).
  const int rpb = p.M <= 1024 ? 1 : 4;
  const dim3 grid((unsigned)((p.M + rpb - 1) / rpb)), block(64 * rpb);
  switch ((p.N + 255) / 256) {
    case 1: launch_reduce_ln_nv<T, 1>(p, grid, block, s); break;
    case 2: launch_reduce_ln_nv<T, 2>(p, grid, block, s); break;
    case 3: launch_reduce_ln_nv<T, 3>(p, grid, block, s); break;
    case 4: launch_reduce_ln_nv<T, 4>(p, grid, block, s); break;
    case 5: launch_reduce_ln_nv<T, 5>(p, grid, block, s); break;
    case 6: launch_reduce_ln_nv<T, 6>(p, grid, block, s); break;
    case 7: launch_reduce_ln_nv<T, 7>(p, grid, block, s); break;
    case 8: launch_reduce_ln_nv<T, 8>(p, grid, block, s); break;
    default: fail("gemm: fused layer_norm needs N <= 2048");
  }
}

// splitk_reduce for one batch with N % 4 == 0 and 4-element aligned
// epilogue operands: each thread owns 4 consecutive outputs, issues every
// load first (up to 8 partials from clamped split indices, then bias,
// residual and mask as vectors, all branch-free) and stores one vector.
// Same sums in the same split order and the same epilogue arithmetic as
// splitk_reduce.
template <typename T, int MS>  // MS: partials loaded up front (the split count rounded up to 2, 4, 8, 16 or 32)
__global__ void __launch_bounds__(256) splitk_reduce_vec(GArgs p) {
  const int64_t total = p.M * p.N;
  const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i >= total) return;
  const int ns = p.splits;
  const int64_t row = i / p.N, col = i % p.N;
  float part[MS][4];
#pragma unroll
  for (int sp = 0; sp < MS; ++sp) {
    const float4 w = *(const float4*)(p.ws + (int64_t)(sp < ns ? sp : 0) * total + i);
    part[sp][0] = w.x; part[sp][1] = w.y; part[sp][2] = w.z; part[sp][3] = w.w;
  }
  // absent epilogue operands are not loaded (the tests are uniform)
  float bias[4] = {}, res[4] = {}, msk[4] = {};
  if (p.bias) ld4f<T>((const T*)p.bias + col, bias);
  if (p.res) ld4f<T>((const T*)p.res + row * p.r_sm + col, res);
  if (p.mask) ld4f<T>((const T*)p.mask + row * p.k_sm + col, msk);
  float o[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    float acc = 0.f;
#pragma unroll
    for (int sp = 0; sp < MS; ++sp) acc += sp < ns ? part[sp][j] : 0.f;
    for (int sp = MS; sp < ns; ++sp) acc += p.ws[(int64_t)sp * total + i + j];
    float x = p.alpha * acc;
    if (p.bias) x += bias[j];
    if (p.act == kActRelu) x = fmaxf(x, 0.f);
    else if (p.act == kActGelu) x = gelu_tanh(x);
    else if (p.act == kActGeluExact) x = 0.5f * x * (1.f + erff(x * 0.70710678118654752f));
    if (p.res) x += res[j];
    if (p.mask) x = msk[j] > 0.f ? x : 0.f;
    o[j] = x;
  }
  st4<T>((T*)p.C + row * p.c_sm + col, o);
}

// Any strides, any float dtype, and int8 B with per-n scales: a plain tiled
// kernel (16x16 threads, 4x4 outputs each) used for layouts the MFMA kernels
// do not take.
template <typename T, typename TB>
__global__ void __launch_bounds__(256) gemm_generic(GArgs p) {
  __shared__ float As[16][65];
  __shared__ float Bs[16][65];
  const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
  const int64_t b = blockIdx.z;
  const int64_t m0 = (int64_t)blockIdx.y * 64, n0 = (int64_t)blockIdx.x * 64;
  const T* A = (const T*)p.A + b * p.a_sb;
  const TB* B = (const TB*)p.B + b * p.b_sb;
  float acc[4][4] = {};
  for (int64_t k0 = 0; k0 < p.K; k0 += 16) {
    for (int e = threadIdx.x; e < 16 * 64; e += 256) {
      int kk = e / 64, r = e % 64;
      int64_t gm = m0 + r, gn = n0 + r, gk = k0 + kk;
      As[kk][r] = (gm < p.M && gk < p.K) ? to_f(A[gm * p.a_sm + gk * p.a_sk]) : 0.f;
      float bv = 0.f;
      if (gn < p.N && gk < p.K) {
        bv = (float)B[gk * p.b_sk + gn * p.b_sn];
        if (p.b_scale) bv *= p.b_scale[gn];
      }
      Bs[kk][r] = bv;
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < 16; ++kk)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] += As[kk][ty * 4 + i] * Bs[kk][tx * 4 + j];
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      int64_t row = m0 + ty * 4 + i, col = n0 + tx * 4 + j;
      if (row < p.M && col < p.N) epilogue_store<T>(p, b, row, col, acc[i][j]);
    }
}

bool al16(const void* p) { return ((uintptr_t)p & 15) == 0; }

enum PlanKind { kGeneric = 0, kNative32 = 1, kMf = 2 };

struct Plan {
  int kind;
  int cfg;          // gemm_mf configuration (kMf)
  int bm, bn, bk;
  int splits;
  int64_t kps;      // k per split, a multiple of bk
};

int64_t tiles_for(const Gemm& g, int bm, int bn) {
  return ((g.M + bm - 1) / bm) * ((g.N + bn - 1) / bn) * g.batch;
}

Plan make_plan(const Gemm& g, int cus) {
  const GemmTune& tu = gemm_tune();
  Plan pl{};
  const bool is16 = g.dt == DType::F16 || g.dt == DType::BF16;
  const bool a_ok = g.a_sk == 1 || g.a_sm == 1;
  const bool b_ok = g.b_sk == 1 || g.b_sn == 1;
  pl.splits = 1;
  // fp32 activations times int8 codes with per-n scales, B k-contiguous.
  const bool int8_b = g.dt == DType::F32 && g.b_dt == DType::I8 && g.b_scale && g.b_sk == 1 && a_ok;
  if (int8_b) {
    pl.kind = kMf;
    pl.cfg = (tu.cfg == 0 || tu.cfg == 6) ? tu.cfg : (tiles_for(g, 128, 128) >= cus ? 0 : 6);
    pl.bm = kMfShape[pl.cfg].bm;
    pl.bn = kMfShape[pl.cfg].bn;
    pl.bk = kMfShape[pl.cfg].bk;
  } else if (!(a_ok && b_ok && g.b_dt == g.dt && !g.b_scale && (g.dt == DType::F32 || is16))) {
    pl.kind = kGeneric;
    pl.bm = pl.bn = 64;
    pl.bk = 16;
    pl.kps = g.K;
    return pl;
  }
  if (int8_b) {
  } else if (g.dt == DType::F32 && tu.f32_mode == kF32Native) {
    pl.kind = kNative32;
    pl.bm = g.M <= 64 ? 64 : 128;
    pl.bn = g.N <= 64 ? 64 : 128;
    pl.bk = 16;
  } else {
    pl.kind = kMf;
    if (tu.cfg >= 0 && tu.cfg < kMfConfigs) {
      pl.cfg = tu.cfg;
    } else {
      // Measured on MI355X (fp32 via bf16x3 and fp16, shapes of the GPT-2,
      // MLP and int8 workloads): 128x128 tiles win once they alone give every
      // CU a block (fp16: with 64-deep K slices), and for fp32 with M >= 256
      // and K >= 2048 when up to 8 K splits make two blocks per CU (the MLP
      // layers); otherwise 64x64 tiles with 64-deep K slices, split across
      // blocks until about two blocks per CU.
      const int64_t t128 = tiles_for(g, 128, 128);
      if (t128 >= cus) pl.cfg = is16 ? 5 : 0;
      else if (!is16 && g.M >= 256 && g.K >= 2048 && t128 * 8 >= 2LL * cus) pl.cfg = 0;
      else pl.cfg = 6;
    }
    pl.bm = kMfShape[pl.cfg].bm;
    pl.bn = kMfShape[pl.cfg].bn;
    pl.bk = kMfShape[pl.cfg].bk;
  }
  const int64_t tiles = tiles_for(g, pl.bm, pl.bn);
  const int64_t nk = (g.K + pl.bk - 1) / pl.bk;
  int splits = 1;
  if (tu.splits > 0) {
    splits = tu.splits;
  } else if (pl.kind == kMf) {
    // Split K across blocks while the grid is short of two blocks per CU and
    // every split keeps at least 3 K slices (at most 8 splits).  A grid that
    // already gives every CU a block is not split: the reduction pass over
    // the whole output costs more than the second block per CU gains (LM
    // head 128 x 50257: 62 us unsplit, 88 us in two splits).
    if (tiles < cus)
      while (tiles * splits < 2LL * cus && nk / (splits * 2) >= 3 && splits < 8) splits *= 2;
  } else {
    while (tiles * splits * 2 <= cus && nk / (splits * 2) >= 8 && splits < 32) splits *= 2;
  }
  if (splits > nk) splits = (int)(nk > 0 ? nk : 1);
  while (splits > 1 && g.batch * splits > 65535) splits /= 2;
  pl.splits = splits;
  pl.kps = ((nk + splits - 1) / splits) * pl.bk;
  return pl;
}

GArgs make_args(const Gemm& g, const Plan& pl) {
  GArgs p{};
  p.pf.first = 0x7fffffff;  // no read-ahead blocks unless a launcher adds them
  p.A = g.A; p.B = g.B; p.C = g.C;
  p.M = g.M; p.N = g.N; p.K = g.K;
  p.a_sm = g.a_sm; p.a_sk = g.a_sk; p.a_sb = g.a_sb;
  p.b_sk = g.b_sk; p.b_sn = g.b_sn; p.b_sb = g.b_sb;
  p.c_sm = g.c_sm; p.c_sb = g.c_sb;
  p.batch = g.batch;
  p.splits = pl.splits;
  p.k_per_split = pl.kps;
  p.alpha = g.alpha;
  p.bias = g.bias;
  p.act = g.act;
  p.res = g.residual; p.r_sm = g.r_sm; p.r_sb = g.r_sb;
  p.mask = g.mask; p.k_sm = g.k_sm; p.k_sb = g.k_sb;
  p.tiles_m = (int)((g.M + pl.bm - 1) / pl.bm);
  p.tiles_n = (int)((g.N + pl.bn - 1) / pl.bn);
  p.b_scale = g.b_scale;
  p.ln_g = g.ln_gamma;
  p.ln_b = g.ln_beta;
  p.ln_eps = g.ln_eps;
  p.pln_g = g.pln_gamma;
  p.pln_b = g.pln_beta;
  p.pln_y = g.pln_y;
  p.pln_eps = g.pln_eps;
  p.a_x3 = g.a_x3;
  p.c_pk = (bf16_t*)g.c_pk;
  p.pln_ypk = (bf16_t*)g.pln_ypk;
  p.rs_out = g.rs_out;
  p.rs_in = g.rs_in;
  p.rs_cs = g.rs_cs;
  p.rs_tiles = g.rs_tiles;
  p.rs_n = g.rs_n;
  p.rs_eps = g.rs_eps;
  p.rowsum_acc = (float*)g.a_rowsum_acc;
  const size_t esz = dtype_size(g.dt);
  const int vw = (int)(16 / esz);  // elements per 16-byte vector
  // Vector loads need 16-byte aligned runs along the contiguous axis.
  const int64_t a_lead = g.a_sk == 1 ? g.a_sm : g.a_sk;
  const int64_t b_lead = g.b_sk == 1 ? g.b_sn : g.b_sk;
  p.vec_a = al16(g.A) && (a_lead % vw == 0) && (g.a_sb % vw == 0);
  const int vwb = (int)(16 / dtype_size(g.b_dt));
  p.vec_b = al16(g.B) && (b_lead % vwb == 0) && (g.b_sb % vwb == 0);
  return p;
}

template <int BM, int BN>
void launch_f32(const GArgs& p, bool ak, bool bk, dim3 grid, hipStream_t s) {
  if (ak && bk) hipLaunchKernelGGL((gemm_f32_mfma<BM, BN, true, true>), grid, dim3(256), 0, s, p);
  else if (ak) hipLaunchKernelGGL((gemm_f32_mfma<BM, BN, true, false>), grid, dim3(256), 0, s, p);
  else if (bk) hipLaunchKernelGGL((gemm_f32_mfma<BM, BN, false, true>), grid, dim3(256), 0, s, p);
  else hipLaunchKernelGGL((gemm_f32_mfma<BM, BN, false, false>), grid, dim3(256), 0, s, p);
}

int cu_count() {
  static int cus = 0;
  if (!cus) {
    hipDeviceProp_t prop;
    cus = hipGetDeviceProperties(&prop, 0) == hipSuccess ? prop.multiProcessorCount : 256;
  }
  return cus;
}

}  // namespace

bool gemm_is_skinny(const Gemm& g) { return skinny_plan(g, cu_count()).use; }

// splitk_reduce_vec's conditions: one batch, rows of whole 4-vectors and
// 4-element aligned output and epilogue operands.
static bool reduce_vec_ok(const Gemm& g) {
  if (g.batch != 1 || g.N % 4 != 0 || g.c_sm % 4 != 0) return false;
  const uintptr_t al = 4 * dtype_size(g.dt) - 1;
  auto ok = [&](const void* q) { return q == nullptr || ((uintptr_t)q & al) == 0; };
  return ok(g.C) && ok(g.bias) && ok(g.residual) && ok(g.mask) && (!g.residual || g.r_sm % 4 == 0) &&
         (!g.mask || g.k_sm % 4 == 0);
}

// The packed-weight plan of g: split-K when the reduction must produce a
// layer_norm of the output.
static X3Plan x3_plan_of(const Gemm& g) {
  return x3_plan(g.M, g.N, g.K, cu_count(), g.a_x3, g.pln_y != nullptr || g.pln_ypk != nullptr);
}

// Whether a split packed-A row-panel launch finishes its tiles in the kernel
// (each tile's last-arriving split sums the splits and runs the epilogue)
// instead of leaving them to a reduction launch: not when the caller wants
// the partial sums, nor when the reduction must compute a layer_norm over
// whole rows.
static bool x3_split_inkernel(const Gemm& g, const X3Plan& pl) {
  return pl.rows && pl.apk && pl.splits > 1 && !g.no_reduce && !g.pln_y && !g.pln_ypk &&
         split_tile_counters(pl.tiles_m * pl.tiles_n) != nullptr;
}

bool gemm_x3_ok(const Gemm& g) {
  if (!g.b_x3 || g.dt != DType::F32 || g.batch != 1 || g.K % 16 != 0 || g.K <= 0 || !al16(g.A) || !al16(g.B) ||
      g.b_scale)
    return false;
  if (g.a_x3) {
    if (g.ln_gamma) return false;
  } else {
    if (g.ln_gamma && (!g.ln_beta || !gemm_x3_ln_ok(g.M, g.N, g.K))) return false;
    if (g.a_sk != 1 || (g.M > 1 && g.a_sm % 4 != 0)) return false;
  }
  if (g.c_pk || g.rs_out || g.rs_in) {
    const X3Plan pl = x3_plan_of(g);
    if (!pl.rows) return false;
    if (pl.splits > 1 && (g.rs_in || !x3_split_inkernel(g, pl))) return false;
    if (g.c_pk && (g.N % 16 != 0 || !al16(g.c_pk))) return false;
    if (g.rs_out && (g.N % 32 != 0 || ((uintptr_t)g.rs_out & 7))) return false;
    if (g.rs_in && (!g.a_x3 || !g.rs_cs || g.rs_tiles < 1 || g.rs_tiles > 48 || g.rs_n < 1 || ((uintptr_t)g.rs_in & 7)))
      return false;
  }
  if (!g.C && !g.c_pk && !g.no_reduce) return false;
  return g.c_sm == g.N;
}

bool gemm_x3_pk_out_ok(int64_t M, int64_t N, int64_t K) { return gemm_x3_panel_ok(M, N, K, true) && N % 16 == 0; }

bool gemm_x3_panel_ok(int64_t M, int64_t N, int64_t K, bool apk) {
  const X3Plan pl = x3_plan(M, N, K, cu_count(), apk, false);
  return pl.rows && pl.splits == 1;
}

bool gemm_x3_rows_out_ok(int64_t M, int64_t N, int64_t K, bool apk) {
  const X3Plan pl = x3_plan(M, N, K, cu_count(), apk, false);
  if (!pl.rows) return false;
  if (pl.splits == 1) return true;
  Gemm g;
  g.M = M; g.N = N; g.K = K;
  g.a_x3 = apk;
  return x3_split_inkernel(g, pl);
}

// The outer-product plan (gemm_x3p.hip) for fp32 products it fits, unless a
// tile configuration, a split count or the native fp32 kernels are forced,
// or its packed operands need more workspace than the caller can give.
static bool use_outer(const Gemm& g) {
  const GemmTune& tu = gemm_tune();
  return tu.cfg < 0 && tu.splits == 0 && tu.f32_mode != kF32Native && gemm_x3_outer_ok(g) &&
         gemm_x3_outer_workspace(g) <= g.max_ws;
}

// The few-row fp32 weight-streaming plan (gemm_f32s.hip), unless a tile
// configuration, a split count or the native fp32 kernels are forced.
static bool use_f32s(const Gemm& g) {
  const GemmTune& tu = gemm_tune();
  return tu.cfg < 0 && tu.splits == 0 && tu.f32_mode != kF32Native && gemm_f32_stream_ok(g, cu_count());
}

// The int8 weight-streaming plan (gemm_i8s.hip), unless a tile configuration
// or a split count is forced.
static bool use_i8s(const Gemm& g) {
  const GemmTune& tu = gemm_tune();
  return tu.cfg < 0 && tu.splits == 0 && gemm_i8_stream_ok(g);
}

// The 16-bit large-tile plan (gemm_h16.hip), unless a configuration or a
// split count is forced.
static bool use_h16(const Gemm& g) {
  const GemmTune& tu = gemm_tune();
  return tu.cfg < 0 && tu.splits == 0 && gemm_h16_ok(g, cu_count());
}

int gemm_splits(const Gemm& g) {
  if (g.b_x3) return x3_plan_of(g).splits;
  if (use_outer(g) || use_h16(g)) return 1;
  if (skinny_plan(g, cu_count()).use || thin_kind(g)) return 1;
  if (use_f32s(g)) return gemm_f32_stream_splits(g, cu_count());
  if (use_i8s(g)) return gemm_i8_stream_splits(g, cu_count());
  const Plan pl = make_plan(g, cu_count());
  return pl.kind == kMf ? pl.splits : 1;
}

// The plans that fold A's row sums in: the outer-product plan (while packing
// A) and the vector-matrix kernel (M == 1: one block also sums A's K values).
bool gemm_a_rowsum_fused(const Gemm& g) {
  if (g.dt != DType::F32 || g.b_x3) return false;
  if (skinny_plan(g, cu_count()).use) return false;
  if (const int tk = thin_kind(g)) return tk == kThinM1 && g.batch == 1;
  return use_outer(g);
}

bool gemm_post_ln_fused(const Gemm& g) {
  if (!g.b_x3 && (skinny_plan(g, cu_count()).use || thin_kind(g))) return false;
  if (g.batch != 1 || g.N > 2048 || g.N % 4 != 0 || g.c_sm != g.N) return false;
  // four-element vector accesses of C, Y and the epilogue operands
  const uintptr_t al = 4 * dtype_size(g.dt) - 1;
  auto ok = [&](const void* q) { return q == nullptr || ((uintptr_t)q & al) == 0; };
  if (!ok(g.C) || !ok(g.bias) || !ok(g.residual) || !ok(g.mask) || !ok(g.pln_gamma) || !ok(g.pln_beta) ||
      !ok(g.pln_y) || (g.residual && g.r_sm % 4 != 0) || (g.mask && g.k_sm % 4 != 0))
    return false;
  // the packed layer_norm output: fp32, whole 16-column k steps, 16-byte aligned
  if (g.pln_ypk && (g.dt != DType::F32 || g.N % 16 != 0 || !al16(g.pln_ypk))) return false;
  if (!g.pln_y && !g.pln_ypk) return false;
  if (!g.C || g.c_pk) return false;
  if (g.b_x3) return x3_plan_of(g).splits > 1;
  {
    Gemm q = g;  // the product itself takes the large-tile plan: no reduction
    q.pln_gamma = q.pln_beta = nullptr;
    q.pln_y = q.pln_ypk = nullptr;
    if (use_h16(q)) return false;
  }
  const Plan pl = make_plan(g, cu_count());
  return pl.kind == kMf && pl.splits > 1;
}

GemmTune& gemm_tune() {
  static GemmTune t = [] {
    GemmTune d;
    const char* m = getenv("APPLEGPU_GEMM_F32");
    if (m && (!strcmp(m, "native") || !strcmp(m, "f32"))) d.f32_mode = kF32Native;
    const char* sk = getenv("APPLEGPU_GEMM_SKINNY");
    if (sk && *sk == '0') d.no_skinny = true;
    const char* ik = getenv("APPLEGPU_SPLIT_INKERNEL");
    if (ik && *ik == '0') d.inkernel_splits = false;
    return d;
  }();
  return t;
}

const char* gemm_plan_name(const Gemm& g) {
  static thread_local char buf[96];
  const SkinnyPlan sp = skinny_plan(g, cu_count());
  if (sp.use) {
    snprintf(buf, sizeof buf, "skinny mfma16 blocks=%lld", (long long)sp.blocks);
    return buf;
  }
  if (const int tk = thin_kind(g)) {
    snprintf(buf, sizeof buf, "thin %s", tk == kThinN1 ? "n1" : tk == kThinM1 ? "m1" : "k1");
    return buf;
  }
  if (use_outer(g)) {
    snprintf(buf, sizeof buf, "x3 outer 128x128 tiles=%lld", (long long)((g.M / 128) * (g.N / 128)));
    return buf;
  }
  if (use_h16(g)) {
    snprintf(buf, sizeof buf, "%s", gemm_h16_name(g, cu_count()));
    return buf;
  }
  if (use_f32s(g)) {
    snprintf(buf, sizeof buf, "f32 stream 256 cols splits=%d", gemm_f32_stream_splits(g, cu_count()));
    return buf;
  }
  if (use_i8s(g)) {
    snprintf(buf, sizeof buf, "i8 stream 256 cols splits=%d", gemm_i8_stream_splits(g, cu_count()));
    return buf;
  }
  Plan pl = make_plan(g, cu_count());
  const char* kind = pl.kind == kGeneric ? "generic" : pl.kind == kNative32 ? "f32-native" : "mf";
  snprintf(buf, sizeof buf, "%s cfg%d %dx%dx%d splits=%d", kind, pl.kind == kMf ? pl.cfg : -1, pl.bm, pl.bn, pl.bk,
           pl.splits);
  return buf;
}

size_t gemm_workspace_bytes(const Gemm& g) {
  if (use_outer(g)) return gemm_x3_outer_workspace(g);
  if (use_h16(g)) return 0;
  if (g.b_x3) {
    const X3Plan xp = x3_plan_of(g);
    return xp.splits > 1 ? (size_t)xp.splits * g.M * g.N * sizeof(float) : 0;
  }
  const SkinnyPlan sp = skinny_plan(g, cu_count());
  if (sp.use || thin_kind(g)) return 0;
  if (use_f32s(g)) return (size_t)gemm_f32_stream_splits(g, cu_count()) * g.M * g.N * sizeof(float);
  if (use_i8s(g)) {
    const int ks = gemm_i8_stream_splits(g, cu_count());
    return ks > 1 ? (size_t)ks * g.M * g.N * sizeof(float) : 0;
  }
  Plan pl = make_plan(g, cu_count());
  if (pl.splits <= 1) return 0;
  return (size_t)pl.splits * g.batch * g.M * g.N * sizeof(float);
}

static void reduce_splits(const Gemm& g, const GArgs& p, hipStream_t s);

bool gemm_outer_pair_ok(const Gemm& g0, const Gemm& g1) {
  return use_outer(g0) && use_outer(g1) && gemm_x3_outer2_ok(g0, g1);
}

void gemm_outer_pair(const Gemm& g0, void* ws0, const Gemm& g1, void* ws1, hipStream_t s) {
  if (!gemm_outer_pair_ok(g0, g1)) fail("gemm: these two products do not take the paired outer-product plan");
  Plan one{};
  one.bm = one.bn = 64;
  one.splits = 1;
  one.kps = g0.K;
  gemm_x3_outer2(g0, make_args(g0, one), ws0, g1, make_args(g1, one), ws1, s);
}

void gemm(const Gemm& g, void* workspace, hipStream_t s) {
  if (g.a_rowsum_acc && !gemm_a_rowsum_fused(g)) fail("internal: A's row sums are fused only into the outer-product plan");
  if (g.M == 0 || g.N == 0 || g.batch == 0) return;
  if (g.b_x3) {
    if (!gemm_x3_ok(g))
      fail("gemm: packed fp32 weights need fp32 A with unit k stride and 16-byte aligned rows, K %% 16 == 0, "
           "one batch and a contiguous output");
    if ((g.pln_y || g.pln_ypk) && !gemm_post_ln_fused(g))
      fail("gemm: this launch cannot fuse layer_norm into its reduction");
    const X3Plan xp = x3_plan_of(g);
    if (g.no_reduce && xp.splits < 2) fail("gemm: partial sums requested from a launch without a K split");
    Plan one{};
    one.bm = xp.rows ? 32 : 128;
    one.bn = xp.rows || !xp.wide ? 32 : 64;
    one.splits = xp.splits;
    one.kps = xp.rows ? (xp.apk ? 128LL * xp.kpw : g.K) : 16LL * xp.kt;
    GArgs p = make_args(g, one);
    p.ws = (float*)workspace;
    if (xp.splits > 1 && !workspace) fail("gemm: split-K workspace missing");
    if (x3_split_inkernel(g, xp)) p.tile_cnt = split_tile_counters(xp.tiles_m * xp.tiles_n);
    gemm_x3p_launch(xp, p, s);
    reduce_splits(g, p, s);
    return;
  }
  if (g.a_x3 || g.c_pk || g.pln_ypk) fail("gemm: packed x3 rows need packed fp32 weights");
  if (g.pln_y && !gemm_post_ln_fused(g)) fail("gemm: this launch cannot fuse layer_norm into its reduction");
  if (g.no_reduce && gemm_splits(g) < 2) fail("gemm: partial sums requested from a launch without a K split");
  const SkinnyPlan sp = skinny_plan(g, cu_count());
  if (sp.use) {
    Plan one{};
    one.bm = one.bn = 1;
    one.splits = 1;
    one.kps = g.K;
    gemm_skinny(g, sp, make_args(g, one), s);
    return;
  }
  if (const int tk = thin_kind(g)) {
    Plan one{};
    one.bm = one.bn = 1;
    one.splits = 1;
    one.kps = g.K;
    gemm_thin(tk, g.dt, make_args(g, one), s);
    return;
  }
  if (g.ln_gamma) fail("gemm: a layer-norm prologue needs the skinny kernel");
  if (g.b_packed) fail("gemm: packed weights need the skinny kernel (at most 16 fp16/bf16 rows)");
  if (use_outer(g)) {
    Plan one{};
    one.bm = one.bn = 64;
    one.splits = 1;
    one.kps = g.K;
    gemm_x3_outer(g, make_args(g, one), workspace, s);
    return;
  }
  if (use_f32s(g)) {
    Plan fs{};
    fs.bm = 64;
    fs.bn = 256;
    fs.splits = gemm_f32_stream_splits(g, cu_count());
    fs.kps = g.K / fs.splits;
    GArgs p = make_args(g, fs);
    p.ws = (float*)workspace;
    if (!workspace) fail("gemm: split-K workspace missing");
    gemm_f32_stream(g, p, cu_count(), s);
    reduce_splits(g, p, s);
    return;
  }
  if (use_i8s(g)) {
    Plan st{};
    st.bm = 64;
    st.bn = 256;
    st.splits = gemm_i8_stream_splits(g, cu_count());
    const int64_t phases = (g.K + 127) / 128;
    st.kps = (phases + st.splits - 1) / st.splits * 128;
    GArgs p = make_args(g, st);
    p.ws = (float*)workspace;
    gemm_i8_stream(g, p, s);
    reduce_splits(g, p, s);
    return;
  }
  if (use_h16(g)) {
    Plan one{};
    one.bm = one.bn = 128;
    one.splits = 1;
    one.kps = g.K;
    gemm_h16(g, make_args(g, one), cu_count(), s);
    return;
  }
  Plan pl = make_plan(g, cu_count());
  GArgs p = make_args(g, pl);
  p.ws = (float*)workspace;
  if (pl.splits > 1 && !workspace) fail("gemm: split-K workspace missing");
  if (pl.kind == kGeneric) {
    if (g.batch > 65535) fail("gemm: batch %lld too large", (long long)g.batch);
    dim3 grid((unsigned)((g.N + 63) / 64), (unsigned)((g.M + 63) / 64), (unsigned)g.batch);
    p.splits = 1;
    if (g.b_scale) {
      if (g.b_dt != DType::I8) fail("gemm: scaled B operand must be int8");
      AGPU_FLOAT_SWITCH(g.dt, hipLaunchKernelGGL((gemm_generic<T, int8_t>), grid, dim3(256), 0, s, p));
    } else {
      AGPU_FLOAT_SWITCH(g.dt, hipLaunchKernelGGL((gemm_generic<T, T>), grid, dim3(256), 0, s, p));
    }
    check_launch("gemm_generic");
    return;
  }
  if (g.batch * pl.splits > 65535) fail("gemm: batch %lld too large", (long long)g.batch);
  const int64_t nblocks = (int64_t)p.tiles_m * p.tiles_n;
  if (nblocks > 0x7fffffff) fail("gemm: too many tiles");
  const bool ak = g.a_sk == 1, bk = g.b_sk == 1;
  dim3 grid((unsigned)nblocks, (unsigned)(g.batch * pl.splits));
  if (pl.kind == kNative32) {
    if (pl.bm == 128 && pl.bn == 128) launch_f32<128, 128>(p, ak, bk, grid, s);
    else if (pl.bm == 128) launch_f32<128, 64>(p, ak, bk, grid, s);
    else if (pl.bn == 128) launch_f32<64, 128>(p, ak, bk, grid, s);
    else launch_f32<64, 64>(p, ak, bk, grid, s);
  } else {
    // Unmasked loads need 16-byte aligned runs and whole 16-byte vectors:
    // K % VW == 0 for an operand contiguous along k, rows % VW == 0 for one
    // contiguous along its rows.
    const int64_t vw = 16 / (int64_t)dtype_size(g.dt);
    const int64_t vwb = 16 / (int64_t)dtype_size(g.b_dt);
    const bool fast = p.vec_a && p.vec_b && (ak ? g.K % vw == 0 : g.M % vw == 0) &&
                      (bk ? g.K % vwb == 0 : g.N % vwb == 0);
    if (g.b_dt == DType::I8) launch_mf_f32_i8(p, pl.cfg, ak, fast, grid, s);
    else if (g.dt == DType::F32) launch_mf_f32(p, pl.cfg, ak, bk, fast, grid, s);
    else if (g.dt == DType::F16) launch_mf_f16(p, pl.cfg, ak, bk, fast, grid, s);
    else launch_mf_bf16(p, pl.cfg, ak, bk, fast, grid, s);
  }
  check_launch("gemm_mfma");
  reduce_splits(g, p, s);
}

namespace {
Prefetch& pending_prefetch() {
  static Prefetch pf;
  return pf;
}
}  // namespace

void set_prefetch(const Prefetch& pf) { pending_prefetch() = pf; }

Prefetch take_prefetch() {
  Prefetch pf = pending_prefetch();
  pending_prefetch() = Prefetch{};
  return pf;
}

PfArgs make_prefetch(int main, int threads) {
  PfArgs a{};
  a.first = main;
  const Prefetch pf = take_prefetch();
  int64_t lines = 0;
  for (int i = 0; i < pf.n && i < 3; ++i) {
    if (!pf.ptr[i] || pf.bytes[i] < 64) continue;
    a.p[a.n] = (const char*)pf.ptr[i];
    a.lines[a.n] = pf.bytes[i] >> 6;
    lines += a.lines[a.n];
    ++a.n;
  }
  if (!a.n) return a;
  // one thread per line per pass; 32 KB (512 lines) per block, at most 256
  // blocks (more blocks measured slower: their dispatch lengthens the launch)
  int64_t blocks = (lines + 511) / 512;
  blocks = blocks < 1 ? 1 : blocks > 256 ? 256 : blocks;
  (void)threads;
  a.blocks = (int)blocks;
  return a;
}

// The split-K tail of a launch: partial sums in p.ws are reduced (in split
// order) into C with the epilogue, and layer_norm(C) into Y when asked.
static void reduce_splits(const Gemm& g, const GArgs& p, hipStream_t s) {
  if (p.splits > 1) {
    if (g.no_reduce || p.tile_cnt) return;  // (tiles finished in the GEMM launch)
    if (g.pln_y || g.pln_ypk) {
      if (!gemm_post_ln_fused(g)) fail("gemm: this launch cannot fuse layer_norm into its reduction");
      AGPU_FLOAT_SWITCH(g.dt, launch_reduce_ln<T>(p, s));
      check_launch("splitk_reduce_ln");
      return;
    }
    int64_t total = g.batch * g.M * g.N;
    if (reduce_vec_ok(g) && (total + 1023) / 1024 <= 0x7fffffff) {
      const dim3 rgrid((unsigned)((total + 1023) / 1024));
      AGPU_FLOAT_SWITCH(g.dt, {
        if (p.splits <= 2) hipLaunchKernelGGL((splitk_reduce_vec<T, 2>), rgrid, dim3(256), 0, s, p);
        else if (p.splits <= 4) hipLaunchKernelGGL((splitk_reduce_vec<T, 4>), rgrid, dim3(256), 0, s, p);
        else if (p.splits <= 8) hipLaunchKernelGGL((splitk_reduce_vec<T, 8>), rgrid, dim3(256), 0, s, p);
        else if (p.splits <= 16) hipLaunchKernelGGL((splitk_reduce_vec<T, 16>), rgrid, dim3(256), 0, s, p);
        else hipLaunchKernelGGL((splitk_reduce_vec<T, 32>), rgrid, dim3(256), 0, s, p);
      });
      check_launch("splitk_reduce");
      return;
    }
    int64_t blocks = (total + 1023) / 1024;
    if (blocks > 65536) blocks = 65536;
    AGPU_FLOAT_SWITCH(g.dt, hipLaunchKernelGGL((splitk_reduce<T>), dim3((unsigned)blocks), dim3(256), 0, s, p));
    check_launch("splitk_reduce");
  } else if (g.pln_y || g.pln_ypk) {
    fail("gemm: layer_norm fusion needs a split-K launch");
  }
}

}  // namespace k
}  // namespace agpu
