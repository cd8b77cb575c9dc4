// fp32 activations of up to a few hundred rows times int8 weight codes with a
// scale per output column (C[m][n] = scale[n] sum_k A[m][k] q[n][k]): each
// code is read once, straight into registers, and becomes a bf16 there.
//
// Bound by the requests that a CU has in flight (8192 x 8192 codes: 19 us at
// one row, 3.5 TB/s; 30 at 64 rows, beside A's loads and splits).  A code
// (-128 .. 127) is exact in bf16, so the fp32 sum needs two products, A's hi
// and lo halves times the code, and the scale once at the end; dequantizing
// first takes three products of split operands, a rounding more, and an LDS
// round trip of the weights.  Where the sum passes fp32's range before the
// scale is applied (values past 2^121), that output is summed again in 64
// bits.  Figures at the dispatch rule below.
//
// A block of 8 wavefronts owns 256 columns and 32 RS rows over one of KS
// ranges of K.  Wavefront w takes 64 columns (strip w % 4) of one half (w / 4)
// of the k: two column strips for each fragment of A that it reads, half the
// LDS reads of one strip (64 rows took the same time with one).  A phase is 128 k: of its half, lane l holds 32 codes from 32 (l / 32)
// of the columns l % 32 and 32 + l % 32, four 16-byte loads, requested two
// phases ahead (64 KB in flight a block).  Step t of a half multiplies codes
// 8 t .. + 7, so A's fragment of lane l at step t is row l % 32, k 32 (l / 32)
// + 8 t .. + 7; the block splits A once a phase into such fragments, in one of
// two LDS buffers while the other is read.  The halves are added through LDS,
// ranges by the split-K reduction in order, so results repeat exactly.
#include "gemm_kernels.hpp"

namespace agpu {
namespace k {

namespace {

constexpr int kI8Phase = 128;  // k per phase: 8 steps of 16
constexpr int kI8Cols = 256;   // columns per block

// 16 codes, from `k` or, where they would pass the end of a ragged row, its
// last 16.
template <bool RAGGED>
__device__ __forceinline__ uint4 i8_load(const int8_t* row, int k, int K) {
  uint4 v;
  __builtin_memcpy(&v, row + (!RAGGED || k < K - 16 ? k : K - 16), 16);
  return v;
}

// The codes of a load that was moved back by `by` bytes, in their own places
// (what is past the row's end meets zeros of A).
__device__ __forceinline__ uint4 i8_shift(uint4 v, int by) {
  uint64_t lo = (uint64_t)v.y << 32 | v.x, hi = (uint64_t)v.w << 32 | v.z;
  if (by >= 8) {
    lo = hi;
    hi = 0;
    by -= 8;
  }
  if (by >= 8) {
    lo = 0;
  } else if (by > 0) {
    lo = lo >> 8 * by | hi << (64 - 8 * by);
    hi >>= 8 * by;
  }
  return uint4{(uint32_t)lo, (uint32_t)(lo >> 32), (uint32_t)hi, (uint32_t)(hi >> 32)};
}

// 8 codes as bf16, exactly: the upper halves of their floats.
__device__ __forceinline__ bf16x8_t i8_bf16(uint32_t a, uint32_t b) {
  uint32_t o[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t w = i < 2 ? a : b;
    const int s = 16 * (i & 1);
    const float x = (float)(int8_t)(w >> s), y = (float)(int8_t)(w >> (s + 8));
    o[i] = __builtin_amdgcn_perm(__float_as_uint(y), __float_as_uint(x), 0x07060302u);
  }
  bf16x8_t r;
  __builtin_memcpy(&r, o, 16);
  return r;
}

// Grid: (column groups x KS, row groups) blocks of 512 threads; p.k_per_split
// is a whole number of phases; K >= 16.  RAGGED: K is not.
template <int RS, bool RAGGED>
__global__ void __launch_bounds__(512, 1) gemm_i8_stream_kernel(GArgs p, int KS) {
  // A's fragments of a phase: strip i, step t, hi or lo: 64 lanes x 8 values,
  // padded by 8, so that the 16 pieces of a row, which one wavefront writes
  // at a time, fall into different banks (two of each)
  constexpr int FRAG = 512 + 8;
  constexpr int BUF = RS * 8 * 2 * FRAG;
  __shared__ __attribute__((aligned(16))) bf16_t sA[2 * BUF];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int64_t grp = blockIdx.x / KS, ks = blockIdx.x % KS;
  const int64_t m0 = (int64_t)blockIdx.y * 32 * RS;
  const int K = (int)p.K, kbeg = (int)(ks * p.k_per_split);
  const int nph = (min(K - kbeg, (int)p.k_per_split) + kI8Phase - 1) / kI8Phase;
  const int half = w >> 2;
  const int64_t n = grp * kI8Cols + (w & 3) * 64 + (lane & 31);  // and n + 32
  const int8_t* Bn[2];
#pragma unroll
  for (int c = 0; c < 2; ++c) Bn[c] = (const int8_t*)p.B + (n + 32 * c < p.N ? n + 32 * c : p.N - 1) * p.b_sn;
  // This thread's piece of A in each row strip: 8 values of row 4 w + l / 16,
  // the l % 16-th of the phase (whole rows of 512 bytes for each 16 lanes): a
  // row past M is row M - 1 again and is not stored.
  const int arw = 4 * w + (lane >> 4), ap = lane & 15;
  const float* arow[RS];
#pragma unroll
  for (int r = 0; r < RS; ++r) {
    const int64_t row = m0 + 32 * r + arw;
    arow[r] = (const float*)p.A + (row < p.M ? row : p.M - 1) * p.a_sm;
  }
  // of half ap / 8, k 32 (ap / 4 % 2) + 8 (ap % 4)
  const int ak = 8 * ap, ast = ((ap >> 3) * 4 + (ap & 3)) * 2 * FRAG + 8 * (arw + 32 * ((ap >> 2) & 1));
  const int bk = 64 * half + 32 * (lane >> 5);
  // Phases run from a start of the block's own, so that at any one time the
  // blocks read different offsets of the rows (rows of a power of two bytes
  // read at one offset fall into few memory channels).
  const int rot = (int)((grp + ks) % nph);
  auto kof = [&](int ph) __attribute__((always_inline)) {
    ph = ph < nph ? ph : nph - 1;  // past the end: read again, never used
    return kbeg + (ph + rot < nph ? ph + rot : ph + rot - nph) * kI8Phase;
  };
  float a[2][RS][8];  // by phase parity
  auto load_a = [&](int ph, auto parity) __attribute__((always_inline)) {
    constexpr int b = decltype(parity)::value;
    const int k = kof(ph) + ak;
    if (!RAGGED || k - ak + kI8Phase <= K) {
#pragma unroll
      for (int r = 0; r < RS; ++r) __builtin_memcpy(a[b][r], arow[r] + k, 32);
    } else {
#pragma unroll
      for (int r = 0; r < RS; ++r)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float v = arow[r][k + e < K ? k + e : K - 1];
          a[b][r][e] = k + e < K ? v : 0.f;
        }
    }
  };
  auto write_a = [&](auto parity) __attribute__((always_inline)) {
    constexpr int b = decltype(parity)::value;
#pragma unroll
    for (int r = 0; r < RS; ++r) {
      bf16x8_t h, l;
#pragma unroll
      for (int e = 0; e < 8; e += 2) {
        bf16x2_t h2, l2;
        split_bf16x2(a[b][r][e], a[b][r][e + 1], h2, l2);
        h[e] = h2.x; h[e + 1] = h2.y;
        l[e] = l2.x; l[e + 1] = l2.y;
      }
      bf16_t* d = sA + b * BUF + r * 16 * FRAG + ast;
      *(bf16x8_t*)d = h;
      *(bf16x8_t*)(d + FRAG) = l;
    }
  };
  const std::integral_constant<int, 0> even;
  const std::integral_constant<int, 1> odd;
  uint4 code[2][2][2];  // phase parity, 16 k, column strip
  load_a(0, even);
#pragma unroll
  for (int b = 0; b < 2; ++b) {
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int c = 0; c < 2; ++c) code[b][j][c] = i8_load<RAGGED>(Bn[c], kof(b) + bk + 16 * j, K);
    if (b == 0) load_a(1, odd);
  }
  write_a(even);
  __syncthreads();
  f32x16 acc[RS][2];
#pragma unroll
  for (int i = 0; i < RS; ++i)
#pragma unroll
    for (int c = 0; c < 2; ++c)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][c][e] = 0.f;
  auto phase = [&](int ph, auto parity) __attribute__((always_inline)) {
    constexpr int b = decltype(parity)::value;
    // both operands two phases ahead: loads return in order, so one phase for
    // A would wait for the codes requested before it
    load_a(ph + 2, parity);
    const bf16_t* f = sA + b * BUF + half * 8 * FRAG + 8 * lane;
    const int k = kof(ph);
    const int knext = kof(ph + 2) + bk;
    const bool whole = !RAGGED || k + kI8Phase <= K;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      // converted before the registers take the next codes: no copies
      bf16x8_t q[2][2];
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        uint4 v = code[b][j][c];
        if (!whole) {
          const int back = k + bk + 16 * j - (K - 16);
          v = i8_shift(v, back <= 0 ? 0 : back < 16 ? back : 16);
        }
        q[0][c] = i8_bf16(v.x, v.y);
        q[1][c] = i8_bf16(v.z, v.w);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int c = 0; c < 2; ++c) code[b][j][c] = i8_load<RAGGED>(Bn[c], knext + 16 * j, K);
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int i = 0; i < RS; ++i) {
          const bf16x8_t h = *(const bf16x8_t*)(f + ((i * 8 + 2 * j + u) * 2) * FRAG);
          const bf16x8_t l = *(const bf16x8_t*)(f + ((i * 8 + 2 * j + u) * 2 + 1) * FRAG);
#pragma unroll
          for (int c = 0; c < 2; ++c) acc[i][c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(l, q[u][c], acc[i][c], 0, 0, 0);
#pragma unroll
          for (int c = 0; c < 2; ++c) acc[i][c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(h, q[u][c], acc[i][c], 0, 0, 0);
        }
      // each load stays where it is (else the scheduler sinks a phase's loads
      // below its products)
      __builtin_amdgcn_sched_barrier(0);
    }
    write_a(std::integral_constant<int, b ^ 1>{});
    __syncthreads();
  };
  int ph = 0;
  for (; ph + 1 < nph; ph += 2) {
    phase(ph, even);
    phase(ph + 1, odd);
  }
  if (ph < nph) phase(ph, even);
  // the second half's sums through LDS: wavefront w takes column strip
  // w / 4 of its 64 columns, the other half's strip of it from LDS (the loop
  // ended with a barrier, A's fragments are done with)
  constexpr int RED = RS * 16 * 64;
  static_assert(8 * RED * 4 <= 4 * BUF, "the sums fit the fragments' space");
  float* red = (float*)sA;
#pragma unroll
  for (int i = 0; i < RS; ++i)
#pragma unroll
    for (int e = 0; e < 16; ++e) red[w * RED + (i * 16 + e) * 64 + lane] = acc[i][half ? 0 : 1][e];
  __syncthreads();
  const int64_t nc = n + 32 * half;
  if (nc >= p.N) return;
  // A scale that is not finite makes its column NaN, as multiplying each code
  // by it and splitting the product does.
  float sc = p.b_scale[nc];
  if (!(fabsf(sc) < INFINITY)) sc = NAN;
  float* ws = p.ws + ks * (p.M * p.N);
  auto put = [&](int64_t row, float v) __attribute__((always_inline)) {
    if (KS > 1) ws[row * p.N + nc] = v;
    else ((float*)p.C)[row * p.c_sm + nc] = v;
  };
  uint32_t over = 0;  // bit 16 i + r: an output whose sum is not finite
#pragma unroll
  for (int i = 0; i < RS; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int64_t row = m0 + 32 * i + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
      if (row < p.M) {
        const float v = (half ? acc[i][1][r] : acc[i][0][r]) + red[(w ^ 4) * RED + (i * 16 + r) * 64 + lane];
        put(row, v * sc);
        if (!(fabsf(v) < INFINITY)) over |= 1u << (16 * i + r);
      }
    }
  const int kend = min(K, kbeg + (int)p.k_per_split);
  const int8_t* q = half ? Bn[1] : Bn[0];
  for (; over; over &= over - 1) {
    const int e = __builtin_ctz(over);
    const int64_t row = m0 + 32 * (e >> 4) + 8 * ((e >> 2) & 3) + 4 * (lane >> 5) + (e & 3);
    const float* a1 = (const float*)p.A + row * p.a_sm;
    double v = 0;
    for (int k = kbeg; k < kend; ++k) v += (double)a1[k] * q[k];
    put(row, (float)(v * sc));
  }
}

int i8s_strips(const Gemm& g) { return g.M <= 32 ? 1 : 2; }

}  // namespace

// Ranges of K, by time: 2.3 us a phase at one row strip and 3.2 at two, a
// launch's start and end spread over the 8 phases that a block of 8192 x 8192
// codes has in it (at more phases each takes 1.5 and 1.9 us), and
// each range writes and the reduction reads M x N floats, about 4 bytes a ps
// for the whole chip, after a launch of 3 us and 0.25 us for each range that
// an output's thread adds (64 x 8192 x 512: 17 us in 32 ranges, 35 in 64).
// Grids stay within one block per CU.  Over 1 to 128 rows of 256 x 512 to 8192
// x 8192 codes the choice is within 2% of the best power of two, 18% at worst
// (32 x 8192 x 512: 11.4 us in 4 ranges, 9.7 in one).
int gemm_i8_stream_splits(const Gemm& g, int cus) {
  const int64_t rows = 32 * i8s_strips(g);
  const int64_t blocks = (g.N + kI8Cols - 1) / kI8Cols * ((g.M + rows - 1) / rows);
  const int64_t phases = (g.K + kI8Phase - 1) / kI8Phase;
  int best = 1;
  double tbest = 0;
  for (int64_t s = 1; s <= 64 && s <= phases && (s == 1 || blocks * s <= cus); ++s) {
    const int64_t per = (phases + s - 1) / s;
    if ((phases + per - 1) / per != s) continue;  // a range would be empty
    if (s > 1 && (size_t)s * g.M * g.N * sizeof(float) > g.max_ws) break;
    const double rounds = (double)((blocks * s + cus - 1) / cus);
    const double t = rounds * per * (rows > 32 ? 3.2 : 2.3) + (s > 1 ? 3.0 + 0.25 * s + s * g.M * g.N * 8 / 4e6 : 0.0);
    if (s == 1 || t < tbest) {
      best = (int)s;
      tbest = t;
    }
  }
  return best;
}

// Where the codes are streamed, over rows x columns x k (us, tiles -> this, codes
// not in cache).  A launch here starts with two phases of loads and ends with a
// reduction; the tiles start faster and have larger grids, so below some k they
// win, the sooner the more rows there are:
//  - to 16 rows from 128 k (16 x 1024 x 64: 5.6 -> 9.1, x 128: equal, 1 x 8192 x
//    8192: 50 -> 23, 8 x 4096 x 4096: 20 -> 13), to 32 rows from 256 k (32 x 1024
//    x 128: 1.1 times as long here, x 512: 0.88);
//  - to 64 rows, two row strips a block, from 4096 k, or 3072 of as many columns
//    (64 x 8192 x 512: 1.4 times as long here, x 2048: 1.1, x 3072: 0.89, x 8192:
//    55 -> 35; 64 x 1024 x 4096: 1.0);
//  - more rows read the codes once per 64 and gain where the codes are many: to
//    128 rows from 6 M codes (100 x 2048 x 2048: 1.0, 128 x 4096 x 2048: 0.97, 128
//    x 8192 x 8192: 0.39), to 256 from 4 M, where the tiles' grid leaves a short
//    last round (256 x 4096 x 2048: 0.79, 256 x 8192 x 768: 0.88, 256 x 4096 x
//    1024: 1.2, so the shorter k only with many columns), each from 2048 k, or
//    with 8192 k whatever the columns (100 x 256 x 8192: 0.75);
//  - rows that 16 bytes do not divide, which the tiles load masked: from 128 k, to
//    256 rows from 192 (64 x 256 x 100: 1.6, 256 x 300 x 300: 20 -> 13, 200 x 8192
//    x 8191: 0.24).
static bool i8_stream_pays(int64_t M, int64_t N, int64_t K) {
  constexpr int64_t kM = 1 << 20;
  if (M <= 16) return K >= 128;
  if (K % 16 != 0) return K >= (M <= 32 ? 128 : 192);
  if (M <= 32) return K >= 256;
  if (M <= 64) return K >= 4096 || (K >= 3072 && N >= 3072);
  if (K >= 8192) return true;
  if (M <= 128) return K >= 2048 && N * K >= 6 * kM;
  return N * K >= 4 * kM && (K >= 2048 || N >= 6144);
}

bool gemm_i8_stream_ok(const Gemm& g) {
  return g.dt == DType::F32 && g.b_dt == DType::I8 && g.b_scale && g.batch == 1 && g.a_sk == 1 && g.b_sk == 1 &&
         g.M >= 1 && g.M <= 256 && g.N >= 1 && g.K >= 16 && g.K < (1LL << 30) &&
         i8_stream_pays(g.M, g.N, g.K) && g.alpha == 1.f && !g.bias && !g.residual &&
         !g.mask && g.act == 0 && !g.b_x3 && !g.a_x3 && !g.b_packed && !g.ln_gamma && !g.c_pk && !g.pln_y && !g.pln_ypk &&
         !g.no_reduce && !g.a_rowsum_acc && !g.rs_out && !g.rs_in && (g.N + kI8Cols - 1) / kI8Cols <= 0x1000000;
}

void gemm_i8_stream(const Gemm& g, const GArgs& p, hipStream_t s) {
  const int rs = i8s_strips(g);
  if (!gemm_i8_stream_ok(g) || p.splits < 1 || p.k_per_split < kI8Phase || p.k_per_split % kI8Phase != 0 ||
      p.k_per_split * (p.splits - 1) >= g.K || p.k_per_split * p.splits < g.K || (p.splits > 1 && !p.ws))
    fail("internal: gemm_i8_stream plan does not match its arguments");
  const dim3 grid((unsigned)((g.N + kI8Cols - 1) / kI8Cols * p.splits), (unsigned)((g.M + 32 * rs - 1) / (32 * rs)));
  const bool ragged = g.K % kI8Phase != 0;
#define AGPU_I8S(RS)                                                                                             \
  do {                                                                                                           \
    if (ragged) hipLaunchKernelGGL((gemm_i8_stream_kernel<RS, true>), grid, dim3(512), 0, s, p, p.splits);       \
    else hipLaunchKernelGGL((gemm_i8_stream_kernel<RS, false>), grid, dim3(512), 0, s, p, p.splits);             \
  } while (0)
  if (rs == 1) AGPU_I8S(1);
  else AGPU_I8S(2);
#undef AGPU_I8S
  check_launch("gemm_i8_stream");
}

}  // namespace k
}  // namespace agpu
