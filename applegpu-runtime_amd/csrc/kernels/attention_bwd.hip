// Backward of fused fp32 attention: with P = softmax(scale Q K^T [causal])
// and delta_i = sum_j P_ij dP_ij,
//   dV = P^T dO,  dP = dO V^T,  dS = P (dP - delta),
//   dQ = scale dS K,  dK = scale dS^T Q.
// P is recomputed tile by tile, so neither P nor dS reaches memory, tiles
// above the causal diagonal are never formed and every gradient has one
// writer and one summation order.  The composition it replaces ran five GEMMs
// over [.., Tq, Tk] arrays with softmax, its backward and three scalings
// between them, causal or not (2 x 12 heads x 777 x 777, D = 64, causal:
// 430 us; 87 us here: 28 for the statistics, 58 for the gradients, a sixth of
// the MFMA peak, latency-bound with one block of each CU in flight).
//
// Two launches.  The first forms each query row's log-sum-exp and delta (two
// products a tile pair).  The second holds both halves of the rest: blocks of
// own rows = keys (dK and dV, four products) and blocks of own rows = queries
// (dQ, three products).  All stream the other side's rows in 64-row tiles
// through LDS.  Products run on bf16 MFMA with every fp32 operand split into
// hi + lo (three MFMAs: lo hi + hi lo + hi hi, fp32 accumulation), as the
// GEMMs do.  The statistics come from the same split products as P and dP:
// rows of P then sum to one and dS to zero up to fp32 rounding, whatever the
// split's own error.  (Taken from the forward's exact fp32 scores and from
// dO . O instead, which saves the first launch's products, the gradients' error
// against float64 grew by 10% at 777 rows and by half at 16.)
//
// A block has four wavefronts: two groups of own rows times two halves of the
// tile's stream rows, so that a fragment read from LDS serves 16 KG own rows.
// With v_mfma_f32_16x16x32 (lane l: A row and B column l % 16 at k = 8 (l /
// 16) .. + 8; C register r: row 4 (l / 16) + r, column l % 16):
//  - S and dP: A = stream rows from LDS, B = the block's own rows, held in
//    registers for the whole kernel.  A lane then has 4 stream rows of one own
//    row in each 16-row subtile;
//  - the second products contract over the stream rows: B = the lane's own P
//    or dS values as they are, A = the stream rows transposed.  The order of k
//    is free as long as A and B agree, so the transposed tile holds each 32
//    rows in the order 8 g + 4 t + r of the row 16 t + 4 g + r, and a fragment
//    is one 16-byte read;
//  - the halves' sums meet in LDS at the end.
// LDS rows are unpadded; 16-byte chunks are exchanged within a row (chunk ^
// row bits) so that the 16 lanes of a fragment read cover every bank.
#include "device.hpp"
#include "gemm_kernels.hpp"  // split_bf16x2

#include <algorithm>
#include <array>
#include <type_traits>

namespace agpu {
namespace k {
using namespace dev;

namespace {

typedef __bf16 bw8 __attribute__((ext_vector_type(8)));
typedef __bf16 bw4 __attribute__((ext_vector_type(4)));
typedef float bwf4 __attribute__((ext_vector_type(4)));

constexpr int kBwRows = 64;  // stream rows per tile

struct BwSide {  // one [B, H, T, D] operand, unit stride along D
  const float* p;
  int64_t sb, sh, st;
};
struct BwArgs {
  BwSide q, k, v, go;
  float *lse, *delta;   // [B, H, Tq]; log-sum-exp in units of log 2
  float *dq, *dk, *dv;  // contiguous [B, H, T, D]
  int BH, H, Tq, Tk;
  float scale;
  int causal;
  int kv_blocks;  // blocks below this own keys, the rest queries
};

// Chunk swizzles: of row-major tiles of D columns, and of transposed tiles
// (64 columns; the writers hold every fourth row).
template <int D>
__device__ __forceinline__ int bw_swz(int row) {
  return (row * (D / 8) / 16) & (D / 8 - 1);
}
__device__ __forceinline__ int bw_swz_t(int d) { return ((d >> 1) ^ (d >> 4)) & 7; }

template <int D>
struct BwTile {
  static constexpr int CG = D / 4;                  // groups of 4 columns
  static constexpr int NB = 2 * 16 * CG / 256;      // 4 x 4 blocks per thread over both operands
  static constexpr int ARR = kBwRows * D;           // elements of one tile array
  float4 x[NB][4];
  // block i of this thread: operand a, rows 4 rg .., columns 4 dg ..
  static __device__ __forceinline__ void where(int i, int tid, int& a, int& rg, int& dg) {
    const int e = tid + 256 * i;
    a = e / (16 * CG);
    rg = e % (16 * CG) / CG;
    dg = e % CG;
  }
  __device__ __forceinline__ void load(const float* y1, int64_t st1, const float* y2, int64_t st2, int row0, int T,
                                       int tid) {
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      int a, rg, dg;
      where(i, tid, a, rg, dg);
      const float* base = (a ? y2 : y1) + 4 * dg;
      const int64_t st = a ? st2 : st1;
#pragma unroll
      for (int y = 0; y < 4; ++y) x[i][y] = *(const float4*)(base + min(row0 + 4 * rg + y, T - 1) * st);
    }
  }
  // s: row-major hi, lo of both operands, then transposed hi, lo of the first
  // TR operands
  template <int TR>
  __device__ __forceinline__ void store(bf16_t* s, int tid) const {
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      int a, rg, dg;
      where(i, tid, a, rg, dg);
      const float* f = (const float*)&x[i][0];
      bf16_t hi[4][4], lo[4][4];
#pragma unroll
      for (int y = 0; y < 4; ++y)
#pragma unroll
        for (int c = 0; c < 4; c += 2) {
          bf16x2_t h, l;
          split_bf16x2(f[4 * y + c], f[4 * y + c + 1], h, l);
          hi[y][c] = h.x; hi[y][c + 1] = h.y;
          lo[y][c] = l.x; lo[y][c + 1] = l.y;
        }
      bf16_t* rm = s + a * 2 * ARR;
#pragma unroll
      for (int y = 0; y < 4; ++y) {
        const int row = 4 * rg + y;
        bf16_t* d = rm + row * D + ((dg >> 1) ^ bw_swz<D>(row)) * 8 + (dg & 1) * 4;
        *(bw4*)d = bw4{hi[y][0], hi[y][1], hi[y][2], hi[y][3]};
        *(bw4*)(d + ARR) = bw4{lo[y][0], lo[y][1], lo[y][2], lo[y][3]};
      }
      if (a >= TR) continue;
      bf16_t* tr = s + (4 + a * 2) * ARR;
      const int r0 = 4 * rg;
      const int pos = (r0 & 32) | ((r0 & 12) << 1) | ((r0 & 16) >> 2);
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int dd = 4 * dg + c;
        bf16_t* d = tr + dd * kBwRows + ((pos >> 3) ^ bw_swz_t(dd)) * 8 + (pos & 7);
        *(bw4*)d = bw4{hi[0][c], hi[1][c], hi[2][c], hi[3][c]};
        *(bw4*)(d + ARR) = bw4{lo[0][c], lo[1][c], lo[2][c], lo[3][c]};
      }
    }
  }
};

__device__ __forceinline__ bwf4 bw_mfma(bw8 a, bw8 b, bwf4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
// c += (ah + al) (bh + bl) without al bl
__device__ __forceinline__ bwf4 bw_mfma3(bw8 ah, bw8 al, bw8 bh, bw8 bl, bwf4 c) {
  c = bw_mfma(al, bh, c);
  c = bw_mfma(ah, bl, c);
  return bw_mfma(ah, bh, c);
}

// 8 consecutive floats as hi and lo fragments
__device__ __forceinline__ void bw_split8(const float* p, bw8& h, bw8& l) {
  float4 a = *(const float4*)p, b = *(const float4*)(p + 4);
  const float f[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
  for (int c = 0; c < 8; c += 2) {
    bf16x2_t hh, ll;
    split_bf16x2(f[c], f[c + 1], hh, ll);
    h[c] = hh.x; h[c + 1] = hh.y;
    l[c] = ll.x; l[c + 1] = ll.y;
  }
}

// (m, l, d) and (m2, l2, d2): running maximum, sum of P and sum of P dP.
__device__ __forceinline__ void bw_merge(float& m, float& l, float& d, float m2, float l2, float d2) {
  const float mx = fmaxf(m, m2), mu = mx == -INFINITY ? 0.f : mx;
  const float a = __builtin_amdgcn_exp2f(m - mu), b = __builtin_amdgcn_exp2f(m2 - mu);
  m = mx;
  l = l * a + l2 * b;
  d = d * a + d2 * b;
}

// Own rows per wavefront group: two 16-row groups, one at D = 128 (where the
// own operands and sums of two would not fit 256 registers).
template <int D> constexpr int kBwGroups = D == 128 ? 1 : 2;
template <int D> constexpr int kBwOwn = 2 * 16 * kBwGroups<D>;

// What a block's own rows are: queries for their statistics or for dQ, or keys.
enum BwKind { kBwStats, kBwQ, kBwKV };

template <int D, BwKind KIND>
__device__ __forceinline__ void bw_block(const BwArgs& p, int blk, bf16_t* s, float (*rowv)[kBwRows]) {
  constexpr int KG = kBwGroups<D>, OWN = kBwOwn<D>, DS = D / 32, DT = D / 16, ARR = kBwRows * D;
  constexpr bool DKV = KIND == kBwKV, STATS = KIND == kBwStats;
  constexpr int NA = DKV ? 2 : STATS ? 0 : 1;  // gradients of the own rows
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int l16 = lane & 15, g = lane >> 4, grp = w >> 1, half = w & 1;
  const int bh = blk % p.BH;
  const int own_T = DKV ? p.Tk : p.Tq, str_T = DKV ? p.Tq : p.Tk;
  const int tiles_own = (own_T + OWN - 1) / OWN;
  // the longest first: the first keys, the last queries
  const int ot = DKV ? blk / p.BH : tiles_own - 1 - blk / p.BH;
  const int own0 = ot * OWN;
  const int b = bh / p.H, h = bh % p.H;
  auto base = [&](const BwSide& x) { return x.p + b * x.sb + h * x.sh; };
  const float* u1 = base(DKV ? p.k : p.q);
  const float* u2 = base(DKV ? p.v : p.go);
  const float* y1 = base(DKV ? p.q : p.k);
  const float* y2 = base(DKV ? p.go : p.v);
  const int64_t u1t = DKV ? p.k.st : p.q.st, u2t = DKV ? p.v.st : p.go.st;
  const int64_t y1t = DKV ? p.q.st : p.k.st, y2t = DKV ? p.go.st : p.v.st;
  float* lse = p.lse + (int64_t)bh * p.Tq;
  float* delta = p.delta + (int64_t)bh * p.Tq;
  const float c2 = p.scale * 1.4426950408889634f;

  // stream tiles with a visible pair
  const int t_end = DKV ? (p.Tq + kBwRows - 1) / kBwRows
                        : ((p.causal ? min(p.Tk, own0 + OWN) : p.Tk) + kBwRows - 1) / kBwRows;
  const int t_begin = DKV && p.causal ? own0 / kBwRows : 0;

  bw8 o1h[KG][DS], o1l[KG][DS], o2h[KG][DS], o2l[KG][DS];
  int lo[KG], lim[KG];             // stream rows lo .. lo + lim - 1 are visible to the lane's own row
  // queries: the row's statistics; while they are formed, the lane's running
  // maximum, sum of P and sum of P dP over the stream rows it has seen
  float own_lse[KG], own_del[KG], own_sum[KG];
#pragma unroll
  for (int gi = 0; gi < KG; ++gi) {
    const int row = own0 + 16 * (KG * grp + gi) + l16;
    const int rc = min(row, own_T - 1);
#pragma unroll
    for (int d = 0; d < DS; ++d) {
      bw_split8(u1 + rc * u1t + 32 * d + 8 * g, o1h[gi][d], o1l[gi][d]);
      bw_split8(u2 + rc * u2t + 32 * d + 8 * g, o2h[gi][d], o2l[gi][d]);
    }
    lo[gi] = DKV && p.causal ? row : 0;
    lim[gi] = DKV ? max(p.Tq - lo[gi], 0) : (p.causal ? min(row + 1, p.Tk) : p.Tk);
    own_lse[gi] = KIND == kBwQ ? lse[rc] : -INFINITY;
    own_del[gi] = KIND == kBwQ ? delta[rc] : 0.f;
    own_sum[gi] = 0.f;
  }
  bwf4 acc[NA ? NA : 1][KG][DT];  // [dK or dQ, dV]
#pragma unroll
  for (int a = 0; a < NA; ++a)
#pragma unroll
    for (int gi = 0; gi < KG; ++gi)
#pragma unroll
      for (int u = 0; u < DT; ++u) acc[a][gi][u] = bwf4{0.f, 0.f, 0.f, 0.f};

  BwTile<D> x;
  float rv = 0.f;
  auto fetch = [&](int it) {
    x.load(y1, y1t, y2, y2t, it * kBwRows, str_T, tid);
    if (DKV && tid < 128) rv = (tid < 64 ? lse : delta)[min(it * kBwRows + (tid & 63), p.Tq - 1)];
  };
  if (t_begin < t_end) fetch(t_begin);
  for (int it = t_begin; it < t_end; ++it) {
    __syncthreads();  // the previous tile's reads are done
    x.template store<NA>(s, tid);
    if (DKV && tid < 128) rowv[tid >> 6][tid & 63] = rv;
    __syncthreads();
    fetch(min(it + 1, t_end - 1));

    const int r0 = 32 * half;
    bw8 ph[KG], pl[KG], dh[KG], dl[KG];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      bwf4 sc[KG], dp[KG];
#pragma unroll
      for (int gi = 0; gi < KG; ++gi) sc[gi] = dp[gi] = bwf4{0.f, 0.f, 0.f, 0.f};
      const int row = r0 + 16 * t + l16;
#pragma unroll
      for (int d = 0; d < DS; ++d) {
        const bf16_t* f = s + row * D + ((4 * d + g) ^ bw_swz<D>(row)) * 8;
        const bw8 a1h = *(const bw8*)f, a1l = *(const bw8*)(f + ARR);
        const bw8 a2h = *(const bw8*)(f + 2 * ARR), a2l = *(const bw8*)(f + 3 * ARR);
#pragma unroll
        for (int gi = 0; gi < KG; ++gi) {
          sc[gi] = bw_mfma3(a1h, a1l, o1h[gi][d], o1l[gi][d], sc[gi]);
          dp[gi] = bw_mfma3(a2h, a2l, o2h[gi][d], o2l[gi][d], dp[gi]);
        }
      }
      const int rr = r0 + 16 * t + 4 * g;  // the lane's first stream row in the tile
      float ls[4], de[4];
      if constexpr (DKV) {
        *(float4*)ls = *(const float4*)&rowv[0][rr];
        *(float4*)de = *(const float4*)&rowv[1][rr];
      }
#pragma unroll
      for (int gi = 0; gi < KG; ++gi) {
        if constexpr (STATS) {
          float v[4], mx = own_lse[gi];
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            v[r] = (unsigned)(it * kBwRows + rr + r) < (unsigned)lim[gi] ? sc[gi][r] * c2 : -INFINITY;
            mx = fmaxf(mx, v[r]);
          }
          const float mu = mx == -INFINITY ? 0.f : mx;
          const float alpha = __builtin_amdgcn_exp2f(own_lse[gi] - mu);
          own_lse[gi] = mx;
          own_sum[gi] *= alpha;
          own_del[gi] *= alpha;
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float e = __builtin_amdgcn_exp2f(v[r] - mu);
            own_sum[gi] += e;
            own_del[gi] += v[r] == -INFINITY ? 0.f : e * dp[gi][r];
          }
          continue;
        }
        float pv[4], dv[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const bool vis = (unsigned)(it * kBwRows + rr + r - lo[gi]) < (unsigned)lim[gi];
          const float e = __builtin_amdgcn_exp2f(fmaf(sc[gi][r], c2, -(DKV ? ls[r] : own_lse[gi])));
          pv[r] = vis ? e : 0.f;
          dv[r] = vis ? e * (dp[gi][r] - (DKV ? de[r] : own_del[gi])) : 0.f;
        }
#pragma unroll
        for (int r = 0; r < 4; r += 2) {
          bf16x2_t hh, ll;
          if constexpr (DKV) {
            split_bf16x2(pv[r], pv[r + 1], hh, ll);
            ph[gi][4 * t + r] = hh.x; ph[gi][4 * t + r + 1] = hh.y;
            pl[gi][4 * t + r] = ll.x; pl[gi][4 * t + r + 1] = ll.y;
          }
          split_bf16x2(dv[r], dv[r + 1], hh, ll);
          dh[gi][4 * t + r] = hh.x; dh[gi][4 * t + r + 1] = hh.y;
          dl[gi][4 * t + r] = ll.x; dl[gi][4 * t + r + 1] = ll.y;
        }
      }
    }
    if constexpr (STATS) continue;
#pragma unroll
    for (int u = 0; u < DT; ++u) {
      const int d = 16 * u + l16;
      const bf16_t* f = s + 4 * ARR + d * kBwRows + ((4 * half + g) ^ bw_swz_t(d)) * 8;
      const bw8 a1h = *(const bw8*)f, a1l = *(const bw8*)(f + ARR);
#pragma unroll
      for (int gi = 0; gi < KG; ++gi) acc[0][gi][u] = bw_mfma3(a1h, a1l, dh[gi], dl[gi], acc[0][gi][u]);
      if constexpr (DKV) {
        const bw8 a2h = *(const bw8*)(f + 2 * ARR), a2l = *(const bw8*)(f + 3 * ARR);
#pragma unroll
        for (int gi = 0; gi < KG; ++gi) acc[NA - 1][gi][u] = bw_mfma3(a2h, a2l, ph[gi], pl[gi], acc[NA - 1][gi][u]);
      }
    }
  }

  // the second half's sums through LDS to the first half's wavefronts
  __syncthreads();
  if constexpr (STATS) {
    // first over the four lanes of an own row, then over the halves
    float* red = (float*)s + grp * (KG * 3 * 16) + l16;
#pragma unroll
    for (int gi = 0; gi < KG; ++gi) {
#pragma unroll
      for (int m = 16; m <= 32; m <<= 1) bw_merge(own_lse[gi], own_sum[gi], own_del[gi], __shfl_xor(own_lse[gi], m, 64),
                                                  __shfl_xor(own_sum[gi], m, 64), __shfl_xor(own_del[gi], m, 64));
      if (half == 1 && g == 0) {
        red[(gi * 3) * 16] = own_lse[gi];
        red[(gi * 3 + 1) * 16] = own_sum[gi];
        red[(gi * 3 + 2) * 16] = own_del[gi];
      }
    }
    __syncthreads();
    if (half == 1 || g != 0) return;
#pragma unroll
    for (int gi = 0; gi < KG; ++gi) {
      bw_merge(own_lse[gi], own_sum[gi], own_del[gi], red[(gi * 3) * 16], red[(gi * 3 + 1) * 16],
               red[(gi * 3 + 2) * 16]);
      const int row = own0 + 16 * (KG * grp + gi) + l16;
      if (row < own_T) {
        lse[row] = own_lse[gi] + log2f(own_sum[gi]);
        delta[row] = own_del[gi] / own_sum[gi];
      }
    }
    return;
  }
  float* red = (float*)s + grp * (NA * KG * DT * 4 * 64) + lane;
  if (half == 1) {
#pragma unroll
    for (int a = 0; a < NA; ++a)
#pragma unroll
      for (int gi = 0; gi < KG; ++gi)
#pragma unroll
        for (int u = 0; u < DT; ++u)
#pragma unroll
          for (int r = 0; r < 4; ++r) red[(((a * KG + gi) * DT + u) * 4 + r) * 64] = acc[a][gi][u][r];
  }
  __syncthreads();
  if (half == 1) return;
#pragma unroll
  for (int a = 0; a < NA; ++a) {
    float* out = (a ? p.dv : DKV ? p.dk : p.dq) + (int64_t)bh * own_T * D;
    const float sc = a ? 1.f : p.scale;
#pragma unroll
    for (int gi = 0; gi < KG; ++gi) {
      const int row = own0 + 16 * (KG * grp + gi) + l16;
#pragma unroll
      for (int u = 0; u < DT; ++u) {
        float o[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) o[r] = (acc[a][gi][u][r] + red[(((a * KG + gi) * DT + u) * 4 + r) * 64]) * sc;
        if (row < own_T) *(float4*)(out + (int64_t)row * D + 16 * u + 4 * g) = make_float4(o[0], o[1], o[2], o[3]);
      }
    }
  }
}

template <int D>
__global__ void __launch_bounds__(256, D == 128 ? 1 : 2) attention_bwd_kernel(BwArgs p) {
  __shared__ __attribute__((aligned(16))) bf16_t s[8 * kBwRows * D];
  __shared__ __attribute__((aligned(16))) float rowv[2][kBwRows];
  if ((int)blockIdx.x < p.kv_blocks) bw_block<D, kBwKV>(p, blockIdx.x, s, rowv);
  else bw_block<D, kBwQ>(p, blockIdx.x - p.kv_blocks, s, rowv);
}

template <int D>
__global__ void __launch_bounds__(256, D == 128 ? 1 : 2) attention_bwd_stats_kernel(BwArgs p) {
  __shared__ __attribute__((aligned(16))) bf16_t s[4 * kBwRows * D];
  bw_block<D, kBwStats>(p, blockIdx.x, s, nullptr);
}

bool bw_rows_ok(const void* p, int64_t sb, int64_t sh, int64_t st) {
  return (uintptr_t)p % 16 == 0 && sb % 4 == 0 && sh % 4 == 0 && st % 4 == 0;
}

}  // namespace

bool attention_backward_rows_ok(const void* p, int64_t sb, int64_t sh, int64_t st) { return bw_rows_ok(p, sb, sh, st); }

bool attention_backward_ok(int64_t B, int64_t H, int64_t Tq, int64_t Tk, int64_t D) {
  const int64_t tiles = (Tq + 31) / 32 + (Tk + 31) / 32;
  return (D == 32 || D == 64 || D == 128) && Tq > 0 && Tk > 0 && B > 0 && H > 0 && Tq < (1 << 28) && Tk < (1 << 28) &&
         B * H < (1 << 28) && B * H * tiles < 0x7fffffffLL;
}

// A block walks the other side's rows one tile after the other, so with few
// heads and a long side most CUs idle for the whole walk, where the
// composition's products spread over the chip.  Both times, in us, from what
// was measured at 1 to 48 heads, 16 to 4096 rows a side, MI355X (fused /
// composed; not causal):
//   heads x Tq x Tk   1 x 2048 x 2048   16 x 1024 x 1024   1 x 16 x 2048
//   D = 32            93 / 130          67 / 251           79 / 91
//   D = 64            168 / 139         107 / 267          117 / 90
//   D = 128           214 / 151         297 / 329          164 / 71
// The walk's time a 64-row tile (statistics; dQ; dK and dV) or, with more
// blocks than CUs, the blocks' shares of it.  The composition: its launches
// and its passes over [Tq, Tk], half as fast where rows of Tk floats are not
// 16-byte aligned.  Of 954 measured shapes the fused kernels lost more than 5%
// at 150 (3.8 times at worst), the choice by these times at 18 (1.4 times).
bool attention_backward_pays(int64_t B, int64_t H, int64_t Tq, int64_t Tk, int64_t D, bool causal) {
  constexpr float kCus = 256.f;
  const int i = D == 32 ? 0 : D == 64 ? 1 : 2;
  const float t_stats = std::array{0.95f, 1.45f, 2.2f}[i], t_q = std::array{1.35f, 2.1f, 2.9f}[i];
  const float t_kv = std::array{1.9f, 3.6f, 4.4f}[i], t_elem = std::array{12.f, 12.5f, 15.f}[i] * 1e-6f;
  const int64_t own = D == 128 ? 32 : 64;
  const float bh = (float)(B * H), q_blocks = bh * (float)((Tq + own - 1) / own);
  const float kv_blocks = bh * (float)((Tk + own - 1) / own);
  const float q_walk = (float)(((causal ? std::min(Tq, Tk) : Tk) + 63) / 64), kv_walk = (float)((Tq + 63) / 64);
  const float seen = causal ? 0.5f : 1.f;
  const float stats = q_walk * t_stats * std::max(1.f, seen * q_blocks / kCus);
  const float grads = std::max({kv_walk * t_kv, q_walk * t_q,
                                seen * (kv_blocks * kv_walk * t_kv + q_blocks * q_walk * t_q) / kCus});
  const float composed = 85.f + t_elem * (Tk % 4 != 0 ? 2.f : 1.f) * bh * (float)Tq * (float)Tk;
  return 12.f + stats + grads <= composed;
}

void attention_backward(const AttnBwd& a, hipStream_t s) {
  if (!attention_backward_ok(a.B, a.H, a.Tq, a.Tk, a.D)) fail("attention_backward: shape not supported");
  auto side = [](const AttnBwd::Rows& r) { return BwSide{(const float*)r.p, r.sb, r.sh, r.st}; };
  for (const AttnBwd::Rows* r : {&a.q, &a.k, &a.v, &a.go})
    if (!bw_rows_ok(r->p, r->sb, r->sh, r->st)) fail("attention_backward: rows must be 16-byte aligned");
  BwArgs p{};
  p.q = side(a.q); p.k = side(a.k); p.v = side(a.v); p.go = side(a.go);
  p.lse = (float*)a.stats;
  p.delta = p.lse + a.B * a.H * a.Tq;
  p.dq = (float*)a.dq; p.dk = (float*)a.dk; p.dv = (float*)a.dv;
  p.BH = (int)(a.B * a.H); p.H = (int)a.H; p.Tq = (int)a.Tq; p.Tk = (int)a.Tk;
  p.scale = a.scale;
  p.causal = a.causal ? 1 : 0;
  auto go = [&](auto dim) {
    constexpr int D = decltype(dim)::value;
    constexpr int OWN = kBwOwn<D>;
    p.kv_blocks = a.dk ? (int)(p.BH * ((a.Tk + OWN - 1) / OWN)) : 0;
    const int q_tiles = (int)(p.BH * ((a.Tq + OWN - 1) / OWN)), q_blocks = a.dq ? q_tiles : 0;
    if (p.kv_blocks + q_blocks == 0) return;
    hipLaunchKernelGGL((attention_bwd_stats_kernel<D>), dim3((unsigned)q_tiles), dim3(256), 0, s, p);
    hipLaunchKernelGGL((attention_bwd_kernel<D>), dim3((unsigned)(p.kv_blocks + q_blocks)), dim3(256), 0, s, p);
  };
  if (a.D == 32) go(std::integral_constant<int, 32>{});
  else if (a.D == 64) go(std::integral_constant<int, 64>{});
  else go(std::integral_constant<int, 128>{});
  check_launch("attention_backward");
}

}  // namespace k
}  // namespace agpu
