// Large fp16 / bf16 GEMMs, both operands contiguous along k: C[M, N] =
// epilogue(A[M, K] B[K, N]) with B given as W [N][K] (torch Linear weights,
// GPT-2's k-major projection weights, the tied LM head).  Same arithmetic as
// the tiled GEMMs (fp32 accumulation over k; the reference's matmul/linear,
// crates/core/src/kernel_templates.rs:987-1072).
//
// One block owns a BM x BN tile over the whole K, in stages of 64 k:
//  - Global -> LDS with buffer loads to LDS of 16 bytes a lane: each wave
//    instruction copies one 1 KB window of 8 rows x 64 k with no register
//    staging.  Lane p of the instruction reads row p / 8 of the window, whose
//    128 bytes are one contiguous read; the row's 16-byte chunks land
//    exchanged (chunk ^ (row / 2) % 8), so that the 16 lanes of a fragment
//    read's phase (16 rows at one chunk) cover all 64 banks.
//  - Two stages in LDS.  A wavefront's fragments of the next 16 k are read
//    while the MFMAs of the current 16 run, across the stage boundary too:
//    the barrier stands before a stage's last 16 k, when every wavefront has
//    all of that stage in registers, so the copies of the stage after next
//    start there and have a stage of MFMAs to land.
//  - WM x WN wavefronts, each TM x TN tiles of 32 x 32 (v_mfma_f32_32x32x16,
//    W as the MFMA's A side: a lane's accumulators are 4 consecutive columns
//    of one output row).
//  - The epilogue goes through LDS, so that bias, residual and C move as 16
//    bytes a lane, whole 128-byte runs of a row, at any alignment (the
//    50257-column head's rows start at odd addresses).
#include "gemm_kernels.hpp"

namespace agpu {
namespace k {
using namespace dev;

namespace {

typedef __attribute__((address_space(3))) void* lds_ptr;

// 16 bytes a lane from base + voff (per lane) + soff to LDS, lane by lane;
// past the resource's end they are zeros.  The buffer form: it counts as a
// vector memory access alone, where global_load_lds also counts as an LDS
// access of unknown order, after which the compiler waited for every
// fragment read before the first MFMA.
__device__ __forceinline__ void lds_copy16(__amdgpu_buffer_rsrc_t src, void* l, int voff, int soff) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(src, (lds_ptr)l, 16, voff, soff, 0, 0);
}
// An offset that is past the end of every resource: what is copied from there
// is zeros.  A resource spans no more than this, however far its tensor
// reaches (a tile's own rows end before half of it, see gemm_h16_ok).
constexpr int kPastEnd = 0x7ffffff0;
// The rows of an operand from `p` on, `bytes` of them.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rows_resource(const void* p, int64_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)(bytes < kPastEnd ? bytes : kPastEnd),
                                           0x00020000);
}

template <typename T> struct Mfma32h;
template <> struct Mfma32h<half_t> {
  typedef f16x8 vec;
  static __device__ __forceinline__ f32x16 run(vec a, vec b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
  }
};
template <> struct Mfma32h<bf16_t> {
  typedef bf16x8 vec;
  static __device__ __forceinline__ f32x16 run(vec a, vec b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
};

template <int ACT>
__device__ __forceinline__ float h16_act(float v) {
  if constexpr (ACT == kActRelu) return fmaxf(v, 0.f);
  else if constexpr (ACT == kActGelu) return gelu_tanh(v);
  else if constexpr (ACT == kActGeluExact) return 0.5f * v * (1.f + erff(v * 0.70710678118654752f));
  else return v;
}

template <typename T, int TM, int TN, int WM, int WN, int ACT>
__global__ void __launch_bounds__(64 * WM * WN, WM * WN <= 4 ? 1 : WM * WN / 4) gemm_h16_kernel(GArgs p) {
  constexpr int NW = WM * WN, BM = 32 * TM * WM, BN = 32 * TN * WN;
  constexpr int BK = 64;                                  // k per stage
  constexpr int CH = BK / 8, WR = 64 / CH, KK = BK / 16;  // chunks per row, rows per 1 KB window, MFMA steps per stage
  constexpr int AW = BM / WR, BW = BN / WR;               // windows per stage
  constexpr int STAGE = (AW + BW) * 512;   // elements
  constexpr int LA = AW / NW, LB = BW / NW, LPW = LA + LB;  // window copies per wavefront per stage
  static_assert(AW % NW == 0 && BW % NW == 0, "tile shape");
  typedef typename Mfma32h<T>::vec V8;
  __shared__ __attribute__((aligned(16))) T lds[2 * STAGE];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int tmi, tni;
  tile_coords(p, tmi, tni);
  const int64_t m0 = (int64_t)tmi * BM, n0 = (int64_t)tni * BN;
  const int nk = (int)((p.K + BK - 1) / BK);
  // chunk c of row r sits at chunk c ^ swz(r)
  auto swz = [](int r) { return (r * CH / 16) & (CH - 1); };

  // This wavefront's windows: LA consecutive ones of A's rows, LB of W's.
  // Rows past M or N read zeros.
  const __amdgpu_buffer_rsrc_t sa =
      rows_resource((const T*)p.A + m0 * p.a_sm, ((p.M - m0 - 1) * p.a_sm + p.K) * (int64_t)sizeof(T));
  const __amdgpu_buffer_rsrc_t sb =
      rows_resource((const T*)p.B + n0 * p.b_sn, ((p.N - n0 - 1) * p.b_sn + p.K) * (int64_t)sizeof(T));
  const int lr = lane / CH;
  int off[LPW];
#pragma unroll
  for (int q = 0; q < LPW; ++q) {
    const int r = (q < LA ? w * LA + q : w * LB + q - LA) * WR + lr;
    off[q] = (int)((r * (q < LA ? p.a_sm : p.b_sn) + ((lane % CH) ^ swz(r)) * 8) * (int64_t)sizeof(T));
  }
  auto issue = [&](int st) __attribute__((always_inline)) {
    T* da = lds + (st % 2) * STAGE + w * LA * 512;
    T* db = lds + (st % 2) * STAGE + (AW + w * LB) * 512;
    const int k = st * (BK * (int)sizeof(T));
    const bool ends = (st + 1) * BK > (int)p.K;
    if (ends) {
      // the last, partial stage (K is a multiple of 8): chunks past K read
      // past the resource's end
      const int left = ((int)p.K - st * BK) / 8;
#pragma unroll
      for (int q = 0; q < LPW; ++q) {
        const int r = (q < LA ? w * LA + q : w * LB + q - LA) * WR + lr;
        const int v = ((lane % CH) ^ swz(r)) < left ? off[q] + k : kPastEnd;
        lds_copy16(q < LA ? sa : sb, q < LA ? da + q * 512 : db + (q - LA) * 512, v, 0);
      }
      return;
    }
#pragma unroll
    for (int q = 0; q < LA; ++q) lds_copy16(sa, da + q * 512, off[q], k);
#pragma unroll
    for (int q = 0; q < LB; ++q) lds_copy16(sb, db + q * 512, off[LA + q], k);
  };

  const int wm = w / WN, wn = w % WN, l31 = lane & 31, hi = lane >> 5;
  // fragment addresses: row r of the operand's part of a stage, chunk c
  auto foff = [&](int r, int c) { return r * BK + ((c ^ swz(r)) * 8); };
  V8 fa[2][TM], fb[2][TN];
  auto read = [&](int set, int st, int kk) __attribute__((always_inline)) {
    const T* a = lds + (st % 2) * STAGE;
    const T* b = a + AW * 512;
#pragma unroll
    for (int j = 0; j < TN; ++j) fb[set][j] = *(const V8*)(b + foff((wn * TN + j) * 32 + l31, 2 * kk + hi));
#pragma unroll
    for (int i = 0; i < TM; ++i) fa[set][i] = *(const V8*)(a + foff((wm * TM + i) * 32 + l31, 2 * kk + hi));
  };
  f32x16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
  auto mul = [&](int set) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = Mfma32h<T>::run(fb[set][j], fa[set][i], acc[i][j]);
  };

  constexpr int kCopies = 0x0f70, kCopiesAndReads = 0x0070;  // waits for this wavefront's copies, and its LDS reads
  issue(0);
  __builtin_amdgcn_s_waitcnt(kCopies);
  __syncthreads();
  if (nk > 1) issue(1);
  read(0, 0, 0);
  for (int st = 0; st < nk; ++st) {
    // the fragments read before the last MFMAs are there by now; without this
    // the compiler, which joins two loop entries here, waits for the next
    // ones too
    __builtin_amdgcn_s_waitcnt(0xc07f);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int kk = 0; kk + 1 < KK; ++kk) {
      read((kk + 1) & 1, st, kk + 1);
      __builtin_amdgcn_sched_barrier(0);
      mul(kk & 1);
      __builtin_amdgcn_sched_barrier(0);
    }
    // this wavefront holds the rest of stage st in registers, and its copies
    // of stage st + 1 have landed; after the barrier so for every wavefront
    __builtin_amdgcn_s_waitcnt(kCopiesAndReads);
    __syncthreads();
    __builtin_amdgcn_sched_barrier(0);
    if (st + 2 < nk) issue(st + 2);
    if (st + 1 < nk) read(0, st + 1, 0);
    __builtin_amdgcn_sched_barrier(0);
    mul((KK - 1) & 1);
  }
  __syncthreads();

  // C^T layout of each 32 x 32 tile: lane l, register e -> row l % 32,
  // column 8 (e / 4) + 4 (l / 32) + e % 4.  Through this wavefront's own part
  // of LDS, 32 rows x 32 TN columns of fp32 at a time, rows 4 floats apart.
  constexpr int CN = 32 * TN, CP = CN + 4;
  constexpr int LPR = CN / 8, RPI = 64 / LPR;  // lanes per row, rows per instruction
  static_assert(NW * 32 * CP * 4 <= 2 * STAGE * (int)sizeof(T), "epilogue staging");
  float* ct = (float*)lds + w * 32 * CP;
  const T* bias = (const T*)p.bias;
  const T* R = (const T*)p.res;
  T* C = (T*)p.C;
  struct V { T e[8]; };
  const int64_t col = n0 + wn * CN + (lane % LPR) * 8;
  const bool full = col + 8 <= p.N;
  float bs[8] = {};
  if (bias) {
    if (full) {
      V b;
      __builtin_memcpy(&b, bias + col, 16);
#pragma unroll
      for (int e = 0; e < 8; ++e) bs[e] = to_f(b.e[e]);
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) bs[e] = col + e < p.N ? to_f(bias[col + e]) : 0.f;
    }
  }
#pragma unroll
  for (int i = 0; i < TM; ++i) {
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *(float4*)(ct + l31 * CP + 32 * j + 8 * g + 4 * hi) =
            make_float4(acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]);
    // the wavefront's own writes and reads: in order, no barrier.  A rolled
    // loop: unrolled, the epilogue's instructions come from memory once per
    // launch and compute unit and took 15 us
#pragma unroll 1
    for (int it = 0; it < 32 / RPI; ++it) {
      const int r = it * RPI + lane / LPR;
      const int64_t row = m0 + (wm * TM + i) * 32 + r;
      float v[8];
      *(float4*)v = *(const float4*)(ct + r * CP + (lane % LPR) * 8);
      *(float4*)(v + 4) = *(const float4*)(ct + r * CP + (lane % LPR) * 8 + 4);
      if (row >= p.M) continue;
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = h16_act<ACT>(p.alpha * v[e] + bs[e]);
      T* out = C + row * p.c_sm + col;
      const T* res = R + row * p.r_sm + col;
      V o;
      if (full) {
        if (R) {
          V x;
          __builtin_memcpy(&x, res, 16);
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] += to_f(x.e[e]);
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) o.e[e] = from_f<T>(v[e]);
        __builtin_memcpy(out, &o, 16);
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (col + e < p.N) out[e] = from_f<T>(v[e] + (R ? to_f(res[e]) : 0.f));
      }
    }
  }
}

bool al16(const void* q) { return ((uintptr_t)q & 15) == 0; }

// The tile for a product: the least time by a model of what was measured on
// MI355X (us; `fixed` = launch, first copies and epilogue, `step[j]` = one 64
// k stage with j + 1 blocks on a compute unit):
//   256 x 256, 8 wavefronts of 128 x 64, one block a CU
//   128 x 128, 4 of 64 x 64, two blocks a CU
//   128 x 64, 4 of 32 x 64, three blocks a CU
// Of the last round the first two wait for most of a whole one, three blocks a
// CU fill each other's gaps.  fp16, us, alone with weights rotating beyond the
// Infinity Cache (in a prefill of 4 x 500 tokens):
//   M x N x K             256 x 256    128 x 128    128 x 64
//   2000 x 3840 x 1280    37 (39)      28 (31)      34 (42)
//   2000 x 5120 x 1280    38 (44)      41 (55)      37 (47)    (with gelu)
//   2000 x 1280 x 1280    32 (43)      18 (24)      16 (22)
//   2000 x 1280 x 5120    101 (123)    54 (70)      46 (65)
//   2000 x 50257 x 1280   333 (318)    350 (335)    409 (390)
//   4096 x 3840 x 1280    45.5         51           59
// against 36, 61, 22, 69 and about 500 in the prefill for the register-staged
// tiles (gemm_mf).
struct H16Tile {
  int bm, bn, per_cu;
  float fixed, act, step[3];
};
constexpr H16Tile kH16Tiles[3] = {
    {256, 256, 1, 8.6f, 2.5f, {1.6f, 0.f, 0.f}},
    {128, 128, 2, 5.8f, 1.f, {0.62f, 1.08f, 0.f}},
    {128, 64, 3, 5.0f, 0.5f, {0.50f, 0.60f, 0.97f}},
};

int64_t h16_tiles(const Gemm& g, const H16Tile& t) {
  return ((g.M + t.bm - 1) / t.bm) * ((g.N + t.bn - 1) / t.bn);
}

float h16_time(const Gemm& g, const H16Tile& t, int cus) {
  const int64_t tiles = h16_tiles(g, t), slots = (int64_t)cus * t.per_cu;
  const float stages = (float)((g.K + 63) / 64), once = t.fixed + (g.act ? t.act : 0.f);
  if (tiles <= slots) {
    // between the steps with j and j + 1 blocks a CU: the CUs with fewer run ahead
    const int j = (int)((tiles + cus - 1) / cus);
    const float part = (float)tiles / (float)cus - (float)(j - 1), lower = t.step[j > 1 ? j - 2 : 0];
    return once + (lower + part * (t.step[j - 1] - lower)) * stages;
  }
  const float whole = (float)((tiles + slots - 1) / slots), share = (float)tiles / (float)slots;
  const float rounds = t.per_cu < 3 ? 0.75f * whole + 0.25f * share : 0.25f * whole + 0.75f * share;
  return rounds * (once + t.step[t.per_cu - 1] * stages);
}

int h16_pick(const Gemm& g, int cus) {
  int best = 0;
  for (int i = 1; i < 3; ++i)
    if (h16_time(g, kH16Tiles[i], cus) < h16_time(g, kH16Tiles[best], cus)) best = i;
  return best;
}

template <typename T, int TM, int TN, int WM, int WN>
void h16_launch(const GArgs& p, hipStream_t s) {
  const dim3 grid((unsigned)(p.tiles_m * p.tiles_n)), block(64 * WM * WN);
#define AGPU_H16(ACT) hipLaunchKernelGGL((gemm_h16_kernel<T, TM, TN, WM, WN, ACT>), grid, block, 0, s, p)
  switch (p.act) {
    case kActNone: AGPU_H16(kActNone); break;
    case kActRelu: AGPU_H16(kActRelu); break;
    case kActGelu: AGPU_H16(kActGelu); break;
    default: AGPU_H16(kActGeluExact);
  }
#undef AGPU_H16
}

template <typename T>
void h16_tile_launch(int tile, const GArgs& p, hipStream_t s) {
  if (tile == 0) h16_launch<T, 4, 2, 2, 4>(p, s);
  else if (tile == 1) h16_launch<T, 2, 2, 2, 2>(p, s);
  else h16_launch<T, 1, 2, 4, 1>(p, s);
}

}  // namespace

// Products with enough 128 x 64 tiles: fewer are left to gemm_mf, whose 64 x 64
// tiles fill the chip or split K (777 x 1280 x 1280, 140 tiles: 17.8 us here,
// 16.9 there; 200 x 248 x 4696, 148 tiles: 7.7 here, 10.9 there).  Where it
// splits K (few rows: fewer than a 64 x 64 tile a CU) it reads twice as fast, but
// pays for the partial sums of every output: it wins from a k that grows with
// their number (us here / there, weights not in cache; M x N x K: 64 x 10240 x 1280
// 19.4 / 17.9, x 8192 99 / 51; 17 x 8192 x 768 12.4 / 9.5; 17 x 10240 x 8192 100 /
// 45; 192 x 5120 x 1280 19 / 21, x 3072 40 / 25; with the weights in cache the two
// meet at half as many k more).
bool gemm_h16_ok(const Gemm& g, int cus) {
  const bool is16 = g.dt == DType::F16 || g.dt == DType::BF16;
  if (!(is16 && g.b_dt == g.dt && g.batch == 1 && !g.b_scale && !g.b_x3 && !g.a_x3 && !g.b_packed && !g.ln_gamma &&
        !g.mask && !g.pln_y && !g.pln_ypk && !g.c_pk && !g.no_reduce && g.K >= 64 && g.K % 8 == 0 && g.a_sk == 1 &&
        g.b_sk == 1 && g.a_sm % 8 == 0 && g.b_sn % 8 == 0 && al16(g.A) && al16(g.B)))
    return false;
  // a tile's rows lie within the 2 GiB that a buffer resource spans
  if (g.a_sm < g.K || g.b_sn < g.K || g.a_sm >= (1 << 21) || g.b_sn >= (1 << 21)) return false;
  const bool mf_splits = (g.M + 63) / 64 * ((g.N + 63) / 64) < cus;
  if (mf_splits && g.K > 600 + g.M * g.N / 1000) return false;
  const int64_t tiles = h16_tiles(g, kH16Tiles[2]);
  return tiles >= (g.K <= 1024 ? cus / 2 : cus * 5 / 8) && tiles < (1LL << 31);
}

void gemm_h16(const Gemm& g, const GArgs& p_in, int cus, hipStream_t s) {
  if (!gemm_h16_ok(g, cus)) fail("gemm: the 16-bit large-tile plan does not fit this product");
  GArgs p = p_in;
  const int tile = h16_pick(g, cus);
  p.tiles_m = (int)((g.M + kH16Tiles[tile].bm - 1) / kH16Tiles[tile].bm);
  p.tiles_n = (int)((g.N + kH16Tiles[tile].bn - 1) / kH16Tiles[tile].bn);
  if (g.dt == DType::F16) h16_tile_launch<half_t>(tile, p, s);
  else h16_tile_launch<bf16_t>(tile, p, s);
  check_launch("gemm_h16");
}

const char* gemm_h16_name(const Gemm& g, int cus) {
  static const char* names[3] = {"lds16 256x256", "lds16 128x128", "lds16 128x64"};
  return names[h16_pick(g, cus)];
}

}  // namespace k
}  // namespace agpu
