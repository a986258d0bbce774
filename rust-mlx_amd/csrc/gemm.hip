// Affine-quantised GEMM on the gfx950 matrix cores for 17..kQmmMaxRows
// activation rows (prefill chunks), called by qmm().
//
// Replaces the same reference interfaces as qmm.hip (Linear::forward_rows,
// src/weights.rs:111-202) beyond 16 rows.  The weights are dequantised in
// registers as w = s q + b in fp32 and split into two bf16 parts, hi = bf16(w)
// and lo = bf16(w - hi) (w - hi is exact in fp32; hi + lo is w to within
// 2^-17 |w|), and the matrix cores multiply x hi + x lo into fp32 accumulators
// over the whole depth, with no scale work per output and group (exact-code
// products with the scales applied to the sums issue half the MFMAs but as
// many vector instructions: 124 us against 91 us at 512 x 12352 x 2048 in one
// and the same 128-row form).
//
// Two forms (gemm_plan chooses by an estimate of their times):
//  gemm_tile_kernel  a workgroup computes 64 weight rows x 32 UW activation
//    rows from LDS, one group at a time.
//  gemm_deep_kernel  few output tiles: every wave of a workgroup takes the
//    same outputs over its own range of k, reads its activations directly
//    (each wave needs other columns of them) and the sums are added in wave
//    order in LDS.  No workspace and no second launch.
#include <utility>

#include "common.hpp"
#include "gemm_plan.hpp"
#include "kernels.hpp"
#include "qmm_core.hpp"

namespace mx {

namespace {

typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
// a native vector: arrays of HIP's uint4 that live across a barrier were left
// in scratch memory
typedef uint32_t uint32x4_t __attribute__((ext_vector_type(4)));

// w = s q + b of eight codes as packed bf16 hi and lo parts.
__device__ __forceinline__ void split8(const float (&q)[8], float sc, float bi, uint4& hi,
                                       uint4& lo) {
  uint32_t h[4], l[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float v0 = fmaf_(sc, q[2 * i], bi), v1 = fmaf_(sc, q[2 * i + 1], bi);
    const bf16x2_t hv = {__bf16(v0), __bf16(v1)};
    h[i] = __builtin_bit_cast(uint32_t, hv);
    const bf16x2_t lv = {__bf16(v0 - u2f(h[i] << 16)), __bf16(v1 - u2f(h[i] & 0xffff0000u))};
    l[i] = __builtin_bit_cast(uint32_t, lv);
  }
  hi = make_uint4(h[0], h[1], h[2], h[3]);
  lo = make_uint4(l[0], l[1], l[2], l[3]);
}

// Eight nibbles of a word in order, as floats.
__device__ __forceinline__ void nibbles(uint32_t w, float (&q)[8]) {
  const uint32_t ev = w & 0x0f0f0f0fu, od = (w >> 4) & 0x0f0f0f0fu;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    q[2 * i] = float((ev >> (8 * i)) & 0xffu);
    q[2 * i + 1] = float((od >> (8 * i)) & 0xffu);
  }
}

// A quarter of a 64-value group of one weight row: 16 codes, scale and bias.
// The codes are kept as they come: 5-bit quarters start at bit 0 or 16 of
// their first word, and shifting them where they are loaded made every group
// wait for the loads that are in flight for a later one (128 x 12352 x 2048:
// 39.3 us against 35.7 before these tiles, now 34.6; up-mix of 32 rows to
// 8192 x 256: 9.8 us, now 8.8).
template <int BITS>
struct Quarter {
  uint32_t c[group_words<BITS>()];
  uint16_t s, b;
};

// Quarter dp of group g.
template <int BITS>
__device__ __forceinline__ void load_quarter(const TileRow& tr, int g, int dp, Quarter<BITS>& q) {
  if constexpr (BITS == 5) {
    const uint32_t* p = tr.codes + 10 * g + (80 * dp >> 5);
#pragma unroll
    for (int i = 0; i < 3; ++i) q.c[i] = p[i];
  } else {
    load_group_codes<BITS>(tr.codes, g, dp, q.c);
  }
  q.s = tr.scales[g];
  q.b = tr.biases[g];
}

// The codes 8 T .. + 7 of quarter dp as bf16 hi and lo parts.
template <int BITS, int T>
__device__ __forceinline__ void dequant_quarter(const Quarter<BITS>& p, int dp, uint4& hi,
                                                uint4& lo) {
  float q[8];
  if constexpr (BITS == 4) {
    nibbles(p.c[T], q);
  } else {
    uint32_t c[group_words<BITS>()];
#pragma unroll
    for (int i = 0; i < group_words<BITS>(); ++i) c[i] = p.c[i];
    if constexpr (BITS == 5) {
      const uint32_t sh = 16u * (dp & 1);
      c[0] = __builtin_amdgcn_alignbit(p.c[1], p.c[0], sh);
      c[1] = __builtin_amdgcn_alignbit(p.c[2], p.c[1], sh);
      c[2] = p.c[2] >> sh;
    }
    [&]<int... V>(std::integer_sequence<int, V...>) {
      ((q[V] = float(code_at<BITS, 8 * T + V>(c))), ...);
    }(std::make_integer_sequence<int, 8>{});
  }
  split8(q, bf16_to_f32(p.s), bf16_to_f32(p.b), hi, lo);
}

// Code v (0..31) of a 32-code piece held in BITS words, value v at bit BITS v.
template <int BITS, int V>
__device__ __forceinline__ uint32_t piece_code(const uint32_t (&w)[BITS]) {
  constexpr int bit = BITS * V, word = bit >> 5, off = bit & 31;
  constexpr uint32_t mask = (1u << BITS) - 1u;
  if constexpr (off + BITS <= 32)
    return (w[word] >> off) & mask;
  else
    return __builtin_amdgcn_alignbit(w[word + 1], w[word], uint32_t(off)) & mask;
}

// Lane quarter kq's piece of one 128-value stage of one weight row: 32 codes,
// scale and bias.
template <int BITS>
struct Piece {
  uint32_t c[BITS];
  uint16_t s, b;
};

// `half`: an odd last stage, of which only quarters 0 and 1 exist (the others
// read quarter kq - 2 and dequantise to zero).
template <int BITS>
__device__ __forceinline__ void load_piece(const TileRow& tr, int stage, int kq, bool half,
                                           Piece<BITS>& p) {
  const int q = half ? (kq & 1) : kq;
  const uint32_t* src = tr.codes + (4 * stage + q) * BITS;
  if constexpr (BITS % 4 == 0) {  // 16-byte aligned pieces
#pragma unroll
    for (int i = 0; i < BITS / 4; ++i) {
      const uint4 v = reinterpret_cast<const uint4*>(src)[i];
      p.c[4 * i] = v.x;
      p.c[4 * i + 1] = v.y;
      p.c[4 * i + 2] = v.z;
      p.c[4 * i + 3] = v.w;
    }
  } else {
#pragma unroll
    for (int i = 0; i < BITS; ++i) p.c[i] = src[i];
  }
  const int g = 2 * stage + (q >> 1);
  p.s = tr.scales[g];
  p.b = tr.biases[g];
  if (half && kq >= 2) p.s = p.b = 0;
}

// The piece's codes 8 ST .. + 7 as bf16 hi and lo parts.
template <int BITS, int ST>
__device__ __forceinline__ void dequant_step(const Piece<BITS>& p, uint4& hi, uint4& lo) {
  float q[8];
  if constexpr (BITS == 4)
    nibbles(p.c[ST], q);
  else
    [&]<int... V>(std::integer_sequence<int, V...>) {
      ((q[V] = float(piece_code<BITS, 8 * ST + V>(p.c))), ...);
    }(std::make_integer_sequence<int, 8>{});
  split8(q, bf16_to_f32(p.s), bf16_to_f32(p.b), hi, lo);
}

// The projection epilogues of N outputs of one weight row (activation rows
// m[i]; those from M on are not stored).  kHcWrite reads every stream of all N
// before it writes the first (written one by one, each read waited for the
// write before it: 256 x 2048 x 4096 in the deep form took 31.3 us, now 28.7).
template <int N>
__device__ __forceinline__ void gemm_epilogue(const ProjEpilogue& e, int n, int M,
                                              const int (&m)[N], int row, const float (&v)[N]) {
  if (e.mode == kPlain) {
#pragma unroll
    for (int i = 0; i < N; ++i)
      if (m[i] < M) e.y[size_t(m[i]) * e.y_stride + row] = f32_to_bf16(v[i]);
  } else if (e.mode == kHcDown) {
#pragma unroll
    for (int i = 0; i < N; ++i) {
      if (m[i] >= M) continue;
      const float tt = round_bf16(round_bf16(v[i]) / float(e.hc));
      if (row < e.rank)
        e.y[size_t(m[i]) * e.y_stride + row] = f32_to_bf16(tt * sigmoid_bf16(tt));
      else
        e.aux[size_t(m[i]) * e.aux_stride + (row - e.rank)] = f32_to_bf16(sigmoid_bf16(tt) * 2.0f);
    }
  } else {  // kHcWrite
    constexpr int kS = 4;  // streams at a time
    for (int s0 = 0; s0 < e.hc; s0 += kS) {
      uint16_t res[N][kS], gate[N][kS];
#pragma unroll
      for (int i = 0; i < N; ++i)
#pragma unroll
        for (int s = 0; s < kS; ++s)
          if (m[i] < M && s0 + s < e.hc) {
            res[i][s] = e.y[size_t(m[i]) * e.y_stride + size_t(s0 + s) * n + row];
            gate[i][s] = e.aux[size_t(m[i]) * e.aux_stride + s0 + s];
          }
#pragma unroll
      for (int i = 0; i < N; ++i)
#pragma unroll
        for (int s = 0; s < kS; ++s)
          if (m[i] < M && s0 + s < e.hc) {
            const float inj = round_bf16(round_bf16(v[i]) * bf16_to_f32(gate[i][s]));
            e.y[size_t(m[i]) * e.y_stride + size_t(s0 + s) * n + row] =
                f32_to_bf16(bf16_to_f32(res[i][s]) + inj);
          }
    }
  }
}

// ---------------------------------------------------------------------------
// Workgroup (blockIdx.x, blockIdx.y): weight rows 16 NT x .., activation rows
// 16 MT y ..; wave kp of KS takes its share of the 128-value stages.  Lane
// quarter kq of MFMA step st covers k = 32 kq + 8 st .. + 7 of a stage on both
// operands, so an operand of four steps is 64 contiguous bytes of an
// activation row and 4 BITS bytes of a weight row.  An odd number of groups
// leaves the last stage's quarters 2 and 3 empty: both operands are zero.
// Bound by the latency of a wave's few stages; splitting k over the waves
// instead of walking it in one keeps 2048 waves busy on 128 output tiles.
// 77 x 2048 x 4096, 4 bits: 15.9 us, 66.8 us with one workgroup per 64
// weight rows walking all of k (weights in a cache; the k split over workgroups,
// where there is room for its sums, 17.7 with the streams' write, 19.5 here).
template <int BITS, int NT, int MT, int KS>
__global__ __launch_bounds__(64 * KS) void gemm_deep_kernel(QWeight w,
                                                            const uint16_t* __restrict__ x,
                                                            int64_t x_stride, int M,
                                                            ProjEpilogue e) {
  __shared__ __align__(16) floatx4_t red[KS][NT * MT][64];
  const int tid = threadIdx.x, lane = tid & 63, kp = tid >> 6;
  const int j = lane & 15, kq = lane >> 4;
  const int n = w.n, G = w.k >> 6, stages = (G + 1) >> 1;
  const int n0 = blockIdx.x * 16 * NT, m0 = blockIdx.y * 16 * MT;
  const int s0 = stages * kp / KS, s1 = stages * (kp + 1) / KS;
  TileRow tr[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t)
    tr[t] = tile_row(w.codes, w.scales, w.biases, w.k, BITS, min(n0 + 16 * t + j, n - 1));
  const uint16_t* xr[MT];  // rows past M repeat the last one; their sums are not stored
#pragma unroll
  for (int u = 0; u < MT; ++u) xr[u] = x + size_t(min(m0 + 16 * u + j, M - 1)) * x_stride;
  floatx4_t y[NT][MT];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int u = 0; u < MT; ++u) y[t][u] = floatx4_t{0.0f, 0.0f, 0.0f, 0.0f};
  Piece<BITS> p[NT];
  auto load_w = [&](int s) {
#pragma unroll
    for (int t = 0; t < NT; ++t) load_piece<BITS>(tr[t], s, kq, 2 * s + 1 == G, p[t]);
  };
  if (s0 < s1) load_w(s0);
  for (int s = s0; s < s1; ++s) {
    const bool half = 2 * s + 1 == G;  // uniform
    const int q = half ? (kq & 1) : kq;
    uint4 a[MT][4];
#pragma unroll
    for (int u = 0; u < MT; ++u)
#pragma unroll
      for (int st = 0; st < 4; ++st) {
        a[u][st] = *reinterpret_cast<const uint4*>(xr[u] + 128 * s + 32 * q + 8 * st);
        if (half && kq >= 2) a[u][st] = make_uint4(0u, 0u, 0u, 0u);
      }
    uint4 hi[NT][4], lo[NT][4];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      dequant_step<BITS, 0>(p[t], hi[t][0], lo[t][0]);
      dequant_step<BITS, 1>(p[t], hi[t][1], lo[t][1]);
      dequant_step<BITS, 2>(p[t], hi[t][2], lo[t][2]);
      dequant_step<BITS, 3>(p[t], hi[t][3], lo[t][3]);
    }
    if (s + 1 < s1) load_w(s + 1);
#pragma unroll
    for (int st = 0; st < 4; ++st)
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
          for (int u = 0; u < MT; ++u)
            y[t][u] = mfma_bf16(a[u][st], h ? lo[t][st] : hi[t][st], y[t][u]);
  }
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int u = 0; u < MT; ++u) red[kp][t * MT + u][lane] = y[t][u];
  __syncthreads();
  for (int i = tid; i < NT * MT * 64; i += 64 * KS) {
    const int tu = i >> 6, l = i & 63;
    floatx4_t v = red[0][tu][l];
#pragma unroll
    for (int z = 1; z < KS; ++z) v = v + red[z][tu][l];
    const int row = n0 + 16 * (tu / MT) + (l & 15);
    const int mb = m0 + 16 * (tu % MT) + 4 * (l >> 4);
    if (row >= n) continue;
    gemm_epilogue<4>(e, n, M, {mb, mb + 1, mb + 2, mb + 3}, row, {v[0], v[1], v[2], v[3]});
  }
}

// ---------------------------------------------------------------------------
// Workgroup (blockIdx.x, blockIdx.y, blockIdx.z): 64 weight rows x, 32 UW
// activation rows y, groups per z .. + per - 1; wave (wn, wm) of its 2 x 2
// owns 32 weight rows x 16 UW activation rows.  One group at a time: thread t
// dequantises quarter t % 4 of weight row t / 4 and stores its pieces of the
// activation rows, both requested one group (weights: two) ahead.  Rows of
// eight 16-byte pieces in LDS, piece c of row r at slot c ^ (r % 8), so that
// the rows a read takes together fall on different banks without padding
// (padded rows measured 8 % slower).  A group at a time instead of two halves
// the LDS and the registers: three to four workgroups per CU overlap one's
// barriers and dequantising with another's matrix-core work.  512 x 12352 x
// 2048, 4 bits: 61 us (UW = 8), 91 us with two groups per stage at two
// workgroups per CU.
// KIND: what becomes of the sums.  Each is a kernel of its own: with the other
// epilogues' code beside it the plain one took 62.6 us at that size.
// kTileMix (kHcUpMix): the 64 weight rows are the four streams' rows s H + c of 16
// columns c, mixed through LDS in the epilogue (dense_kernel's arithmetic).
// kTileSplit: fp32 partial sums to e.part, added by gemm_reduce_kernel.
enum : int { kTilePlain, kTileSplit, kTileMix, kTileEpilogue };
template <int BITS, int UW, int KIND>
__global__ __launch_bounds__(256) void gemm_tile_kernel(QWeight w, const uint16_t* __restrict__ x,
                                                        int64_t x_stride, int M, int per,
                                                        ProjEpilogue e) {
  constexpr int kM = 32 * UW, kLd = 64;
  constexpr bool MIX = KIND == kTileMix, SPLIT = KIND == kTileSplit;
  __shared__ __align__(16) uint16_t lds[(kM + 2 * 64) * kLd];
  uint16_t* xs = lds;              // [kM][64]
  uint16_t* wh = lds + kM * kLd;   // [64][64]
  uint16_t* wl = wh + 64 * kLd;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int j = lane & 15, kq = lane >> 4;
  const int wn = wave & 1, wm = wave >> 1;
  const int n = w.n, G = w.k >> 6;
  const int mb = blockIdx.y * kM;
  const int gbeg = blockIdx.z * per, gend = min(G, gbeg + per);
  const int cb = int(blockIdx.x) * 16;  // MIX: the workgroup's first column
  const int dr = tid >> 2, dp = tid & 3;
  const int wrow = MIX ? (dr >> 4) * e.hidden + min(cb + (dr & 15), e.hidden - 1)
                       : min(int(blockIdx.x) * 64 + dr, n - 1);
  const TileRow tr = tile_row(w.codes, w.scales, w.biases, w.k, BITS, wrow);
  const int sc = tid & 7, sr = tid >> 3;
  const uint16_t* xp[UW];  // rows past M repeat the last one; their sums are not stored
#pragma unroll
  for (int i = 0; i < UW; ++i)
    xp[i] = x + size_t(min(mb + sr + 32 * i, M - 1)) * x_stride + 8 * sc;
  uint32x4_t xv[UW];
  auto load_x = [&](int g) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < UW; ++i) xv[i] = *reinterpret_cast<const uint32x4_t*>(xp[i] + 64 * g);
  };
  auto load_w = [&](int g, Quarter<BITS>& q) __attribute__((always_inline)) {
    load_quarter<BITS>(tr, min(g, gend - 1), dp, q);  // past the slice: loaded and dropped
  };
  floatx4_t y[2][UW];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int u = 0; u < UW; ++u) y[t][u] = floatx4_t{0.0f, 0.0f, 0.0f, 0.0f};
  Quarter<BITS> w0, w1;
  load_w(gbeg, w0);
  load_w(gbeg + 1, w1);
  load_x(min(gbeg, G - 1));  // (a last slice may be empty)
  for (int g = gbeg; g < gend; ++g) {
    Quarter<BITS> w2;
    load_w(g + 2, w2);
    __syncthreads();  // every wave is done with the previous group
#pragma unroll
    for (int i = 0; i < UW; ++i)
      *reinterpret_cast<uint32x4_t*>(xs + (sr + 32 * i) * kLd + 8 * (sc ^ (sr & 7))) = xv[i];
    uint4 hi[2], lo[2];
    dequant_quarter<BITS, 0>(w0, dp, hi[0], lo[0]);
    dequant_quarter<BITS, 1>(w0, dp, hi[1], lo[1]);
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int at = dr * kLd + 8 * ((2 * dp + t) ^ (dr & 7));
      *reinterpret_cast<uint4*>(wh + at) = hi[t];
      *reinterpret_cast<uint4*>(wl + at) = lo[t];
    }
    __syncthreads();
    if (g + 1 < gend) load_x(g + 1);  // in flight during this group
#pragma unroll
    for (int st = 0; st < 2; ++st) {
      const int slot = 8 * ((4 * st + kq) ^ (j & 7));
      uint4 b[2][2], a[UW];
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        b[0][t] = *reinterpret_cast<const uint4*>(wh + (wn * 32 + 16 * t + j) * kLd + slot);
        b[1][t] = *reinterpret_cast<const uint4*>(wl + (wn * 32 + 16 * t + j) * kLd + slot);
      }
#pragma unroll
      for (int u = 0; u < UW; ++u)
        a[u] = *reinterpret_cast<const uint4*>(xs + (wm * 16 * UW + 16 * u + j) * kLd + slot);
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int u = 0; u < UW; ++u) y[t][u] = mfma_bf16(a[u], b[h][t], y[t][u]);
    }
    w0 = w1;
    w1 = w2;
  }
  __syncthreads();  // the last group's operands are read
  float* ex = reinterpret_cast<float*>(lds);
  if constexpr (MIX) {
    // stream s = 2 wn + t of column cb + j: bf16(p) into LDS [row][s][column]
    static_assert(!MIX || UW == 4, "the tile's sums fill the LDS of 128 rows");
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int u = 0; u < UW; ++u)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          ex[((wm * 16 * UW + 16 * u + 4 * kq + r) * 4 + 2 * wn + t) * 16 + j] =
              round_bf16(y[t][u][r]);
    __syncthreads();
    for (int i = tid; i < kM * 16; i += 256) {
      const int ml = i >> 4, c = i & 15, m = mb + ml;
      if (m >= M || cb + c >= e.hidden) continue;
      float sum = 0.0f;
#pragma unroll
      for (int st = 0; st < 4; ++st) {
        const float xn =
            bf16_to_f32(e.xn[size_t(m) * e.xn_stride + size_t(st) * e.hidden + cb + c]);
        sum = sum + round_bf16(sigmoid_bf16(ex[(ml * 4 + st) * 16 + c]) * xn);
      }
      e.y[size_t(m) * e.y_stride + cb + c] = f32_to_bf16(round_bf16(sum) / 4.0f);
    }
  } else if constexpr (KIND == kTilePlain) {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int row = int(blockIdx.x) * 64 + wn * 32 + 16 * t + j;
#pragma unroll
      for (int u = 0; u < UW; ++u)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int m = mb + wm * 16 * UW + 16 * u + 4 * kq + r;
          if (m < M && row < n) e.y[size_t(m) * e.y_stride + row] = f32_to_bf16(y[t][u][r]);
        }
    }
  } else {
    // sixteen rows at a time through this wave's own part of LDS, so that a
    // row's 32 outputs are written together
    constexpr int kOut = 32 + 1;
    float* out = ex + wave * 16 * kOut;
#pragma unroll
    for (int u = 0; u < UW; ++u) {
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) out[(4 * kq + r) * kOut + 16 * t + j] = y[t][u][r];
      wave_sync();
      const int row = int(blockIdx.x) * 64 + wn * 32 + (lane & 31);
      const int m0 = mb + wm * 16 * UW + 16 * u;
// two rows at a time: more need more registers than the products do
#pragma unroll 1
      for (int b = 0; b < 4 && row < n; ++b) {
        const int r = 4 * b + (lane >> 5);
        const float v0 = out[r * kOut + (lane & 31)], v1 = out[(r + 2) * kOut + (lane & 31)];
        if constexpr (SPLIT) {
          if (m0 + r < M) e.part[(size_t(blockIdx.z) * M + m0 + r) * n + row] = v0;
          if (m0 + r + 2 < M) e.part[(size_t(blockIdx.z) * M + m0 + r + 2) * n + row] = v1;
        } else {
          gemm_epilogue<2>(e, n, M, {m0 + r, m0 + r + 2}, row, {v0, v1});
        }
      }
      wave_sync();
    }
  }
}

// The k slices' partial sums added in slice order, then the epilogue.
__global__ __launch_bounds__(256) void gemm_reduce_kernel(int n, int M, int slices,
                                                          ProjEpilogue e) {
  const size_t i = size_t(blockIdx.x) * 256 + threadIdx.x;
  if (i >= size_t(M) * n) return;
  const int m = int(i / n), row = int(i - size_t(m) * n);
  float v = e.part[i];
  for (int z = 1; z < slices; ++z) v = v + e.part[size_t(z) * M * n + i];
  gemm_epilogue<1>(e, n, M, {m}, row, {v});
}

// ---------------------------------------------------------------------------
template <int BITS, int UW, int KIND>
void launch_tile(const QWeight& w, const uint16_t* x, int64_t xs, int m, int per, dim3 grid,
                 const ProjEpilogue& e, hipStream_t s) {
  hipLaunchKernelGGL((gemm_tile_kernel<BITS, UW, KIND>), grid, dim3(256), 0, s, w, x, xs, m, per,
                     e);
}

template <int BITS, int NT, int MT>
void launch_deep(const QWeight& w, const uint16_t* x, int64_t xs, int m, const ProjEpilogue& e,
                 hipStream_t s) {
  hipLaunchKernelGGL((gemm_deep_kernel<BITS, NT, MT, kDeepWaves>),
                     dim3(div_up(w.n, 16 * NT), div_up(m, 16 * MT)), dim3(64 * kDeepWaves), 0, s, w,
                     x, xs, m, e);
}

template <int BITS>
void launch_gemm(const QWeight& w, const uint16_t* x, int64_t xs, int m, const ProjEpilogue& e,
                 hipStream_t s) {
  const int G = w.k >> 6;
  if (e.mode == kHcUpMix) {
    launch_tile<BITS, 4, kTileMix>(w, x, xs, m, G, dim3(div_up(e.hidden, 16), div_up(m, 128)), e,
                                   s);
    return;
  }
  const GemmPlan p =
      gemm_plan(m, w.n, w.k, BITS, e.mode == kHcWrite, e.part ? e.part_floats : 0);
  if (p.form == GemmPlan::kDeep) {
    switch (p.a * 10 + p.b) {
      case 12: launch_deep<BITS, 1, 2>(w, x, xs, m, e, s); break;
      case 13: launch_deep<BITS, 1, 3>(w, x, xs, m, e, s); break;
      case 22: launch_deep<BITS, 2, 2>(w, x, xs, m, e, s); break;
      case 23: launch_deep<BITS, 2, 3>(w, x, xs, m, e, s); break;
      default: launch_deep<BITS, 2, 4>(w, x, xs, m, e, s); break;
    }
    return;
  }
  const int per = div_up(G, p.b);
  const dim3 grid(div_up(w.n, 64), div_up(m, 32 * p.a), p.b);
#define MX_TILE(U)                                                            \
  case U:                                                                     \
    if (p.b > 1)                                                              \
      launch_tile<BITS, U, kTileSplit>(w, x, xs, m, per, grid, e, s);         \
    else if (e.mode == kPlain)                                                \
      launch_tile<BITS, U, kTilePlain>(w, x, xs, m, per, grid, e, s);         \
    else                                                                      \
      launch_tile<BITS, U, kTileEpilogue>(w, x, xs, m, per, grid, e, s);      \
    break;
  switch (p.a) { MX_TILE(2) MX_TILE(3) MX_TILE(4) MX_TILE(8) }
#undef MX_TILE
  if (p.b > 1)
    hipLaunchKernelGGL(gemm_reduce_kernel, dim3(unsigned((size_t(m) * w.n + 255) / 256)),
                       dim3(256), 0, s, w.n, m, p.b, e);
}

}  // namespace

int qmm_gemm(const QWeight& w, const uint16_t* x, int64_t x_stride, int m, const ProjEpilogue& e,
             hipStream_t s) {
  switch (w.bits) {
    case 4: launch_gemm<4>(w, x, x_stride, m, e, s); break;
    case 5: launch_gemm<5>(w, x, x_stride, m, e, s); break;
    case 6: launch_gemm<6>(w, x, x_stride, m, e, s); break;
    default: launch_gemm<8>(w, x, x_stride, m, e, s); break;
  }
  return hipGetLastError() == hipSuccess ? MX_OK : MX_EHIP;
}

}  // namespace mx
