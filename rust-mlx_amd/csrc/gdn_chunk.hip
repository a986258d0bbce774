// Chunked GatedDeltaNet prefill scan (gfx950 matrix cores).
//
// Reference: the delta-rule recurrence of gdn_kernel::recurrent
// (src/gdn_kernel.rs:7-71, kernels/gated_delta.metal), per value head:
//   S_t = g_t S_{t-1} + k_t d_t^T,  d_t = beta_t (v_t - g_t S_{t-1}^T k_t),
//   y_t = bf16(S_t^T q_t)
// with S fp32 [dk][dv] (dk-major, as the decode kernels keep it).
//
// Chunked form over chunks of C = 64 tokens (gamma_t = prod_{r<=t} g_r within
// the chunk, S_0 the state entering it):
//   S_t = gamma_t S_0 + sum_{s<=t} (gamma_t / gamma_s) k_s d_s^T
//   (I + A) D = beta V - (beta gamma K) S_0,  A[t][s] = beta_t (gamma_t/gamma_s) k_t.k_s (s < t)
//   so D = U - W S_0 with T = (I + A)^-1, U = T (beta V), W = T (beta gamma K);
//   O = (gamma Q) S_0 + P D = Q' S_0 + P U with Q' = gamma Q - P W,
//   P[t][s] = (gamma_t/gamma_s) q_t.k_s (s <= t);
//   S_C = gamma_C S_0 + K'^T D,  K'_s = kappa_s k_s, kappa_s = gamma_C / gamma_s.
// Q' takes the output off the chain from chunk to chunk, which is D, then S_C.
// Every product that touches the fp32 state is an fp32 matrix-core product
// (v_mfma_f32_16x16x4_f32), so the state agrees with the sequential fp32
// recurrence to rounding; the Gram matrices K K^T and Q K^T of bf16 inputs
// are exact products with fp32 sums on the bf16 matrix cores.  Decay ratios
// come from an fp64 prefix sum of log2 g (no underflow of the ratios; g = 0
// is clamped to 2^-200, i.e. a full reset).
//
//  chunk_prep_kernel (chunks x heads x groups, parallel): the per-chunk
//    quantities above, written to a workspace in matrix-core operand order.
//  chunk_scan_kernel (16-column state slices x heads x groups): walks the
//    chunks in order, carrying its 128 x 16 slice of the state in LDS.
//
// An fp32 MFMA step takes one k from each lane quarter; which one is free as
// long as both operands agree, so a matrix that is read as an operand is laid
// out for sixteen bytes (four steps) per lane, neighbouring lanes together.
#include "common.hpp"
#include "kernels.hpp"
#include "skinny_core.hpp"

namespace mx {

namespace {

constexpr int kC = 64;   // tokens per chunk
constexpr int kD = 128;  // head dim (dk == dv)
constexpr int kSlice = 16;
constexpr int kLd = kC + 1;      // padded LDS row of a C x C matrix
constexpr int kBLd = kD + 8;     // padded LDS row of a bf16 chunk
constexpr int kPrepThreads = 512;
constexpr int kScanThreads = 512;

// Workspace of one (group, head, chunk), in floats.  A-operand order of an
// R x 128 matrix: [R / 16 tiles][8][64 lanes][4], element (row, k) in lane
// 16 (k / 32) + row % 16 at [(k % 32) / 4][k % 4]; of an R x 64 one:
// [R / 16][4][64][4], element (row, s) in lane 16 (s / 16) + row % 16 at
// [(s % 16) / 4][s % 4] (K^T, bf16: [8][2][64][8] at [(s % 16) / 8][s % 8]).  U as the B operand of P U: [8 slices][4][64][4],
// element (s, column) in lane 16 (s / 16) + column % 16 likewise.
constexpr int kWOff = 0;                // W
constexpr int kQOff = kWOff + kC * kD;  // Q'
constexpr int kKOff = kQOff + kC * kD;  // K^T as bf16, then kappa_s = gamma_C / gamma_s
constexpr int kKappa = kKOff + kC * kD / 2;
constexpr int kPOff = kKOff + kC * kD;  // P
constexpr int kUOff = kPOff + kC * kC;  // U
constexpr int kGOff = kUOff + kC * kD;  // gamma_C
constexpr int kWsFloats = kGOff + 16;

typedef float floatx4_t __attribute__((ext_vector_type(4)));
typedef uint32_t uint32x4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ floatx4_t mfma4(float a, float b, floatx4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// acc += X Y for 16 x 16 blocks in LDS (row-major, leading dims ldx / ldy):
// lane l supplies X[l%16][4kk + l/16] and Y[4kk + l/16][l%16].
__device__ __forceinline__ floatx4_t mm16(const float* X, int ldx, const float* Y, int ldy,
                                          floatx4_t acc) {
  const int lane = threadIdx.x & 63, j = lane & 15, q = lane >> 4;
#pragma unroll
  for (int kk = 0; kk < 4; ++kk) acc = mfma4(X[j * ldx + 4 * kk + q], Y[(4 * kk + q) * ldy + j], acc);
  return acc;
}

// Stores a 16 x 16 D block (lane: rows 4q + r, column j) scaled by `scale`.
__device__ __forceinline__ void store16(float* Z, int ldz, floatx4_t v, float scale) {
  const int lane = threadIdx.x & 63, j = lane & 15, q = lane >> 4;
#pragma unroll
  for (int r = 0; r < 4; ++r) Z[(4 * q + r) * ldz + j] = v[r] * scale;
}

// ---------------------------------------------------------------------------
// Eight waves; wave w owns columns 16 w .. + 15 of W, Q' and U for all tokens.
// W is formed in both orientations from the same operands (products with the
// operands swapped): transposed it is four consecutive k per lane, as it is
// stored; untransposed its registers are the A operand of P W.  72 KB of LDS
// (V takes A's place once T is known): two workgroups per CU.  Bound by the
// serial inverse and the barriers between its steps (matrix cores 35 % busy); at
// 32 heads x 32 chunks 50 us, 159 us with four waves, the scales formed per product and every
// result stored one float per lane.
__global__ __launch_bounds__(kPrepThreads) void chunk_prep_kernel(
    const uint16_t* __restrict__ q, const uint16_t* __restrict__ k,
    const uint16_t* __restrict__ v, const float* __restrict__ g,
    const uint16_t* __restrict__ beta, int hk, int hv, int t, int nchunks, int64_t v_stride,
    float* __restrict__ ws) {
  __shared__ double Ls[kC];                            // inclusive prefix sum of log2 g
  __shared__ float bs[kC], bg[kC], kp[kC], gm[kC];     // beta, beta gamma, kappa, gamma
  __shared__ __align__(16) char av[kC * kBLd * 2];     // K K^T, then A; V once T is known
  __shared__ float QKm[kC * kLd];                      // Q K^T, then P
  __shared__ float Tm[kC * kLd];                       // T = (I + A)^-1
  __shared__ float tmp[3][16 * 17];                    // level products of the blocked inverse
  __shared__ __align__(16) uint16_t Ks[kC * kBLd];     // K chunk
  static_assert(kC * kLd * 4 <= kC * kBLd * 2, "A fits V's place");
  float* Am = reinterpret_cast<float*>(av);
  uint16_t* Vs = reinterpret_cast<uint16_t*>(av);
  const int c = blockIdx.x, h = blockIdx.y, grp = blockIdx.z;
  const int kh = h / (hv / hk);
  const int t0 = c * kC;
  const int len = min(kC, t - t0);
  const int tid = threadIdx.x, lane = tid & 63, j = lane & 15, qd = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // uniform: whole waves branch
  const size_t row0 = size_t(grp) * t + t0;
  float* out = ws + ((size_t(grp) * hv + h) * nchunks + c) * kWsFloats;

  // K chunk into LDS, V chunk into registers (rows past len are zero)
  uint4 vreg[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int u = tid + i * kPrepThreads;  // 16-byte piece
    const int r = u >> 4, cu = u & 15;
    const bool ok = r < len;
    const size_t rr = row0 + (ok ? r : 0);
    uint4 kv = *reinterpret_cast<const uint4*>(k + (rr * hk + kh) * kD + cu * 8);
    vreg[i] = *reinterpret_cast<const uint4*>(v + rr * v_stride + h * kD + cu * 8);
    if (!ok) kv = vreg[i] = make_uint4(0u, 0u, 0u, 0u);
    *reinterpret_cast<uint4*>(Ks + r * kBLd + cu * 8) = kv;
  }
  // log2 g prefix (fp64, wave 0), beta and the scales made of them
  if (tid < kC) {
    const bool ok = tid < len;
    const float gv = ok ? g[(row0 + tid) * hv + h] : 1.0f;
    const float bv = ok ? bf16_to_f32(beta[(row0 + tid) * hv + h]) : 0.0f;
    double l = double(gv > 0x1p-126f ? __builtin_amdgcn_logf(gv) : -200.0f);
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const double n = __shfl_up(l, o, 64);
      if (lane >= o) l += n;
    }
    const double lc = __shfl(l, kC - 1, 64);
    const float gt = __builtin_amdgcn_exp2f(float(l));
    Ls[tid] = l;
    bs[tid] = bv;
    gm[tid] = gt;
    bg[tid] = bv * gt;
    kp[tid] = __builtin_amdgcn_exp2f(float(lc - l));
    if (tid == kC - 1) out[kGOff] = gt;
  }
  // this wave's Gram rows: K (waves 0..3, from LDS) or Q (waves 4..7)
  const int rt = wave & 3;
  uint4 ga[kD / 32];
  if (wave >= 4) {
    const bool rok = 16 * rt + j < len;
    const uint16_t* qr = q + ((row0 + (rok ? 16 * rt + j : 0)) * hk + kh) * kD + 8 * qd;
#pragma unroll
    for (int kk = 0; kk < kD / 32; ++kk) {
      ga[kk] = *reinterpret_cast<const uint4*>(qr + 32 * kk);
      if (!rok) ga[kk] = make_uint4(0u, 0u, 0u, 0u);
    }
  }
  __syncthreads();
  {
    if (wave < 4)
#pragma unroll
      for (int kk = 0; kk < kD / 32; ++kk)
        ga[kk] = *reinterpret_cast<const uint4*>(Ks + (16 * rt + j) * kBLd + 32 * kk + 8 * qd);
    float* dst = wave < 4 ? Am : QKm;
#pragma unroll
    for (int ct = 0; ct < 4; ++ct) {
      sk::floatx4_t gr = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int kk = 0; kk < kD / 32; ++kk)
        gr = sk::mfma(ga[kk],
                      *reinterpret_cast<const uint4*>(Ks + (16 * ct + j) * kBLd + 32 * kk + 8 * qd),
                      gr);
      // A (strictly lower) and P (lower incl. diagonal) with the decay ratios
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int tr = 16 * rt + 4 * qd + r, sc = 16 * ct + j;
        const float ratio = sc <= tr ? __builtin_amdgcn_exp2f(float(Ls[tr] - Ls[sc])) : 0.0f;
        dst[tr * kLd + sc] =
            wave >= 4 ? ratio * gr[r] : sc < tr ? bs[tr] * ratio * gr[r] : 0.0f;
      }
    }
  }
  __syncthreads();
  // T = (I + A)^-1, blocked 4 x 4 over 16 x 16 blocks.
  // Diagonal blocks: wave w < 4, lane j < 16 owns column j of block w.
  if (wave < 4 && j == lane) {
    const int b0 = 16 * wave;
    float col[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      float acc = r == j ? 1.0f : 0.0f;
#pragma unroll
      for (int p = 0; p < r; ++p) acc = fmaf_(-Am[(b0 + r) * kLd + b0 + p], col[p], acc);
      col[r] = acc;
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) Tm[(b0 + r) * kLd + b0 + j] = col[r];
  }
  if (wave >= 4) {  // meanwhile: K^T, kappa and P, eight or four s per lane
    for (int f = tid - 256; f < kC * kD / 8; f += 256) {
      const int l = f & 63, d = 16 * (f >> 7) + (l & 15), s = 16 * (l >> 4) + 8 * ((f >> 6) & 1);
      uint32_t o[4];
#pragma unroll
      for (int i = 0; i < 4; ++i)
        o[i] = uint32_t(Ks[(s + 2 * i) * kBLd + d]) | (uint32_t(Ks[(s + 2 * i + 1) * kBLd + d]) << 16);
      reinterpret_cast<uint4*>(out + kKOff)[f] = make_uint4(o[0], o[1], o[2], o[3]);
    }
    if (tid - 256 < kC) out[kKappa + tid - 256] = kp[tid - 256];
    for (int f = tid - 256; f < kC * kC / 4; f += 256) {
      const int l = f & 63, i4 = (f >> 6) & 3, tr = 16 * (f >> 8) + (l & 15), s = 16 * (l >> 4) + 4 * i4;
      const float* p = QKm + tr * kLd + s;
      reinterpret_cast<float4*>(out + kPOff)[f] = make_float4(p[0], p[1], p[2], p[3]);
    }
  }
  __syncthreads();
  // off-diagonal blocks by distance: T_ij = -T_ii sum_{m=j}^{i-1} A_im T_mj
  // (blocks above the diagonal are never read)
  for (int dist = 1; dist < 4; ++dist) {
    const int bi = wave + dist, bj = wave;  // waves 0 .. 3 - dist
    const bool act = bi < 4;
    if (act) {
      floatx4_t acc = {0.0f, 0.0f, 0.0f, 0.0f};
      for (int m = bj; m < bi; ++m)
        acc = mm16(Am + (16 * bi) * kLd + 16 * m, kLd, Tm + (16 * m) * kLd + 16 * bj, kLd, acc);
      store16(tmp[wave], 17, acc, 1.0f);
      wave_sync();
      acc = floatx4_t{0.0f, 0.0f, 0.0f, 0.0f};
      acc = mm16(Tm + (16 * bi) * kLd + 16 * bi, kLd, tmp[wave], 17, acc);
      store16(Tm + (16 * bi) * kLd + 16 * bj, kLd, acc, -1.0f);
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int u = tid + i * kPrepThreads;
    *reinterpret_cast<uint4*>(Vs + (u >> 4) * kBLd + (u & 15) * 8) = vreg[i];
  }
  __syncthreads();
  // columns 16 wave + j of K and V as operands: k-step i takes s = 4 i + qd
  float kc[16], vc[16];
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int s = 4 * i + qd;
    kc[i] = bf16_to_f32(Ks[s * kBLd + 16 * wave + j]) * bg[s];
    vc[i] = bf16_to_f32(Vs[s * kBLd + 16 * wave + j]) * bs[s];
  }
  floatx4_t wn[4];  // W rows 16 tt + 4 qd + r, column 16 wave + j
#pragma unroll
  for (int tt = 0; tt < 4; ++tt) {
    floatx4_t wt = {0.0f, 0.0f, 0.0f, 0.0f}, un = wt;
    wn[tt] = wt;
#pragma unroll
    for (int i = 0; i < 4 * (tt + 1); ++i) {
      const float a = Tm[(16 * tt + j) * kLd + 4 * i + qd];
      wt = mfma4(kc[i], a, wt);
      wn[tt] = mfma4(a, kc[i], wn[tt]);
      un = mfma4(a, vc[i], un);
    }
    // W^T tile: lane token 16 tt + j, k = 16 wave + 4 qd ..
    reinterpret_cast<floatx4_t*>(out + kWOff)[(tt * 8 + 4 * (wave & 1) + qd) * 64 +
                                              (wave >> 1) * 16 + j] = wt;
    // U tile: tokens 16 tt + 4 qd .., column 16 wave + j
    reinterpret_cast<floatx4_t*>(out + kUOff)[(wave * 4 + qd) * 64 + tt * 16 + j] = un;
  }
  // Q'^T tile: lane token 16 tt + j, k = 16 wave + 4 qd ..; k-step (b, r) takes
  // s = 16 b + 4 qd + r
#pragma unroll
  for (int tt = 0; tt < 4; ++tt) {
    floatx4_t pw = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int b = 0; b <= tt; ++b)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        pw = mfma4(wn[b][r], QKm[(16 * tt + j) * kLd + 16 * b + 4 * qd + r], pw);
    const int tr = 16 * tt + j;
    const bool ok = tr < len;
    const uint2 qv = *reinterpret_cast<const uint2*>(
        q + ((row0 + (ok ? tr : 0)) * hk + kh) * kD + 16 * wave + 4 * qd);
    const float gt = ok ? gm[tr] : 0.0f;
    floatx4_t qo;
    qo[0] = fmaf_(gt, u2f(qv.x << 16), -pw[0]);
    qo[1] = fmaf_(gt, u2f(qv.x & 0xffff0000u), -pw[1]);
    qo[2] = fmaf_(gt, u2f(qv.y << 16), -pw[2]);
    qo[3] = fmaf_(gt, u2f(qv.y & 0xffff0000u), -pw[3]);
    reinterpret_cast<floatx4_t*>(out + kQOff)[(tt * 8 + 4 * (wave & 1) + qd) * 64 +
                                              (wave >> 1) * 16 + j] = qo;
  }
}

// ---------------------------------------------------------------------------
// One 16-column slice of one head's state, chunk after chunk.  Waves 0..3
// carry the chain (wave w: rows 16 w .. of D, then state row tiles 2 w and
// 2 w + 1), waves 4..7 the outputs (wave 4 + w: tokens 16 w ..), which only
// read the state that enters the chunk.  State and D lie in LDS by column, so
// an operand is sixteen bytes per lane; both copies of the state alternate, so
// a chunk takes two barriers.  Operands are requested a chunk ahead (they do
// not depend on the state).  At 32 heads x 32 chunks 104 us, 3.25 us a chunk,
// 213 us with one wave per SIMD doing both, the output after D.  Bound by fp32
// matrix-core time (46 % of the cycles: 64 products of 32 cycles on each SIMD for
// the chain and 48 for the outputs of a chunk), by the chain's two barriers and by
// the workspace's way from L2 (every slice reads 98 KB a chunk; with chunk 0's
// operands throughout a form of 114 us took 89; fp32 K'^T and all of P cost 14 us,
// slices of a head on different XCDs 16 us).
__global__ __launch_bounds__(kScanThreads) void chunk_scan_kernel(
    const float* __restrict__ ws, int hv, int t, int nchunks, const int32_t* __restrict__ slots,
    float* __restrict__ state, uint16_t* __restrict__ y) {
  constexpr int kSLd = kD + 4, kDLd = kC + 4;
  __shared__ __align__(16) float Sl[2][kSlice * kSLd];  // state slice [column][d]
  __shared__ __align__(16) float Dl[kSlice * kDLd];     // D of the chunk [column][s]
  // the eight slices of a head read the same workspace: on one XCD (workgroup
  // ids mod 8) they share its L2, when the heads divide among the XCDs
  static_assert(kD / kSlice == 8, "eight slices");
  const int id = blockIdx.x + 8 * (blockIdx.y + gridDim.y * blockIdx.z);
  const bool even = (gridDim.y * gridDim.z) % 8 == 0;
  const int slice = even ? (id >> 3) & 7 : id & 7;
  const int head = even ? (id >> 6) * 8 + (id & 7) : id >> 3;  // of all groups
  const int h = head % hv, grp = head / hv;
  const int i0 = slice * kSlice;
  const int tid = threadIdx.x, lane = tid & 63, j = lane & 15, qd = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // uniform: whole waves branch
  const int w = wave & 3;
  float* sp = state + (size_t(slots[grp]) * hv + h) * kD * kD + i0;
  for (int e = tid; e < kD * kSlice; e += kScanThreads)
    Sl[0][(e & 15) * kSLd + (e >> 4)] = sp[size_t(e >> 4) * kD + (e & 15)];
  const float* in = ws + (size_t(grp) * hv + h) * nchunks * kWsFloats;
  const floatx4_t zero = {0.0f, 0.0f, 0.0f, 0.0f};
  if (wave < 4) {
    struct Ops {
      floatx4_t w[8], u, kappa;
      uint32x4_t k[2][2];
      float gc;
    };
    auto load = [&](int c, Ops& o) __attribute__((always_inline)) {
      const floatx4_t* p = reinterpret_cast<const floatx4_t*>(in + size_t(c) * kWsFloats);
#pragma unroll
      for (int i = 0; i < 8; ++i) o.w[i] = p[kWOff / 4 + (w * 8 + i) * 64 + lane];
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int i = 0; i < 2; ++i)
          o.k[u][i] = reinterpret_cast<const uint32x4_t*>(
              p)[kKOff / 4 + ((2 * w + u) * 2 + i) * 64 + lane];
      o.kappa = p[kKappa / 4 + 4 * w + qd];
      o.u = p[kUOff / 4 + (slice * 4 + qd) * 64 + w * 16 + j];  // tokens 16 w + 4 qd ..
      o.gc = in[size_t(c) * kWsFloats + kGOff];
    };
    Ops cur, nxt;
    load(0, cur);
    __syncthreads();
    for (int c = 0; c < nchunks; ++c) {
      load(min(c + 1, nchunks - 1), nxt);
      const float* S = Sl[c & 1];
      floatx4_t d0 = zero, d1 = zero;  // two chains: even and odd pieces of k
#pragma unroll
      for (int i = 0; i < 8; i += 2) {
        const floatx4_t s0 = *reinterpret_cast<const floatx4_t*>(S + j * kSLd + 32 * qd + 4 * i);
        const floatx4_t s1 = *reinterpret_cast<const floatx4_t*>(S + j * kSLd + 32 * qd + 4 * i + 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          d0 = mfma4(cur.w[i][e], s0[e], d0);
          d1 = mfma4(cur.w[i + 1][e], s1[e], d1);
        }
      }
      // kappa D: K'^T D is K^T (kappa D), with K as it came
      floatx4_t dk = cur.u - (d0 + d1);
#pragma unroll
      for (int r = 0; r < 4; ++r) dk[r] = dk[r] * cur.kappa[r];
      *reinterpret_cast<floatx4_t*>(Dl + j * kDLd + 16 * w + 4 * qd) = dk;
      __syncthreads();  // D is whole
      floatx4_t a[2] = {zero, zero};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const floatx4_t dv = *reinterpret_cast<const floatx4_t*>(Dl + j * kDLd + 16 * qd + 4 * i);
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int u = 0; u < 2; ++u) {
            const uint32_t kw = cur.k[u][i >> 1][2 * (i & 1) + (e >> 1)];
            a[u] = mfma4(u2f((e & 1) ? (kw & 0xffff0000u) : (kw << 16)), dv[e], a[u]);
          }
      }
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int at = j * kSLd + 16 * (2 * w + u) + 4 * qd;
        const floatx4_t old = *reinterpret_cast<const floatx4_t*>(S + at);
#pragma unroll
        for (int r = 0; r < 4; ++r) a[u][r] = fmaf_(cur.gc, old[r], a[u][r]);
        *reinterpret_cast<floatx4_t*>(Sl[(c + 1) & 1] + at) = a[u];
      }
      __syncthreads();  // the next state is whole
      cur = nxt;
    }
  } else {
    struct Ops {
      floatx4_t q[8], p[4], u[4];
    };
    auto load = [&](int c, Ops& o) __attribute__((always_inline)) {
      const floatx4_t* p = reinterpret_cast<const floatx4_t*>(in + size_t(c) * kWsFloats);
#pragma unroll
      for (int i = 0; i < 8; ++i) o.q[i] = p[kQOff / 4 + (w * 8 + i) * 64 + lane];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        // quarters past the tile's tokens multiply nothing (P is lower triangular)
        o.p[i] = o.u[i] = zero;
        if (qd <= w) {
          o.p[i] = p[kPOff / 4 + (w * 4 + i) * 64 + lane];
          o.u[i] = p[kUOff / 4 + (slice * 4 + i) * 64 + lane];
        }
      }
    };
    Ops cur, nxt;
    load(0, cur);
    __syncthreads();
    for (int c = 0; c < nchunks; ++c) {
      load(min(c + 1, nchunks - 1), nxt);
      const float* S = Sl[c & 1];
      floatx4_t o0 = zero, o1 = zero;
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if (i & 1)
            o1 = mfma4(cur.p[i][e], cur.u[i][e], o1);
          else
            o0 = mfma4(cur.p[i][e], cur.u[i][e], o0);
        }
      // half of the state's products before the barrier on D, half after it
      // (the chain has the matrix cores to itself for as long either way)
      auto half = [&](int i) __attribute__((always_inline)) {
        const floatx4_t s0 = *reinterpret_cast<const floatx4_t*>(S + j * kSLd + 32 * qd + 4 * i);
        const floatx4_t s1 = *reinterpret_cast<const floatx4_t*>(S + j * kSLd + 32 * qd + 4 * i + 4);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          o0 = mfma4(cur.q[i][e], s0[e], o0);
          o1 = mfma4(cur.q[i + 1][e], s1[e], o1);
        }
      };
      half(0);
      __syncthreads();
      half(2);
      half(4);
      half(6);
      const floatx4_t o = o0 + o1;
      const int t0 = c * kC;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int tr = t0 + 16 * w + 4 * qd + r;
        if (tr < t) y[((size_t(grp) * t + tr) * hv + h) * kD + i0 + j] = f32_to_bf16(o[r]);
      }
      __syncthreads();
      cur = nxt;
    }
  }
  for (int e = tid; e < kD * kSlice; e += kScanThreads)
    sp[size_t(e >> 4) * kD + (e & 15)] = Sl[nchunks & 1][(e & 15) * kSLd + (e >> 4)];
}

}  // namespace

size_t gdn_chunk_workspace_bytes(int groups, int hv, int t) {
  const size_t nchunks = (size_t(t) + kC - 1) / kC;
  return size_t(groups) * hv * nchunks * kWsFloats * sizeof(float);
}

int gdn_prefill_chunked(const uint16_t* q, const uint16_t* k, const uint16_t* v, const float* g,
                        const uint16_t* beta, GdnDims d, int groups, int t, const int32_t* slots,
                        float* state, uint16_t* y, float* workspace, hipStream_t s,
                        int64_t v_stride) {
  if (d.dk != kD || d.dv != kD || d.hk <= 0 || d.hv % d.hk != 0) return MX_EUNSUPPORTED;
  if (groups <= 0 || t <= 0) return MX_OK;
  const int nchunks = (t + kC - 1) / kC;
  if (v_stride <= 0) v_stride = int64_t(d.hv) * kD;
  hipLaunchKernelGGL(chunk_prep_kernel, dim3(nchunks, d.hv, groups), dim3(kPrepThreads), 0, s, q, k, v, g,
                     beta, d.hk, d.hv, t, nchunks, v_stride, workspace);
  hipLaunchKernelGGL(chunk_scan_kernel, dim3(kD / kSlice, d.hv, groups), dim3(kScanThreads), 0, s,
                     workspace, d.hv, t, nchunks, slots, state, y);
  return hipGetLastError() == hipSuccess ? MX_OK : MX_EHIP;
}

}  // namespace mx
