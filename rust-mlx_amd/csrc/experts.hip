// Expert MLPs of a prefill chunk (more than eight rows) on the gfx950 matrix
// cores, for depths whose activation rows fit LDS whole; qmm.hip holds the
// general forms and chooses.
//
// Replaces the same reference interfaces as qmm.hip's chunk kernels (the
// expert gate/up/down of MoE::parts, src/hybrid.rs:192-287) with the
// arithmetic of qmm_core.hpp: codes as exact bf16 integers, fp32 sums per
// 64-value group, scale and bias applied in fp32.
//
// A workgroup serves one item of the ChunkPlan (an expert and
// up to 16 of its routes).  The item's activation rows lie in LDS whole, in
// operand order (permute_x), with their group sums beside them, so after one
// barrier every wave streams its own weight rows to the end without meeting
// the others: units of two 16-row tiles x four groups, the next unit's codes
// in flight while this one is multiplied.
#include "common.hpp"
#include "kernels.hpp"
#include "qmm_core.hpp"

namespace mx {

namespace {

constexpr int kExWaves = 8;      // gate/up: the rows of a deep item fill half of a CU's LDS
constexpr int kExDownWaves = 4;  // down: registers, not LDS, bound the waves of a CU
constexpr int kExRowPad = 8;  // bf16 of padding: the 16 rows of a read fall on different banks

constexpr int ex_row(int k) { return k + kExRowPad; }
constexpr int ex_lds(int k) { return 16 * ex_row(k) * 2 + (k >> 6) * 16 * 4; }

struct ExItem {
  int m, expert, start;
};

__device__ __forceinline__ ExItem ex_item(const ChunkPlan* __restrict__ plan, int item) {
  return ExItem{plan->m[item], plan->expert[item], plan->start[item]};
}

// Loads of a unit (two tiles x four groups).  Lane 4 r + q reads quarter q of
// each group of row r, so four neighbouring lanes share one access of the
// vector L1 (it serves one per lane otherwise: with neighbouring lanes on
// different rows a gate/up kernel that only loaded took 221 us where this one
// takes 155); ds_bpermute moves the words to lane 16 q + r,
// where the matrix cores want them.  Scales and biases come once per pair of
// units: lane 4 r + q reads eight groups of row r, of tile q / 2's scales (q
// even) or biases (q odd).
template <int BITS>
struct ExUnit {
  uint32_t c[4][2][group_words<BITS>()];
};

template <int BITS>
__device__ __forceinline__ void ex_load(const TileRow (&tr)[2], int g, ExUnit<BITS>& u) {
  const int q = threadIdx.x & 3;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int t = 0; t < 2; ++t) load_group_codes<BITS>(tr[t].codes, g + i, q, u.c[i][t]);
}

// a native vector: HIP's uint4 was left in scratch memory here
typedef uint32_t uint32x4_t __attribute__((ext_vector_type(4)));

// This lane's scale or bias row (see ex_load); the pointers by value, since a
// choice among array elements leaves the array in scratch memory.
__device__ __forceinline__ const uint16_t* ex_scale_row(const uint16_t* s0, const uint16_t* b0,
                                                        const uint16_t* s1, const uint16_t* b1) {
  const uint64_t v[4] = {uint64_t(s0), uint64_t(b0), uint64_t(s1), uint64_t(b1)};
  const int q = threadIdx.x & 3;
  const uint64_t lo = q & 1 ? v[1] : v[0], hi = q & 1 ? v[3] : v[2];
  return reinterpret_cast<const uint16_t*>(q & 2 ? hi : lo);
}

__device__ __forceinline__ uint32x4_t ex_load_scales(const uint16_t* row, int g) {
  return *reinterpret_cast<const uint32x4_t*>(row + g);
}

__device__ __forceinline__ uint32_t from_lane(int lane, uint32_t v) {
  return uint32_t(__builtin_amdgcn_ds_bpermute(4 * lane, int(v)));
}

// ODD: the pair's second unit.
template <int BITS, bool ODD>
__device__ __forceinline__ void ex_multiply(const ExUnit<BITS>& u, const uint32x4_t& scales,
                                            const uint16_t* arow, const float* sums, int g,
                                            floatx4_t (&y)[2]) {
  const int lane = threadIdx.x & 63, j = lane & 15, kq = lane >> 4;
  const float off = code_offset<BITS>();
  uint32_t sw[2][2], bw[2][2];
#pragma unroll
  for (int t = 0; t < 2; ++t)
#pragma unroll
    for (int w = 0; w < 2; ++w) {
      const uint32_t v = scales[(ODD ? 2 : 0) + w];
      sw[t][w] = from_lane(4 * j + 2 * t, v);
      bw[t][w] = from_lane(4 * j + 2 * t + 1, v);
    }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint4* xp = reinterpret_cast<const uint4*>(arow + 64 * (g + i) + 16 * kq);
    const uint4 a0 = xp[0], a1 = xp[1];
    const floatx4_t sx = *reinterpret_cast<const floatx4_t*>(sums + 16 * (g + i) + 4 * kq);
    uint32_t c[2][group_words<BITS>()];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int w = 0; w < group_words<BITS>(); ++w) c[t][w] = from_lane(4 * j + kq, u.c[i][t][w]);
    floatx4_t acc[2];
#pragma unroll
    for (int t = 0; t < 2; ++t)
      acc[t] = mfma_bf16(a0, codes_operand<BITS, 0>(c[t]), floatx4_t{0.f, 0.f, 0.f, 0.f});
#pragma unroll
    for (int t = 0; t < 2; ++t) acc[t] = mfma_bf16(a1, codes_operand<BITS, 1>(c[t]), acc[t]);
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const uint32_t sv = sw[t][i >> 1], bv = bw[t][i >> 1];
      const float sc = u2f((i & 1) ? (sv & 0xffff0000u) : (sv << 16));
      const float bi = fmaf_(-off, sc, u2f((i & 1) ? (bv & 0xffff0000u) : (bv << 16)));
#pragma unroll
      for (int r = 0; r < 4; ++r) y[t][r] = fmaf_(sc, acc[t][r], fmaf_(bi, sx[r], y[t][r]));
    }
  }
}

// The item's rows into LDS: T threads a member, thread t every T-th 16-byte
// piece of member t / T's row (eight neighbouring threads hold one group).
// Rows past the item's members stay as they are: what they give is not stored.
template <int T>
__device__ __forceinline__ void ex_stage(const uint16_t* __restrict__ src, bool live, int k,
                                         uint16_t* xs, float* sums) {
  const int mem = threadIdx.x / T, p0 = threadIdx.x % T;
  if (live)
    for (int p = p0; p < (k >> 3); p += T) {  // k % 256 == 0: whole rounds
      const uint4 v = *reinterpret_cast<const uint4*>(src + 8 * p);
      *reinterpret_cast<uint4*>(xs + mem * ex_row(k) + 8 * p) = permute_x(v);
      const uint32_t w[4] = {v.x, v.y, v.z, v.w};
      float s = 0.0f;
#pragma unroll
      for (int i = 0; i < 4; ++i) s = s + (u2f(w[i] << 16) + u2f(w[i] & 0xffff0000u));
      s = s + __shfl_xor(s, 1, 64);
      s = s + __shfl_xor(s, 2, 64);
      s = s + __shfl_xor(s, 4, 64);
      if ((p0 & 7) == 0) sums[16 * (p >> 3) + mem] = s;
    }
}

__device__ __forceinline__ QWeight ex_weight(const QBank& b, int expert, const QWeight& shared) {
  if (expert < 0) return shared;
  const size_t cs = size_t(b.n) * b.k * b.bits / 32;
  const size_t ss = size_t(b.n) * (b.k / b.group_size);
  return QWeight{b.codes + cs * expert, b.scales + ss * expert, b.biases + ss * expert, b.n, b.k,
                 b.bits, b.group_size};
}

// gate/up: wave w of workgroup x takes gate and up rows 16 (8 x + w) .. + 15.
// Bound by the weight stream (604 MB at 301 rows over 512 experts of 2 x 512 x
// 2048, 4 bits: 152 us, 4.0 TB/s; 193 us with the rows passing through LDS in
// batches between barriers, both under the profiler).  At 4 bits 124 registers
// let two workgroups run per CU; a second pair of tiles per wave needs 135 and
// took 171 us.
template <int BITS>
__global__ __launch_bounds__(64 * kExWaves) void chunk_gate_up_lds_kernel(
    const uint16_t* __restrict__ x, const ChunkPlan* __restrict__ plan, int top_k, QBank gate,
    QBank up, QWeight sgate, QWeight sup, uint16_t* __restrict__ h, int hs) {
  if (int(blockIdx.y) >= plan->nitems) return;
  extern __shared__ __align__(16) uint16_t ex_mem[];
  const ExItem it = ex_item(plan, blockIdx.y);
  const QWeight gw = ex_weight(gate, it.expert, sgate);
  const QWeight uw = ex_weight(up, it.expert, sup);
  const int hidden = gate.k, G = hidden >> 6, inter = gw.n;
  if (int(blockIdx.x) * 16 * kExWaves >= inter) return;
  float* sums = reinterpret_cast<float*>(ex_mem + 16 * ex_row(hidden));
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int j = lane & 15, kq = lane >> 4;
  const int base = (blockIdx.x * kExWaves + wave) * 16;
  const int row = min(base + (lane >> 2), inter - 1);
  const TileRow tr[2] = {tile_row(gw.codes, gw.scales, gw.biases, hidden, BITS, row),
                         tile_row(uw.codes, uw.scales, uw.biases, hidden, BITS, row)};
  ExUnit<BITS> u0, u1;
  const uint16_t* srow = ex_scale_row(tr[0].scales, tr[0].biases, tr[1].scales, tr[1].biases);
  uint32x4_t s0 = ex_load_scales(srow, 0), s1 = s0;
  ex_load<BITS>(tr, 0, u0);
  {
    const int mem = threadIdx.x / (4 * kExWaves);
    const bool live = mem < it.m;
    ex_stage<4 * kExWaves>(x + size_t(plan->row[it.start + (live ? mem : 0)]) * hidden, live, hidden, ex_mem,
             sums);
  }
  __syncthreads();
  if (base >= inter) return;
  const uint16_t* arow = ex_mem + j * ex_row(hidden);
  floatx4_t y[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
  for (int g = 0; g < G; g += 8) {  // a pair of units
    ex_load<BITS>(tr, g + 4, u1);
    ex_multiply<BITS, false>(u0, s0, arow, sums, g, y);
    if (g + 8 < G) {
      ex_load<BITS>(tr, g + 8, u0);
      s1 = ex_load_scales(srow, g + 8);
    }
    ex_multiply<BITS, true>(u1, s0, arow, sums, g + 4, y);
    s0 = s1;
  }
  const int c = base + j;
  if (c >= inter) return;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int m = 4 * kq + r;
    if (m >= it.m) continue;
    const float gv = round_bf16(y[0][r]);
    const float uv = round_bf16(y[1][r]);
    const float silu = round_bf16(gv * sigmoid_bf16(gv));
    const size_t to = size_t(plan->row[it.start + m]) * (top_k + 1) + plan->slot[it.start + m];
    h[to * hs + c] = f32_to_bf16(silu * uv);
  }
}

// down: wave w of workgroup x takes kExPasses pairs of 16-row tiles, one after
// the other (a pair is few units at these depths), the next pair's first unit
// in flight during the last one of this.  370 MB at 301 rows, 5 bits: 111 us
// (one pair per wave 142, two 124, eight 116; 144 us with the batches).
constexpr int kExPasses = 4;
constexpr int kExDownRows = kExDownWaves * kExPasses * 32;  // rows of a workgroup

template <int BITS>
__global__ __launch_bounds__(64 * kExDownWaves) void chunk_down_lds_kernel(
    const uint16_t* __restrict__ h, const ChunkPlan* __restrict__ plan,
    const uint16_t* __restrict__ scores, int top_k, QBank down, QWeight sdown,
    uint16_t* __restrict__ p, int hs, int kmax) {
  if (int(blockIdx.y) >= plan->nitems) return;
  extern __shared__ __align__(16) uint16_t ex_mem[];
  const ExItem it = ex_item(plan, blockIdx.y);
  const QWeight dw = ex_weight(down, it.expert, sdown);
  const int hidden = dw.n, inter = dw.k, pairs = inter >> 9;
  float* sums = reinterpret_cast<float*>(ex_mem + 16 * ex_row(kmax));
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int j = lane & 15, kq = lane >> 4;
  const int base0 = blockIdx.x * kExDownRows + wave * kExPasses * 32;
  auto rows_of = [&](int pass, TileRow(&tr)[2]) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < 2; ++t)
      tr[t] = tile_row(dw.codes, dw.scales, dw.biases, inter, BITS,
                       min(base0 + 32 * pass + 16 * t + (lane >> 2), hidden - 1));
  };
  // pair of units i: groups 8 (i % pairs) .. of pass i / pairs
  const int total = kExPasses * pairs;
  ExUnit<BITS> u0, u1;
  TileRow tr[2];
  rows_of(0, tr);
  const uint16_t* srow = ex_scale_row(tr[0].scales, tr[0].biases, tr[1].scales, tr[1].biases);
  uint32x4_t s0 = ex_load_scales(srow, 0), s1 = s0;
  ex_load<BITS>(tr, 0, u0);
  {
    const int mem = threadIdx.x / (4 * kExDownWaves);
    const bool live = mem < it.m;
    const int at = it.start + (live ? mem : 0);
    ex_stage<4 * kExDownWaves>(h + (size_t(plan->row[at]) * (top_k + 1) + plan->slot[at]) * hs, live, inter, ex_mem,
             sums);
  }
  size_t to[4];
  float sc[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int at = it.start + min(4 * kq + r, it.m - 1);
    const int row = plan->row[at], slot = plan->slot[at];
    to[r] = (size_t(row) * (top_k + 1) + slot) * hidden;
    sc[r] = slot < top_k ? bf16_to_f32(scores[size_t(row) * top_k + slot]) : 1.0f;
  }
  __syncthreads();
  const uint16_t* arow = ex_mem + j * ex_row(inter);
  floatx4_t y[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
  for (int i = 0; i < total; ++i) {
    const int g = 8 * (i % pairs);
    ex_load<BITS>(tr, g + 4, u1);
    ex_multiply<BITS, false>(u0, s0, arow, sums, g, y);
    if (i + 1 < total) {
      const int gn = 8 * ((i + 1) % pairs);
      if (gn == 0) {
        rows_of((i + 1) / pairs, tr);
        srow = ex_scale_row(tr[0].scales, tr[0].biases, tr[1].scales, tr[1].biases);
      }
      ex_load<BITS>(tr, gn, u0);
      s1 = ex_load_scales(srow, gn);
    }
    ex_multiply<BITS, true>(u1, s0, arow, sums, g + 4, y);
    s0 = s1;
    if ((i + 1) % pairs != 0) continue;
    const int c0 = base0 + 32 * (i / pairs);
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const int c = c0 + 16 * t + j;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        if (c < hidden && 4 * kq + r < it.m) {
          const float dv = round_bf16(y[t][r]);
          p[to[r] + c] = f32_to_bf16(it.expert >= 0 ? dv * sc[r] : dv);
        }
        y[t][r] = 0.0f;
      }
    }
  }
}

}  // namespace

// Whole pairs of units, and room in LDS for two workgroups per CU (k <= 2048).
bool chunk_lds_ok(int k) { return k > 0 && k % 512 == 0 && ex_lds(k) <= 80 * 1024; }

int chunk_gate_up_lds(const uint16_t* x, const ChunkPlan* plan, int items, int top_k,
                      const QBank& gate, const QBank& up, const QWeight& sgate,
                      const QWeight& sup, uint16_t* h, hipStream_t s) {
  const int hs = gate.n > sgate.n ? gate.n : sgate.n;
  const dim3 grid((hs + 16 * kExWaves - 1) / (16 * kExWaves), items);
  const int lds = ex_lds(gate.k);
#define MX_GU(B)                                                                                \
  case B:                                                                                       \
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(chunk_gate_up_lds_kernel<B>),         \
                            hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess)     \
      return MX_EHIP;                                                                           \
    hipLaunchKernelGGL((chunk_gate_up_lds_kernel<B>), grid, dim3(64 * kExWaves), lds, s, x, plan,  \
                       top_k, gate, up, sgate, sup, h, hs);                                     \
    break;
  switch (gate.bits) {
    MX_GU(4) MX_GU(5) MX_GU(6) MX_GU(8)
    default: return MX_EUNSUPPORTED;
  }
#undef MX_GU
  return hipGetLastError() == hipSuccess ? MX_OK : MX_EHIP;
}

int chunk_down_lds(const uint16_t* h, const ChunkPlan* plan, const uint16_t* scores, int items,
                   int top_k, int hs, const QBank& down, const QWeight& sdown, uint16_t* p,
                   hipStream_t s) {
  const dim3 grid((down.n + kExDownRows - 1) / kExDownRows, items);
  const int kmax = down.k > sdown.k ? down.k : sdown.k;
  const int lds = ex_lds(kmax);
#define MX_DN(B)                                                                                \
  case B:                                                                                       \
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(chunk_down_lds_kernel<B>),            \
                            hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess)     \
      return MX_EHIP;                                                                           \
    hipLaunchKernelGGL((chunk_down_lds_kernel<B>), grid, dim3(64 * kExDownWaves), lds, s, h, plan,     \
                       scores, top_k, down, sdown, p, hs, kmax);                                \
    break;
  switch (down.bits) {
    MX_DN(4) MX_DN(5) MX_DN(6) MX_DN(8)
    default: return MX_EUNSUPPORTED;
  }
#undef MX_DN
  return hipGetLastError() == hipSuccess ? MX_OK : MX_EHIP;
}

}  // namespace mx
