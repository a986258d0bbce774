// Which form of the GEMM beyond 16 rows runs (gemm.hip), by an estimate of
// their times.  Host code with no device types.
#pragma once

#include <cstddef>
#include <cstdint>
#include <type_traits>

namespace mx {

struct GemmPlan {
  enum Form { kTile, kDeep } form;
  int a, b;  // tile: UW and slices; deep: NT and MT
};

constexpr int kDeepWaves = 8;

inline int div_up(int a, int b) { return (a + b - 1) / b; }

// (a^3 + b^3)^(1/3) and (a^4 + b^4)^(1/4) to half a per cent, without roots: the
// choice is made anew for every call, on the host path of its launch (0.14 us, 0.3
// where k may be split).
inline double soft_max3(double a, double b) {
  const double hi = a > b ? a : b, x = (a > b ? b : a) / hi, c = x * x * x;
  return hi * (1.0 + c * (1.0 / 3 - 0.0734 * c));
}
inline double soft_max4(double a, double b) {
  const double hi = a > b ? a : b, x = (a > b ? b : a) / hi, c = x * x * x * x;
  return hi * (1.0 + c * (0.25 - 0.0608 * c));
}

// Estimated microseconds on 256 CUs, fitted to sweeps of every form over 17 ..
// 512 rows x 64 .. 20000 weight rows x k 256 .. 8192 at all widths, once with
// the weights from memory (a model's layers follow one another: none of its
// weights are in a cache) and once with one matrix again and again.  The form
// this chooses takes 0.6 % longer than the fastest on average over the sweeps,
// 5 % at the 95th percentile.  From memory, against 128-row tiles with k split
// to 256 workgroups: 2048 x 4096 with the streams' write 26.9 -> 25.0 us at 256
// rows (tiles, k in eight slices; deep 28.7) and 19.9 both at 128 (deep 20.5),
// 260 x 8192 at 512 23.4 -> 21.6, 513 x 2048 at 512 17.1 -> 12.5, 12352 x 2048
// at 512 91.7 -> 61.3.
//
// tile: every group costs a workgroup its latency or, with several on a CU,
// their matrix-core time.
template <int UW>
double gemm_tile_us(int m, int n, int k, int bits, bool streams, int slices) {
  // workgroups of a CU, by the registers of the kernel for these outputs
  const int resident = UW == 2   ? (streams && slices == 1 ? 5 : 6)
                       : UW == 3 ? (streams || slices > 1 ? 4 : 5)
                       : UW == 4 ? 4
                                 : 2;
  const double per_cu = double(div_up(n, 64)) * div_up(m, 32 * UW) * slices * (1.0 / 256);
  const double latency = 0.498 + 0.115 * UW;
  const double busy = 0.231 + 0.076 * UW + (bits == 4 ? 0.0 : 0.019);
  const int rounds = int(per_cu / resident);
  const double rest = per_cu - rounds * resident;
  double group = rounds > 0 ? rounds * soft_max3(latency, resident * busy) : 0.0;
  if (rest > 0) {
    const int whole = int(rest) < rest ? int(rest) + 1 : int(rest);
    group += soft_max3(latency, (rest + whole) / 2 * busy);
  }
  const double outs = double(m) * n * 1e-6;
  double t = 3.58 + div_up(k >> 6, slices) * group + 0.261 * per_cu * (slices > 1 ? UW : UW / 2.0);
  if (slices > 1) t += 5.78 + 0.095 * outs * (4 * slices + 2);  // the reduction
  // kHcWrite reads and writes four streams, here two rows of a wave at a time
  if (streams) t += slices > 1 ? 1.61 * outs : 4.14 * outs + 2.82 * UW;
  return t;
}

// deep: every stage costs a round of workgroups its latency, or the memory
// system the weights and the activations that each wave reads for itself.
template <int NT, int MT>
double gemm_deep_us(int m, int n, int k, int bits, bool streams) {
  constexpr int resident = NT * MT == 2 ? 2 : 1;
  const int G = k >> 6;
  const double groups = double(div_up(n, 16 * NT)) * div_up(m, 16 * MT);
  const double per_cu = groups * (1.0 / 256);
  const double share = per_cu / resident;
  const int rounds = int(share) < share ? int(share) + 1 : int(share);
  const double stage = 0.115 + 0.516 * MT + 1.42 * NT + 0.093 * MT * NT;
  const double two = resident == 2 ? 1.646 : 1.0;  // both workgroups of a CU
  const double walk = div_up(div_up(G, 2), kDeepWaves) * stage *
                      ((rounds - 1) * two + (per_cu - (rounds - 1) * resident > 1 ? two : 1.0));
  const double read = double(n) * k * (bits / 8.0 + 0.0625) / 13.1e6 +
                      groups * G * (2048.0 * MT + 128.0 * NT * bits) / 10.2e6;
  const double t = 0.71 + soft_max4(walk, read);
  return streams ? t + 2.47 + 2.33e-6 * m * n : t;
}

// m activation rows, weights n x k; streams: the kHcWrite epilogue;
// part_floats: room for partial sums of k slices.
inline GemmPlan gemm_plan(int m, int n, int k, int bits, bool streams, size_t part_floats) {
  GemmPlan best{GemmPlan::kTile, 4, 1};
  double least = 1e30;
  auto take = [&](double t, GemmPlan p) {
    if (t < least) {
      least = t;
      best = p;
    }
  };
  // (the shapes as template arguments: the divisions by them are by constants)
  auto tiles = [&](auto shape) {
    constexpr int UW = decltype(shape)::value;
    for (int slices = 1; slices <= 16; slices *= 2) {
      // (slices of fewer groups cost more than the estimate says: 16 slices of
      // four groups at 64 x 2048 x 4096 17.9 us, 8 of eight 15.9)
      if (slices > 1 && ((k >> 6) < 6 * slices || size_t(slices) * m * n > part_floats)) break;
      take(gemm_tile_us<UW>(m, n, k, bits, streams, slices), {GemmPlan::kTile, UW, slices});
    }
  };
  tiles(std::integral_constant<int, 2>());
  tiles(std::integral_constant<int, 3>());
  tiles(std::integral_constant<int, 4>());
  tiles(std::integral_constant<int, 8>());
  take(gemm_deep_us<1, 2>(m, n, k, bits, streams), {GemmPlan::kDeep, 1, 2});
  take(gemm_deep_us<1, 3>(m, n, k, bits, streams), {GemmPlan::kDeep, 1, 3});
  take(gemm_deep_us<2, 2>(m, n, k, bits, streams), {GemmPlan::kDeep, 2, 2});
  take(gemm_deep_us<2, 3>(m, n, k, bits, streams), {GemmPlan::kDeep, 2, 3});
  take(gemm_deep_us<2, 4>(m, n, k, bits, streams), {GemmPlan::kDeep, 2, 4});
  return best;
}

}  // namespace mx
