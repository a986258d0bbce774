// Which form of the GEMM beyond 16 rows runs (gemm.hip), by an estimate of
// their times.  Host code with no device types.
#pragma once

#include <cmath>
#include <cstddef>
#include <cstdint>
#include <initializer_list>

namespace mx {

struct GemmPlan {
  enum Form { kTile, kDeep } form;
  int a, b;  // tile: UW and slices; deep: NT and MT
};

constexpr int kDeepWaves = 8;

inline int div_up(int a, int b) { return (a + b - 1) / b; }

// max(a, b), rounded off where they are about equal.
inline double soft_max(double a, double b) { return std::cbrt(a * a * a + b * b * b); }

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
inline double gemm_tile_us(int m, int n, int k, int bits, bool streams, int uw, int slices) {
  // workgroups of a CU, by the registers of the kernel for these outputs
  const int resident = uw == 2   ? (streams && slices == 1 ? 5 : 6)
                       : uw == 3 ? (streams || slices > 1 ? 4 : 5)
                       : uw == 4 ? 4
                                 : 2;
  const double per_cu = double(div_up(n, 64)) * div_up(m, 32 * uw) * slices / 256.0;
  const double latency = 0.498 + 0.115 * uw;
  const double busy = 0.231 + 0.076 * uw + (bits == 4 ? 0.0 : 0.019);
  const double rounds = std::floor(per_cu / resident), rest = per_cu - rounds * resident;
  double group = rounds * soft_max(latency, resident * busy);
  if (rest > 0) group += soft_max(latency, (rest + std::ceil(rest)) / 2 * busy);
  const double outs = double(m) * n * 1e-6;
  double t = 3.58 + div_up(k >> 6, slices) * group + 0.261 * per_cu * (slices > 1 ? uw : uw / 2.0);
  if (slices > 1) t += 5.78 + 0.095 * outs * (4 * slices + 2);  // the reduction
  // kHcWrite reads and writes four streams, here two rows of a wave at a time
  if (streams) t += slices > 1 ? 1.61 * outs : 4.14 * outs + 2.82 * uw;
  return t;
}

// deep: every stage costs a round of workgroups its latency, or the memory
// system the weights and the activations that each wave reads for itself.
inline double gemm_deep_us(int m, int n, int k, int bits, bool streams, int nt, int mt) {
  const int G = k >> 6, resident = nt * mt == 2 ? 2 : 1;
  const double groups = double(div_up(n, 16 * nt)) * div_up(m, 16 * mt);
  const double per_cu = groups / 256.0;
  const int rounds = int(std::ceil(per_cu / resident));
  const double stage = 0.115 + 0.516 * mt + 1.42 * nt + 0.093 * mt * nt;
  const double two = resident == 2 ? 1.646 : 1.0;  // both workgroups of a CU
  const double walk = div_up(div_up(G, 2), kDeepWaves) * stage *
                      ((rounds - 1) * two + (per_cu - (rounds - 1) * resident > 1 ? two : 1.0));
  const double read = double(n) * k * (bits / 8.0 + 0.0625) / 13.1e6 +
                      groups * G * (2048.0 * mt + 128.0 * nt * bits) / 10.2e6;
  const double t = 0.71 + std::sqrt(std::sqrt(walk * walk * walk * walk + read * read * read * read));
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
  for (int uw : {2, 3, 4, 8})
    for (int slices = 1; slices <= 16; slices *= 2) {
      // (slices of fewer groups cost more than the estimate says: 16 slices of
      // four groups at 64 x 2048 x 4096 17.9 us, 8 of eight 15.9)
      if (slices > 1 && ((k >> 6) / slices < 6 || size_t(slices) * m * n > part_floats)) break;
      take(gemm_tile_us(m, n, k, bits, streams, uw, slices), {GemmPlan::kTile, uw, slices});
    }
  constexpr int deep[][2] = {{1, 2}, {1, 3}, {2, 2}, {2, 3}, {2, 4}};
  for (const auto& d : deep)
    take(gemm_deep_us(m, n, k, bits, streams, d[0], d[1]), {GemmPlan::kDeep, d[0], d[1]});
  return best;
}

}  // namespace mx
