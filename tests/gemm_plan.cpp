// The GEMM's choice of a form, for tests (built by the gemm_plan fixture).
#include "../rust-mlx_amd/csrc/gemm_plan.hpp"

extern "C" void gemm_plan(int m, int n, int k, int bits, int streams, size_t part_floats, int* out) {
  const mx::GemmPlan p = mx::gemm_plan(m, n, k, bits, streams != 0, part_floats);
  out[0] = p.form == mx::GemmPlan::kDeep;
  out[1] = p.a;
  out[2] = p.b;
}
