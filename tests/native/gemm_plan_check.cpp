// The complex GEMM's launch plan (csrc/hip/gemm_plan.hpp) for the host tests.
#include "../../sparse-dft_amd/csrc/hip/gemm_plan.hpp"

extern "C" void gemm_plan_of(int fp64, int m, int n, int k, int out[3]) {
  const sdft_hip::GemmPlan p = sdft_hip::gemm_plan(fp64 != 0, m, n, k);
  out[0] = p.cfg;
  out[1] = p.splits;
  out[2] = p.kps;
}
