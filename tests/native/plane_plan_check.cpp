// The plane kernel's workgroup rule (csrc/hip/plane_plan.hpp) for the host tests.
#include "../../sparse-dft_amd/csrc/hip/plane_plan.hpp"

extern "C" int plane_group_waves_of(long fixed, long per_wave, long limit, int register_waves, int most_waves) {
  return sdft_hip::plane_group_waves(std::size_t(fixed), std::size_t(per_wave), std::size_t(limit), register_waves,
                                     most_waves);
}
