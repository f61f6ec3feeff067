// Workgroup of the local Hamiltonian's plane kernel (plane_local_impl.hpp). Free of
// HIP so that a host program can walk the rule.
#pragma once

#include <cstddef>

namespace sdft_hip {

constexpr std::size_t kLdsPerCu = 160 * 1024;

// Waves of a workgroup, 4 or 8, whichever leaves more of them on a CU, and 4 where both
// leave as many (0: neither fits): by the LDS, `fixed` bytes a workgroup and `per_wave`
// a wave, of which one workgroup may have `limit`, and by the registers, which hold
// `register_waves` waves a CU of the kernel that runs. Eight waves share the lines of a
// plane, so the LDS alone speaks for them from 48 x 48 in FP64 on, where the registers
// hold one such workgroup but three of four waves. Local H alone, us, by the LDS / by
// both: 120 columns of 49^3 151 / 111, 100 of 54^3 171 / 126, 80 of 60^3 187 / 139, 96 of
// 48 x 48 x 96 309 / 241, 37 of 70 x 35 x 35 85 / 54; FP32 and 72 x 72 take the same
// workgroup either way.
inline int plane_group_waves(std::size_t fixed, std::size_t per_wave, std::size_t limit, int register_waves,
                             int most_waves) {
  int waves = 0, best = 0;
  for (int nw = 4; nw <= most_waves; nw *= 2) {
    const std::size_t lds = fixed + std::size_t(nw) * per_wave;
    if (lds > limit) continue;
    const int by_lds = int(kLdsPerCu / lds), by_registers = register_waves / nw;
    const int resident = nw * (by_lds < by_registers ? by_lds : by_registers);
    if (resident > best) {
      best = resident;
      waves = nw;
    }
  }
  return waves;
}

}  // namespace sdft_hip
