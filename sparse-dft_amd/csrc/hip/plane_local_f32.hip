// The local Hamiltonian's plane kernel in FP32 (plane_local_impl.hpp).
#include "plane_local_impl.hpp"

namespace sdft_hip {

template bool plan_plane_local<float>(const GridPlanDev&, PlaneLocalPlan&);
template hipError_t launch_plane_local<float>(const GridPlanDev&, const PlaneLocalPlan&, const void*, void*, long,
                                              hipStream_t);

// Loads this file's code object on the calling thread (see module_prime.hpp) and asks
// what the launch rule will want to know, so that no application does.
hipError_t prime_module_plane_local_f32() {
  (void)plane_local::register_waves<float, true, false>();
  (void)plane_local::register_waves<float, false, true>();
  (void)plane_local::register_waves<float, false, false>();
  hipFuncAttributes a{};
  return hipFuncGetAttributes(&a, reinterpret_cast<const void*>(plane_local::k_plane_local<float, false, true>));
}

}  // namespace sdft_hip
