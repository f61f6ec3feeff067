// Kernels of the sphere-restricted FFT pipeline that local_h.hip chains.
#pragma once
#include <hip/hip_runtime_api.h>

#include <cstddef>

#include "local_h.hpp"

namespace sdft_hip {

// Launch shape of the local Hamiltonian's plane kernel for one grid plan.
struct PlaneLocalPlan {
  int waves = 0;                // waves of a workgroup
  int low = 0, high = 0;        // x-lines [0, low) and [high, n0) hold sticks
  int buffer_elements = 0;      // each wave's exchange buffer
  bool wide = false;            // a register DFT longer than 10 occurs
  bool half = false;            // both axes are empty in the middle (half_empty)
  std::size_t lds_bytes = 0;
};

// False when the plane's active lines and the waves' buffers do not fit the LDS
// of one workgroup (or the lines are no two runs from the ends of the axis).
template <typename T>
bool plan_plane_local(const GridPlanDev& p, PlaneLocalPlan& plan);

// Sticks of every z slot and column through one xy-plane each: y and x
// transforms to slot order, x V(r), and back; t1, t2: [column][z slot][stick].
template <typename T>
hipError_t launch_plane_local(const GridPlanDev& p, const PlaneLocalPlan& plan, const void* t1, void* t2, long columns,
                              hipStream_t stream);

// z-transforms of the sticks: x(:, c) gathered from the sphere into
// t1[column][z slot][stick], and back with y = diag .* x + (transform) / count
// (diag - shift_scale shift[c] in the place of diag with a shift).
template <typename T>
hipError_t launch_sticks_backward(const GridPlanDev& p, const double* x, long ldx, long columns, void* t1,
                                  hipStream_t stream);
template <typename T>
hipError_t launch_sticks_forward(const GridPlanDev& p, const void* t2, long columns, const double* x, long ldx,
                                 const double* diag, double* y, long ldy, hipStream_t stream,
                                 const double* shift = nullptr, double shift_scale = 0);

}  // namespace sdft_hip
