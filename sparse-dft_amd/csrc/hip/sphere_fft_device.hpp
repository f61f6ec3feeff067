// Device helpers shared by the kernels of the sphere-restricted FFT pipeline.
#pragma once
#include <hip/hip_runtime.h>

#include "fft_device.hpp"
#include "fft_dispatch.hpp"
#include "fft_lengths.hpp"
#include "lds_barrier.hpp"

namespace sdft_hip {

// Factors above 10 need so many registers that they get kernels of their own;
// the others are compiled without them.
constexpr bool wide_split(int l1, int l2) { return l1 > 10 || l2 > 10; }

// The strided step of a length L1 * L2 line (element i + L1 n, n < L2) whose
// elements lie in [0, low) and [high, L): when the sphere leaves the middle of
// the axis empty, only the first and last kept_digits(L2) values of n occur and
// the DFT drops the others at compile time. An alias-free grid (at least twice
// the sphere's width) always does.
constexpr int kept_digits(int l2) { return (l2 + 1) / 3; }
inline bool half_empty(int l1, int l2, int low, int high) {
  const int kept = kept_digits(l2);
  return 2 * kept < l2 && low <= kept * l1 && high >= (l2 - kept) * l1;
}
template <int L2, bool HALF>
constexpr bool keeps(int n) {
  return !HALF || n < kept_digits(L2) || n >= L2 - kept_digits(L2);
}

// Orders a wave's LDS accesses: they complete in program order, so only the
// compiler has to be kept from moving them.
__device__ __forceinline__ void wave_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// A buffer accessed by 32-bit byte offsets: one past the end (kOutside, or that
// of element -1) reads zero and writes nothing, so a gather needs no branch.
constexpr int kOutside = 1 << 30;
struct BufferView {
  __amdgpu_buffer_rsrc_t rsrc;
  __device__ __forceinline__ BufferView(const void* base, long bytes)
      : rsrc(__builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, int(bytes), 0x00027000)) {}
  __device__ __forceinline__ int load_int(int offset) const {
    return int(__builtin_amdgcn_raw_buffer_load_b32(rsrc, offset, 0, 0));
  }
  // `uniform` is a wave-uniform byte offset added to it
  __device__ __forceinline__ void load(double& v, int offset, int uniform) const {
    v = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(rsrc, offset, uniform, 0));
  }
  __device__ __forceinline__ void load(float& v, int offset, int uniform) const {
    v = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, offset, uniform, 0));
  }
  __device__ __forceinline__ void load(cx<double>& v, int offset, int uniform = 0) const {
    v = __builtin_bit_cast(cx<double>, __builtin_amdgcn_raw_buffer_load_b128(rsrc, offset, uniform, 0));
  }
  __device__ __forceinline__ void load(cx<float>& v, int offset, int uniform = 0) const {
    v = __builtin_bit_cast(cx<float>, __builtin_amdgcn_raw_buffer_load_b64(rsrc, offset, uniform, 0));
  }
  __device__ __forceinline__ void store(cx<double> v, int offset, int uniform = 0) const {
    typedef unsigned u4 __attribute__((ext_vector_type(4)));
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4, v), rsrc, offset, uniform, 0);
  }
  __device__ __forceinline__ void store(cx<float> v, int offset, int uniform = 0) const {
    typedef unsigned u2 __attribute__((ext_vector_type(2)));
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u2, v), rsrc, offset, uniform, 0);
  }
};

// Runs CALL(length, l1, l2) for the case of `length`.
#define SDFT_HIP_LENGTH_SWITCH(LENGTH, CALL) \
  switch (LENGTH) {                          \
    SDFT_HIP_FOR_EACH_LENGTH(CALL)           \
    default:                                 \
      break;                                 \
  }

}  // namespace sdft_hip
