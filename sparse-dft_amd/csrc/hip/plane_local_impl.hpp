// One xy-plane of the local Hamiltonian per workgroup: the sticks of one z slot
// of one column go in, V(r) is applied in slot order, the sticks come out.
//
// A wave owns whole lines in every stage, so the two steps of a line FFT meet
// through LDS inside the wave and the workgroup needs two barriers per plane:
//
//   y in   the wave gathers the sticks of its x-lines from T1 straight into the
//          registers of the first DFT step (no zeroed plane, no scatter), and
//          leaves the lines in slot order in `rows`, which holds only the x-lines
//          the sphere touches, plus a row of zeros and one that is never read;
//   x      the wave takes C columns of `rows` through a buffer of its own: first
//          step (lines outside the sphere read the zeros), second step, x V,
//          first step of the transform back on the same registers, last step;
//   y out  first step in `rows`, last step from registers straight to T2.
#pragma once
#include "local_h.hpp"
#include "plane_plan.hpp"
#include "sphere_fft.hpp"
#include "sphere_fft_device.hpp"

namespace sdft_hip {
namespace plane_local {

// Lanes of a wave over lines of length L1 * L2: C lines at a time, one lane per
// (line, first digit) in the strided step and per (line, group) in the other.
template <int L1, int L2>
struct WaveLines {
  static constexpr int kLines = 64 / (L1 > L2 ? L1 : L2);
};

// Plane coordinates: `rows` keeps the x-lines [0, low) and [high, n0) of natural
// x, in this order, as rows of stride n1p; row `count` holds zeros.
struct PlaneRows {
  int low, high, count, n1, n1p;
  __device__ __forceinline__ bool holds(int x) const { return x < low || x >= high; }
  __device__ __forceinline__ int row(int x) const { return x < low ? x : x - (high - low); }
  __device__ __forceinline__ int x_of(int r) const { return r < low ? r : r + (high - low); }
};

template <int L1, int L2, typename T, bool HALF>
__device__ __forceinline__ void y_in(cx<T>* rows, const PlaneRows& pr, const BufferView& map, const BufferView& in,
                                     const cx<T>* __restrict__ tw, int wave, int waves, int lane) {
  constexpr int C = WaveLines<L1, L2>::kLines;
  const int i = lane % L1, js = lane / L1;  // strided step: consecutive lanes, consecutive sticks
  const int jg = lane % C, b = lane / C;
  auto sticks = [&](int t, int (&s)[L2]) {
    const int r = t + js;
    const int m = js < C && r < pr.count ? (pr.x_of(r) * pr.n1 + i) * 4 : kOutside;
#pragma unroll
    for (int n = 0; n < L2; ++n)
      if (keeps<L2, HALF>(n)) s[n] = map.load_int(m + n * L1 * 4);
  };
  auto gather = [&](const int (&s)[L2], cx<T> (&v)[L2]) {
#pragma unroll
    for (int n = 0; n < L2; ++n) {
      if (keeps<L2, HALF>(n))
        in.load(v[n], s[n] * int(sizeof(cx<T>)));
      else
        v[n] = cx<T>{T(0), T(0)};
    }
  };
  cx<T> w[L2];
#pragma unroll
  for (int k = 1; k < L2; ++k) w[k] = tw[i * k];
  auto lines = [&](int t, cx<T> (&v)[L2]) {
    const int r = t + js, rg = t + jg;
    if (js < C && r < pr.count) {
      Dft<L2, +1, T>::run(v);
      cx<T>* p = rows + r * pr.n1p + i;
      p[0] = v[0];
#pragma unroll
      for (int k = 1; k < L2; ++k) p[k * L1] = cmul_cs(v[k], w[k].x, w[k].y);
    }
    wave_fence();
    if (b < L2 && rg < pr.count) {
      cx<T>* p = rows + rg * pr.n1p + b * L1;
      cx<T> u[L1];
#pragma unroll
      for (int a = 0; a < L1; ++a) u[a] = p[a];
      Dft<L1, +1, T>::run(u);
#pragma unroll
      for (int a = 0; a < L1; ++a) p[a] = u[a];
    }
  };
  // two sets of lines at a time: the gathers of both are in flight before the
  // first is transformed
  const int step = waves * C;
  for (int t = wave * C; t < pr.count; t += 2 * step) {
    int s0[L2], s1[L2];
    cx<T> v0[L2], v1[L2];
    const bool two = t + step < pr.count;
    sticks(t, s0);
    if (two) sticks(t + step, s1);
    gather(s0, v0);
    if (two) gather(s1, v1);
    lines(t, v0);
    if (two) lines(t + step, v1);
  }
}

template <int L1, int L2, typename T, bool HALF>
__device__ __forceinline__ void x_both(cx<T>* rows, cx<T>* buffer, const PlaneRows& pr, const BufferView& potential,
                                       const cx<T>* __restrict__ tw, int wave, int waves, int lane) {
  constexpr int C = WaveLines<L1, L2>::kLines;
  const int j = lane % C, i = lane / C;
  const int step = waves * C;
  // V of the lane's group in the plane's rows [a + L1 i][y]
  auto load_potential = [&](int t, T (&pot)[L1]) {
    const int y = t + j;
    const int at = i < L2 && y < pr.n1 ? (L1 * i * pr.n1 + y) * int(sizeof(T)) : kOutside;
#pragma unroll
    for (int a = 0; a < L1; ++a) potential.load(pot[a], at, a * pr.n1 * int(sizeof(T)));
  };
  T pot[L1], next[L1];
  load_potential(wave * C, pot);
  cx<T> ws[L2], wg[L1];
#pragma unroll
  for (int k = 1; k < L2; ++k) ws[k] = tw[(i < L1 ? i : 0) * k];
#pragma unroll
  for (int k = 1; k < L1; ++k) wg[k] = tw[(i < L2 ? i : 0) * k];
  // rows of the lane's elements: lines outside the sphere read the row of zeros
  // and write the one after it
  int from[L2], to[L2];
#pragma unroll
  for (int n = 0; n < L2; ++n) {
    const int x = i + L1 * n;
    const bool held = i < L1 && pr.holds(x);
    from[n] = (held ? pr.row(x) : pr.count) * pr.n1p;
    to[n] = (held ? pr.row(x) : pr.count + 1) * pr.n1p;
  }
  lds_barrier();
  for (int t = wave * C; t < pr.n1; t += step) {
    const int y = t + j;
    const bool strided = i < L1 && y < pr.n1, group = i < L2 && y < pr.n1;
    if (t + step < pr.n1) load_potential(t + step, next);
    if (strided) {
      cx<T> v[L2];
#pragma unroll
      for (int n = 0; n < L2; ++n) {
        v[n] = cx<T>{T(0), T(0)};
        if (keeps<L2, HALF>(n)) v[n] = rows[from[n] + y];
      }
      Dft<L2, +1, T>::run(v);
      cx<T>* p = buffer + i * C + j;
      p[0] = v[0];
#pragma unroll
      for (int k = 1; k < L2; ++k) p[k * L1 * C] = cmul_cs(v[k], ws[k].x, ws[k].y);
    }
    wave_fence();
    if (group) {
      cx<T>* p = buffer + i * L1 * C + j;
      cx<T> u[L1];
#pragma unroll
      for (int a = 0; a < L1; ++a) u[a] = p[a * C];
      Dft<L1, +1, T>::run(u);
#pragma unroll
      for (int a = 0; a < L1; ++a) {
        u[a].x *= pot[a];
        u[a].y *= pot[a];
      }
      Dft<L1, -1, T>::run(u);
      p[0] = u[0];
#pragma unroll
      for (int k = 1; k < L1; ++k) p[k * C] = cmul_cs(u[k], wg[k].x, -wg[k].y);
    }
    wave_fence();
    if (strided) {
      const cx<T>* p = buffer + i * C + j;
      cx<T> v[L2];
#pragma unroll
      for (int n = 0; n < L2; ++n) v[n] = p[n * L1 * C];
      Dft<L2, -1, T>::run(v);
#pragma unroll
      for (int n = 0; n < L2; ++n)
        if (keeps<L2, HALF>(n)) rows[to[n] + y] = v[n];
    }
    wave_fence();
#pragma unroll
    for (int a = 0; a < L1; ++a) pot[a] = next[a];
  }
}

template <int L1, int L2, typename T, bool HALF>
__device__ __forceinline__ void y_out(cx<T>* rows, const PlaneRows& pr, const BufferView& map, const BufferView& out,
                                      const cx<T>* __restrict__ tw, int wave, int waves, int lane) {
  constexpr int C = WaveLines<L1, L2>::kLines;
  const int i = lane % L1, js = lane / L1;
  const int jg = lane % C, b = lane / C;
  cx<T> w[L1];
#pragma unroll
  for (int k = 1; k < L1; ++k) w[k] = tw[(b < L2 ? b : 0) * k];
  auto sticks = [&](int t, int (&s)[L2]) {
    const int r = t + js;
    const int m = js < C && r < pr.count ? (pr.x_of(r) * pr.n1 + i) * 4 : kOutside;
#pragma unroll
    for (int n = 0; n < L2; ++n)
      if (keeps<L2, HALF>(n)) s[n] = map.load_int(m + n * L1 * 4);
  };
  const int step = waves * C;
  int s[L2], next[L2];
  if (wave * C < pr.count) sticks(wave * C, s);
  lds_barrier();
  for (int t = wave * C; t < pr.count; t += step) {
    const int r = t + js, rg = t + jg;
    if (t + step < pr.count) sticks(t + step, next);
    if (b < L2 && rg < pr.count) {
      cx<T>* p = rows + rg * pr.n1p + b * L1;
      cx<T> u[L1];
#pragma unroll
      for (int a = 0; a < L1; ++a) u[a] = p[a];
      Dft<L1, -1, T>::run(u);
      p[0] = u[0];
#pragma unroll
      for (int k = 1; k < L1; ++k) p[k] = cmul_cs(u[k], w[k].x, -w[k].y);
    }
    wave_fence();
    if (js < C && r < pr.count) {
      const cx<T>* p = rows + r * pr.n1p + i;
      cx<T> v[L2];
#pragma unroll
      for (int n = 0; n < L2; ++n) v[n] = p[n * L1];
      Dft<L2, -1, T>::run(v);
#pragma unroll
      for (int n = 0; n < L2; ++n)
        if (keeps<L2, HALF>(n)) out.store(v[n], s[n] * int(sizeof(cx<T>)));
    }
#pragma unroll
    for (int n = 0; n < L2; ++n) s[n] = next[n];
  }
}

// grid (n2 z slots, columns). Bound: vector issue in FP32 (96 % of the cycles),
// latency in FP64 (half of them; the registers hold three waves a SIMD, the LDS two of
// them at 72 x 72); HBM carries only the sticks. Measured alone, in-place plane kernel ->
// this one: 160 columns of 72^3 627 -> 308 us FP64 and 301 -> 163 us FP32, 96 columns of
// 48 x 48 x 96 311 -> 121 us FP64, 37 columns of 70 x 35 x 35 56 -> 26 us FP64; without
// the dropped digits, the branch-free gathers, the loads ahead of the barriers and the
// bounds below 371, 186, 238 and 44. HALF, which drops the empty middle, is kept to the
// registers of three waves a SIMD (168 in FP64, six more spilled: 28 bytes a lane; the
// full kernel would spill 46): 222 -> 198 us on 48 x 48 with two of them resident, 121
// with three, unchanged on 72 x 72.
template <typename T, bool WIDE, bool HALF>
__global__ __launch_bounds__(WIDE ? 256 : 512) __attribute__((amdgpu_waves_per_eu(WIDE ? 1 : HALF ? 3 : 2))) void k_plane_local(
    const cx<T>* __restrict__ t1, cx<T>* __restrict__ t2, const int* __restrict__ stick_map, int nsticks, int n0,
    int n1, int n2, const cx<T>* __restrict__ tw_x, const cx<T>* __restrict__ tw_y, const T* __restrict__ v_slots,
    int low, int high, int buffer_elements) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, waves = blockDim.x >> 6;
  const PlaneRows pr{low, high, low + n0 - high, n1, line_stride(n1)};
  cx<T>* rows = reinterpret_cast<cx<T>*>(smem_raw);
  cx<T>* buffer = rows + (pr.count + 2) * pr.n1p + wave * buffer_elements;
  for (int e = threadIdx.x; e < pr.n1p; e += blockDim.x) rows[pr.count * pr.n1p + e] = cx<T>{T(0), T(0)};
  const long plane = (long)blockIdx.y * n2 + blockIdx.x;
  const BufferView map(stick_map, long(n0) * n1 * 4);
  const BufferView in(t1 + plane * nsticks, long(nsticks) * sizeof(cx<T>));
  const BufferView out(t2 + plane * nsticks, long(nsticks) * sizeof(cx<T>));
  const BufferView potential(v_slots + (long)blockIdx.x * n0 * n1, long(n0) * n1 * sizeof(T));
#define SDFT_HIP_Y_IN(L, A, B) \
  case L:                      \
    if constexpr (WIDE || !wide_split(A, B)) y_in<A, B, T, HALF>(rows, pr, map, in, tw_y, wave, waves, lane); \
    break;
#define SDFT_HIP_X(L, A, B) \
  case L:                   \
    if constexpr (WIDE || !wide_split(A, B)) x_both<A, B, T, HALF>(rows, buffer, pr, potential, tw_x, wave, waves, lane); \
    break;
#define SDFT_HIP_Y_OUT(L, A, B) \
  case L:                       \
    if constexpr (WIDE || !wide_split(A, B)) y_out<A, B, T, HALF>(rows, pr, map, out, tw_y, wave, waves, lane); \
    break;
  SDFT_HIP_LENGTH_SWITCH(n1, SDFT_HIP_Y_IN)
  SDFT_HIP_LENGTH_SWITCH(n0, SDFT_HIP_X)
  SDFT_HIP_LENGTH_SWITCH(n1, SDFT_HIP_Y_OUT)
#undef SDFT_HIP_Y_IN
#undef SDFT_HIP_X
#undef SDFT_HIP_Y_OUT
}

// Waves of the kernel that a CU's registers hold (8 where the runtime does not say)
template <typename T, bool WIDE, bool HALF>
int register_waves() {
  static const int waves = [] {
    int groups = 0;
    const void* kernel = reinterpret_cast<const void*>(k_plane_local<T, WIDE, HALF>);
    return hipOccupancyMaxActiveBlocksPerMultiprocessor(&groups, kernel, 256, 0) == hipSuccess && groups > 0 ? 4 * groups : 8;
  }();
  return waves;
}

}  // namespace plane_local

template <typename T>
bool plan_plane_local(const GridPlanDev& p, PlaneLocalPlan& plan) {
  int a0 = 0, b0 = 0, a1 = 0, b1 = 0;
  if (!length_split(p.n0, a0, b0) || !length_split(p.n1, a1, b1)) return false;
  // lines [0, low) and [high, n0) of natural x
  plan.low = 0;
  plan.high = p.n0;
  for (int r = 0; r < 2; ++r) {
    if (!p.xlines[r]) continue;
    if (p.xstart[r] == 0) plan.low = p.xlines[r];
    else if (p.xstart[r] + p.xlines[r] == p.n0) plan.high = p.xstart[r];
    else return false;
  }
  const int rows = plan.low + p.n0 - plan.high;
  if (rows <= 0 || plan.high < plan.low) return false;
  plan.wide = wide_split(a0, b0) || wide_split(a1, b1);
  plan.half = !plan.wide && half_empty(a0, b0, plan.low, plan.high) && half_empty(a1, b1, p.ylow, p.yhigh);
  plan.buffer_elements = p.n0 * (64 / (a0 > b0 ? a0 : b0));
  const std::size_t fixed = std::size_t(rows + 2) * line_stride(p.n1) * sizeof(cx<T>);
  const std::size_t per_wave = std::size_t(plan.buffer_elements) * sizeof(cx<T>);
  const int registers = plan.wide   ? plane_local::register_waves<T, true, false>()
                        : plan.half ? plane_local::register_waves<T, false, true>()
                                    : plane_local::register_waves<T, false, false>();
  plan.waves = plane_group_waves(fixed, per_wave, std::size_t(max_lds_bytes()), registers, plan.wide ? 4 : 8);
  plan.lds_bytes = fixed + std::size_t(plan.waves) * per_wave;
  return plan.waves > 0;
}

template <typename T>
hipError_t launch_plane_local(const GridPlanDev& p, const PlaneLocalPlan& plan, const void* t1, void* t2, long columns,
                              hipStream_t stream) {
  using plane_local::k_plane_local;
  const cx<T>* twx = reinterpret_cast<const cx<T>*>(sizeof(T) == 8 ? p.tw64[0] : p.tw32[0]);
  const cx<T>* twy = reinterpret_cast<const cx<T>*>(sizeof(T) == 8 ? p.tw64[1] : p.tw32[1]);
  const T* v = reinterpret_cast<const T*>(sizeof(T) == 8 ? (const void*)p.v64 : (const void*)p.v32);
  const dim3 grid(p.n2, (unsigned)columns);
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(64 * plan.waves), plan.lds_bytes, stream,
                       reinterpret_cast<const cx<T>*>(t1), reinterpret_cast<cx<T>*>(t2), p.stick_map, p.nsticks, p.n0,
                       p.n1, p.n2, twx, twy, v, plan.low, plan.high, plan.buffer_elements);
  };
  if (plan.wide) go(k_plane_local<T, true, false>);
  else if (plan.half) go(k_plane_local<T, false, true>);
  else go(k_plane_local<T, false, false>);
  return hipGetLastError();
}

}  // namespace sdft_hip
