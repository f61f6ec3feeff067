// The z-transforms of the sphere's sticks, both ways (the first and last kernel
// of the local Hamiltonian, and of the density and real-space transforms).
//
// A workgroup takes 256 / max(L1, L2) sticks (64 / max for few columns), so each
// DFT step of the line FFT is one round of its threads: the gather from the
// sphere's coefficients (or from the stick buffer) feeds the registers of the
// first step, the steps meet once in LDS, and the second step stores from
// registers to the stick buffer (or onto the sphere); the loads that only the end
// needs are issued before the exchange. Bound: the scattered 16-byte accesses to the
// coefficients, which the caller keeps in |G| order. Measured alone against moving
// every element through LDS three times, 160 columns of 72^3: into the sticks 71 ->
// 58 us FP64, 65 -> 54 us FP32; back 120 -> 108 and 90 -> 73; 37 columns of
// 70 x 35 x 35 FP64 11 -> 7 and 12 -> 7 (one-wave workgroups).
#include <hip/hip_runtime.h>

#include <type_traits>

#include "local_h.hpp"
#include "sphere_fft.hpp"
#include "sphere_fft_device.hpp"

namespace sdft_hip {
namespace {

template <int L1, int L2>
constexpr int sticks_of(int threads) {
  return threads / (L1 > L2 ? L1 : L2);
}

// x(:, column) gathered into the sticks, natural -> slot order, to
// t1[column][z slot][stick]
template <int L1, int L2, typename T, bool HALF, int NT>
__device__ __forceinline__ void backward(cx<T>* lines, const double* __restrict__ x, long n,
                                         const int* __restrict__ stick_g, int nsticks,
                                         const cx<T>* __restrict__ tw, cx<T>* __restrict__ out) {
  constexpr int S = sticks_of<L1, L2>(NT), L = L1 * L2, LS = L | 1;
  const int tid = threadIdx.x, first = blockIdx.x * S;
  if (first >= nsticks) return;
  {
    const int i = tid % L1, s = tid / L1;
    const bool live = s < S && first + s < nsticks;
    const BufferView index(stick_g + (long)first * L, long(nsticks - first) * L * 4);
    const BufferView in(x, n * 16);
    const int at = live ? (s * L + i) * 4 : kOutside;
    int g[L2];
#pragma unroll
    for (int k = 0; k < L2; ++k)
      if (keeps<L2, HALF>(k)) g[k] = index.load_int(at + k * L1 * 4);
    cx<double> raw[L2];
#pragma unroll
    for (int k = 0; k < L2; ++k)
      if (keeps<L2, HALF>(k)) in.load(raw[k], g[k] * 16);
    cx<T> w[L2];
#pragma unroll
    for (int k = 1; k < L2; ++k) w[k] = tw[i * k];
    cx<T> v[L2];
#pragma unroll
    for (int k = 0; k < L2; ++k) {
      v[k] = cx<T>{T(0), T(0)};
      if (keeps<L2, HALF>(k)) v[k] = cx<T>{T(raw[k].x), T(raw[k].y)};
    }
    if (live) {
      Dft<L2, +1, T>::run(v);
      cx<T>* p = lines + s * LS + i;
      p[0] = v[0];
#pragma unroll
      for (int k = 1; k < L2; ++k) p[k * L1] = cmul_cs(v[k], w[k].x, w[k].y);
    }
  }
  if (NT == 64) wave_fence();
  else lds_barrier();
  const int s = tid % S, b = tid / S;
  if (b < L2 && first + s < nsticks) {
    const cx<T>* p = lines + s * LS + b * L1;
    cx<T> u[L1];
#pragma unroll
    for (int a = 0; a < L1; ++a) u[a] = p[a];
    Dft<L1, +1, T>::run(u);
    cx<T>* o = out + (long)b * L1 * nsticks + first + s;
#pragma unroll
    for (int a = 0; a < L1; ++a) o[(long)a * nsticks] = u[a];
  }
}

// a / b with inv = 1 / b rounded, for a count b: the quotient corrected once by its
// exact residual is the rounded quotient (Markstein, IBM J. Res. Dev. 34, 1990), in
// three operations and a select instead of the compiler's general division. An
// infinite a has no residual (inf - inf): its quotient stands.
__device__ __forceinline__ double divide(double a, double b, double inv) {
  const double q = a * inv;
  const double rounded = __builtin_fma(__builtin_fma(-q, b, a), inv, q);
  return __builtin_isinf(q) ? q : rounded;
}

// t2[column][z slot][stick], slot -> natural order, onto the sphere:
// y = diag .* x + (line value) / count
template <int L1, int L2, typename T, bool HALF, int NT>
__device__ __forceinline__ void forward(cx<T>* lines, const cx<T>* __restrict__ in, const int* __restrict__ stick_g,
                                        int nsticks, const cx<T>* __restrict__ tw, const double* __restrict__ x,
                                        const double* __restrict__ diag, double* __restrict__ y, long n, double count,
                                        double lower) {
  constexpr int S = sticks_of<L1, L2>(NT), L = L1 * L2, LS = L | 1;
  const int tid = threadIdx.x, first = blockIdx.x * S;
  if (first >= nsticks) return;
  const double inv = 1.0 / count;
  const int i = tid % L1, s = tid / L1;
  const bool live = s < S && first + s < nsticks;
  const BufferView index(stick_g + (long)first * L, long(nsticks - first) * L * 4);
  const BufferView xs(x, n * 16), ds(diag, n * 8), ys(y, n * 16);
  const int at = live ? (s * L + i) * 4 : kOutside;
  int g[L2];
#pragma unroll
  for (int k = 0; k < L2; ++k)
    if (keeps<L2, HALF>(k)) g[k] = index.load_int(at + k * L1 * 4);
  {
    const int sg = tid % S, b = tid / S;
    if (b < L2 && first + sg < nsticks) {
      const cx<T>* o = in + (long)b * L1 * nsticks + first + sg;
      cx<T> u[L1];
#pragma unroll
      for (int a = 0; a < L1; ++a) u[a] = o[(long)a * nsticks];
      Dft<L1, -1, T>::run(u);
      cx<T>* p = lines + sg * LS + b * L1;
      p[0] = u[0];
#pragma unroll
      for (int k = 1; k < L1; ++k) {
        const cx<T> w = tw[b * k];
        p[k] = cmul_cs(u[k], w.x, -w.y);
      }
    }
  }
  // the coefficients the results combine with: in flight over the exchange
  cx<double> old[L2];
  double d[L2];
#pragma unroll
  for (int k = 0; k < L2; ++k)
    if (keeps<L2, HALF>(k)) {
      const int e = live ? g[k] : -1;
      xs.load(old[k], e * 16);
      ds.load(d[k], e * 8, 0);
    }
  if (NT == 64) wave_fence();
  else lds_barrier();
  if (live) {
    const cx<T>* p = lines + s * LS + i;
    cx<T> v[L2];
#pragma unroll
    for (int k = 0; k < L2; ++k) v[k] = p[k * L1];
    Dft<L2, -1, T>::run(v);
#pragma unroll
    for (int k = 0; k < L2; ++k)
      if (keeps<L2, HALF>(k)) {
        const double t = d[k] - lower;
        const cx<double> r{t * old[k].x + divide(double(v[k].x), count, inv),
                           t * old[k].y + divide(double(v[k].y), count, inv)};
        ys.store(r, g[k] * 16);
      }
  }
}

// grid (groups of sticks, columns)
template <typename T, bool WIDE, bool HALF, int NT>
__global__ __launch_bounds__(NT) void k_sticks_backward(const double* __restrict__ x, long ldx, long n,
                                                        const int* __restrict__ stick_g, int nsticks, int n2,
                                                        const cx<T>* __restrict__ tw, cx<T>* __restrict__ t1) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  cx<T>* lines = reinterpret_cast<cx<T>*>(smem_raw);
  const long column = blockIdx.y;
  const double* xc = x + 2 * column * ldx;
  cx<T>* out = t1 + column * (long)n2 * nsticks;
#define SDFT_HIP_BACKWARD(L, A, B) \
  case L:                          \
    if constexpr (wide_split(A, B) == WIDE) backward<A, B, T, HALF, NT>(lines, xc, n, stick_g, nsticks, tw, out); \
    break;
  SDFT_HIP_LENGTH_SWITCH(n2, SDFT_HIP_BACKWARD)
#undef SDFT_HIP_BACKWARD
}

template <typename T, bool WIDE, bool HALF, int NT>
__global__ __launch_bounds__(NT) void k_sticks_forward(const cx<T>* __restrict__ t2, const int* __restrict__ stick_g,
                                                       int nsticks, int n2, const cx<T>* __restrict__ tw,
                                                       const double* __restrict__ x, long ldx,
                                                       const double* __restrict__ diag, double* __restrict__ y,
                                                       long ldy, long n, double count,
                                                       const double* __restrict__ shift, double shift_scale) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  cx<T>* lines = reinterpret_cast<cx<T>*>(smem_raw);
  const long column = blockIdx.y;
  const cx<T>* in = t2 + column * (long)n2 * nsticks;
  const double* xc = x + 2 * column * ldx;
  double* yc = y + 2 * column * ldy;
  const double lower = shift ? shift_scale * shift[column] : 0.0;
#define SDFT_HIP_FORWARD(L, A, B) \
  case L:                         \
    if constexpr (wide_split(A, B) == WIDE) forward<A, B, T, HALF, NT>(lines, in, stick_g, nsticks, tw, xc, diag, yc, n, count, lower); \
    break;
  SDFT_HIP_LENGTH_SWITCH(n2, SDFT_HIP_FORWARD)
#undef SDFT_HIP_FORWARD
}

struct StickShape {
  dim3 grid;
  std::size_t lds = 0;
  bool wide = false, half = false, narrow = false;
};

template <typename T>
StickShape stick_shape(const GridPlanDev& p, long columns) {
  StickShape s;
  int l1 = 0, l2 = 0;
  if (!length_split(p.n2, l1, l2)) return s;  // grid.x 0: unsupported
  const int longest = l1 > l2 ? l1 : l2;
  s.wide = wide_split(l1, l2);
  s.half = !s.wide && half_empty(l1, l2, p.zlow, p.zhigh);
  // one-wave workgroups while four-wave ones would number less than two a CU
  // (4 columns of 32^3, FP64: 6.4 -> 4 us in, 8.6 -> 3.3 us back)
  s.narrow = long((p.nsticks + 256 / longest - 1) / (256 / longest)) * columns < 512;
  const int sticks = (s.narrow ? 64 : 256) / longest;
  s.grid = dim3((p.nsticks + sticks - 1) / sticks, (unsigned)columns);
  s.lds = std::size_t(sticks) * line_stride(p.n2) * sizeof(cx<T>);
  return s;
}

// Runs go(bool constants WIDE, HALF, int constant NT) for the shape.
template <typename F>
void for_shape(const StickShape& s, F go) {
  using std::integral_constant;
  if (s.narrow) {
    if (s.wide) go(integral_constant<bool, true>{}, integral_constant<bool, false>{}, integral_constant<int, 64>{});
    else if (s.half) go(integral_constant<bool, false>{}, integral_constant<bool, true>{}, integral_constant<int, 64>{});
    else go(integral_constant<bool, false>{}, integral_constant<bool, false>{}, integral_constant<int, 64>{});
  } else {
    if (s.wide) go(integral_constant<bool, true>{}, integral_constant<bool, false>{}, integral_constant<int, 256>{});
    else if (s.half) go(integral_constant<bool, false>{}, integral_constant<bool, true>{}, integral_constant<int, 256>{});
    else go(integral_constant<bool, false>{}, integral_constant<bool, false>{}, integral_constant<int, 256>{});
  }
}

}  // namespace

template <typename T>
hipError_t launch_sticks_backward(const GridPlanDev& p, const double* x, long ldx, long columns, void* t1,
                                  hipStream_t stream) {
  const StickShape s = stick_shape<T>(p, columns);
  if (!s.grid.x || !s.lds) return hipErrorInvalidConfiguration;
  const cx<T>* tw = reinterpret_cast<const cx<T>*>(sizeof(T) == 8 ? p.tw64[2] : p.tw32[2]);
  for_shape(s, [&](auto wide, auto half, auto nt) {
    hipLaunchKernelGGL((k_sticks_backward<T, wide(), half(), nt()>), s.grid, dim3(nt()), s.lds, stream, x, ldx, p.points,
                       p.stick_g, p.nsticks, p.n2, tw, reinterpret_cast<cx<T>*>(t1));
  });
  return hipGetLastError();
}

template <typename T>
hipError_t launch_sticks_forward(const GridPlanDev& p, const void* t2, long columns, const double* x, long ldx,
                                 const double* diag, double* y, long ldy, hipStream_t stream, const double* shift,
                                 double shift_scale) {
  const StickShape s = stick_shape<T>(p, columns);
  if (!s.grid.x || !s.lds) return hipErrorInvalidConfiguration;
  const cx<T>* tw = reinterpret_cast<const cx<T>*>(sizeof(T) == 8 ? p.tw64[2] : p.tw32[2]);
  for_shape(s, [&](auto wide, auto half, auto nt) {
    hipLaunchKernelGGL((k_sticks_forward<T, wide(), half(), nt()>), s.grid, dim3(nt()), s.lds, stream,
                       reinterpret_cast<const cx<T>*>(t2), p.stick_g, p.nsticks, p.n2, tw, x, ldx, diag, y, ldy,
                       p.points, double(p.count), shift, shift_scale);
  });
  return hipGetLastError();
}

template hipError_t launch_sticks_backward<double>(const GridPlanDev&, const double*, long, long, void*, hipStream_t);
template hipError_t launch_sticks_backward<float>(const GridPlanDev&, const double*, long, long, void*, hipStream_t);
template hipError_t launch_sticks_forward<double>(const GridPlanDev&, const void*, long, const double*, long,
                                                  const double*, double*, long, hipStream_t, const double*, double);
template hipError_t launch_sticks_forward<float>(const GridPlanDev&, const void*, long, const double*, long,
                                                 const double*, double*, long, hipStream_t, const double*, double);

// Loads this file's code object on the calling thread (see module_prime.hpp).
hipError_t prime_module_sticks() {
  hipFuncAttributes a{};
  return hipFuncGetAttributes(&a, reinterpret_cast<const void*>(k_sticks_backward<double, false, true, 256>));
}

}  // namespace sdft_hip
