// Householder reduction of a Hermitian matrix to real symmetric tridiagonal
// form in one launch (the Rayleigh-Ritz eigensolve of the block Davidson). Output
// follows LAPACK zhetrd with uplo = 'L' (d, e, tau and the reflector tails
// v(k+2:n) in column k), so that a tridiagonal eigensolver and zunmtr complete the
// decomposition.
//
// Layout: every workgroup keeps the rows g, g + G, g + 2G, ... of the matrix in
// LDS for the whole reduction (the matrix never returns to HBM). Step k starts
// with reflector k formed and p_i = sum_j A_ij v_j of every row i > k published
// together with the pre-update A_{i,k+1}:
//   1. every thread polls the published values of its entries until all have
//      arrived and reduces (tau p)^H v over the workgroup;
//   2. w = tau p - (tau/2)(tau p)^H v v (in registers), the next column for all
//      rows from the published A_{i,k+1}, the rank-2 update of the own rows and
//      |column tail|^2 over the workgroup;
//   3. reflector k + 1 from the new column, formed redundantly by every workgroup
//      (identical code and data, so identical bits everywhere), and the products of
//      step k + 1 on the updated rows with the unscaled column (the scale follows),
//      each published by the wave that formed it.
// The exchange is one memory round trip a column: the values themselves say that
// they have arrived. A word not yet published is all ones (a NaN that is never
// published); three buffers take turns, and a workgroup refills its own
// entries of the one that every other has left, completed before its next
// publication. A workgroup leaves before a step that it would read without publishing
// the next (tridiag_exchange.hpp), so that whoever has all of step k knows that nobody
// reads step k - 1. Waits are bounded: on expiry an abort flag ends every workgroup.
// Every published word is stored and loaded with agent-scope relaxed atomics
// (sc1 accesses, coherent across the XCDs' L2 caches), which needs no L2 write-back
// or invalidate (an agent-scope fence would issue one on every column).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdlib>

#include "tridiag.hpp"
#include "tridiag_exchange.hpp"
#include "wave_sum.hpp"

namespace sdft_hip {
namespace {

constexpr int kThreads = 512;
constexpr int kWaves = kThreads / 64;
constexpr long kSpinLimit = 1L << 20;
constexpr unsigned long long kMissing = ~0ull;  // a published word that has not arrived
constexpr int kWords = 4;  // of one published row: p_i, A_{i,k+1}

// Aligned to 16 bytes: one element is one 128-bit LDS access (the dynamic LDS
// base is declared 16-byte aligned below, past the static variables).
struct alignas(16) Z {
  double x, y;
};
__device__ inline Z zmul(Z a, Z b) { return {a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x}; }
__device__ inline Z zconj(Z a) { return {a.x, -a.y}; }
__device__ inline Z zadd(Z a, Z b) { return {a.x + b.x, a.y + b.y}; }
__device__ inline Z zsub(Z a, Z b) { return {a.x - b.x, a.y - b.y}; }
__device__ inline Z zscale(Z a, double s) { return {a.x * s, a.y * s}; }

__device__ inline double wave_sum(double v) { return wave::sum(v); }

__device__ inline void publish(unsigned long long* slot, Z p, Z c) {
  const double v[kWords] = {p.x, p.y, c.x, c.y};
#pragma unroll
  for (int w = 0; w < kWords; ++w) {
    unsigned long long bits = __builtin_bit_cast(unsigned long long, v[w]);
    if (bits == kMissing) bits = 0x7FF8000000000000ull;  // an input's NaN of all ones becomes the plain one
    __hip_atomic_store(slot + w, bits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

// Polls one row's words until all have arrived; false when the wait expired or
// another workgroup gave up.
__device__ bool receive(const unsigned long long* slot, int* abort_flag, Z& p, Z& c) {
  unsigned long long w[kWords];
  for (long spin = 0;; ++spin) {
#pragma unroll
    for (int u = 0; u < kWords; ++u)
      w[u] = __hip_atomic_load(slot + u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (w[0] != kMissing && w[1] != kMissing && w[2] != kMissing && w[3] != kMissing) break;
    if ((spin & 15) == 15 &&
        __hip_atomic_load(abort_flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != kHetrdRunning)
      return false;
    if (spin > kSpinLimit) {
      __hip_atomic_store(abort_flag, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      return false;
    }
  }
  p = {__builtin_bit_cast(double, w[0]), __builtin_bit_cast(double, w[1])};
  c = {__builtin_bit_cast(double, w[2]), __builtin_bit_cast(double, w[3])};
  return true;
}

// s_waitcnt vmcnt(0) with the other counters unconstrained (gfx9 encoding)
constexpr int kWaitStores = 0x0F70;

// LDS of one workgroup: rpw matrix rows, the current column, the current
// reflector, the staged products of the own rows, wave partials of two sums.
struct HetrdLds {
  Z *rows, *col, *v, *staged, *dot;
  double* norm;
  __device__ HetrdLds(double* base, int n, int rpw) {
    rows = reinterpret_cast<Z*>(base);
    col = rows + size_t(rpw) * n;
    v = col + n;
    staged = v + n;
    dot = staged + rpw;
    norm = reinterpret_cast<double*>(dot + kWaves);
  }
};
size_t lds_bytes(int n, int rpw) {
  return (size_t(rpw) * n + 2 * size_t(n) + size_t(rpw) + kWaves) * sizeof(Z) + kWaves * sizeof(double);
}

// KP entries of a column per thread (n <= KP * kThreads).
template <int KP>
__global__ __launch_bounds__(kThreads) void k_hetrd_lds(const Z* __restrict__ a, long lda, int n, int rpw,
                                                        Z* __restrict__ refl, long ldr, double* __restrict__ d,
                                                        double* __restrict__ e, Z* __restrict__ tau,
                                                        unsigned long long* __restrict__ pub,
                                                        int* __restrict__ abort_flag) {
  extern __shared__ __attribute__((aligned(16))) double lds_raw[];
  __shared__ int expired;
  __shared__ Z first_p;  // tau p of the first row
  const HetrdLds lds(lds_raw, n, rpw);
  const int G = gridDim.x, g = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int out = hetrd_last_group(n, G);  // writes d, e, tau and the reflectors
  auto slot = [&](int step, int row) { return pub + kWords * (size_t(step % kHetrdBuffers) * n + row); };
  auto first_row = [&](int i0) { return hetrd_first_row(G, g, i0); };  // first r with g + r G >= i0

  // Reflector of the column in lds.col at rows c0 + 1 .. n - 1 (LAPACK zlarfg
  // conventions; |tail|^2 as wave partials in lds.norm, the workgroup's barrier
  // passed), this thread's entries of it in vj and its copy in lds.v, the outputs,
  // and the products of the own rows, published for step c0. Returns tau.
  auto reflect = [&](int c0, Z (&vj)[KP]) {
    const int m = n - c0 - 1;
    const Z* col = lds.col;
    double xn2 = 0.;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) xn2 += lds.norm[w];
    const Z alpha = col[1];
    Z t{0., 0.}, scale{0., 0.};
    double beta;
    if (xn2 == 0. && alpha.y == 0.) {
      // column already reduced: H = I - 2 e1 e1^T (beta = -alpha) instead of
      // LAPACK's tau = 0; rocSOLVER zunmtr returned NaN columns for reflector
      // sets with tau = 0 at orders of a few hundred (real tridiagonal inputs)
      beta = -alpha.x;
      t = {2., 0.};
    } else {
      const double nrm = sqrt(alpha.x * alpha.x + alpha.y * alpha.y + xn2);
      beta = alpha.x >= 0. ? -nrm : nrm;
      t = {(beta - alpha.x) / beta, -alpha.y / beta};
      const Z den{alpha.x - beta, alpha.y};  // 1 / (alpha - beta)
      const double dd = den.x * den.x + den.y * den.y;
      scale = {den.x / dd, -den.y / dd};
    }
    // one wave a row: sum_j A_ij col_j over the tail, scaled, plus A_{i,c0+1} (v = 1)
    for (int r = first_row(c0 + 1) + wave; r < rpw; r += kWaves) {
      const int i = g + r * G;
      if (i >= n) break;
      const Z* row = lds.rows + size_t(r) * n + c0;
      Z acc{0., 0.};
      for (int j = 2 + lane; j <= m; j += 64) acc = zadd(acc, zmul(row[j], col[j]));
      acc.x = wave_sum(acc.x);
      acc.y = wave_sum(acc.y);
      if (lane == 0) {
        const Z head = row[1], p = zadd(head, zmul(scale, acc));
        publish(slot(c0, i), p, head);
        lds.staged[r] = p;
      }
    }
#pragma unroll
    for (int q = 0; q < KP; ++q) {
      const int j = tid + q * kThreads;
      if (j < m) {
        vj[q] = j == 0 ? Z{1., 0.} : zmul(col[1 + j], scale);
        lds.v[j] = vj[q];
        if (g == out && j > 0) refl[(c0 + 1 + j) + size_t(c0) * ldr] = vj[q];
      }
    }
    if (g == out && tid == 0) {
      d[c0] = col[0].x;
      e[c0] = beta;
      tau[c0] = t;
    }
    return t;
  };
  // |tail|^2 of the thread's entries of the column at c0 (entry j at row c0 + j) into
  // the wave partials, the entries into lds.col
  auto column = [&](const Z (&cv)[KP], int length) {
    double part = 0.;
#pragma unroll
    for (int q = 0; q < KP; ++q) {
      const int j = tid + q * kThreads;
      if (j < length) {
        lds.col[j] = cv[q];
        if (j >= 2) part += cv[q].x * cv[q].x + cv[q].y * cv[q].y;
      }
    }
    part = wave_sum(part);
    if (lane == 0) lds.norm[wave] = part;
  };

  // row i of the Hermitian input is the conjugate of column i (coalesced read)
  for (int r = 0; r < rpw; ++r) {
    const int i = g + r * G;
    if (i >= n) break;
    for (int j = tid; j < n; j += kThreads) lds.rows[size_t(r) * n + j] = zconj(a[j + size_t(i) * lda]);
  }
  Z cv[KP], vj[KP];
#pragma unroll
  for (int q = 0; q < KP; ++q) {
    const int j = tid + q * kThreads;
    cv[q] = j < n ? a[j] : Z{0., 0.};
  }
  if (tid == 0) expired = 0;
  column(cv, n);
  __syncthreads();
  Z t = reflect(0, vj);
  for (int k = 0; k + 1 < n; ++k) {
    const int m = n - k - 1, first = first_row(k + 1);
    if (!hetrd_reads(n, G, g, k)) return;
    // ---- 1. the published products of every row; partial (tau p)^H v
    Z p[KP], c[KP];
    bool ok = true;
    Z dot{0., 0.};
#pragma unroll
    for (int q = 0; q < KP; ++q) {
      const int j = tid + q * kThreads;
      if (j < m) {
        ok = receive(slot(k, k + 1 + j), abort_flag, p[q], c[q]) && ok;
        p[q] = zmul(t, p[q]);  // tau p
        dot = zadd(dot, zmul(zconj(p[q]), vj[q]));
      }
    }
    dot.x = wave_sum(dot.x);
    dot.y = wave_sum(dot.y);
    if (lane == 0) lds.dot[wave] = dot;
    if (!ok) expired = 1;
    if (tid == 0) first_p = p[0];
    __syncthreads();
    if (expired) return;
    // step k is complete, so nobody reads step k - 1 (hetrd_reads): its buffer is free
    if (tid < rpw && k > 0) {
      const int i = g + tid * G;
      if (i < n && i >= k) {
        unsigned long long* s = slot(k + 2, i);
#pragma unroll
        for (int w = 0; w < kWords; ++w)
          __hip_atomic_store(s + w, kMissing, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
    dot = {0., 0.};
#pragma unroll
    for (int w = 0; w < kWaves; ++w) dot = zadd(dot, lds.dot[w]);
    // ---- 2. w = tau p + a2 v; next column for all rows; rank-2 update of the own rows
    const Z a2 = zscale(zmul(t, dot), -0.5);
    const Z w0c = zconj(zadd(first_p, a2));  // v[0] = 1
    Z wc[KP], vc[KP];
#pragma unroll
    for (int q = 0; q < KP; ++q) {
      const int j = tid + q * kThreads;
      if (j < m) {
        const Z w = zadd(p[q], zmul(a2, vj[q]));
        cv[q] = zsub(c[q], zadd(zmul(vj[q], w0c), w));
        wc[q] = zconj(w);
        vc[q] = zconj(vj[q]);
      }
    }
    for (int r = first; r < rpw; ++r) {
      const int i = g + r * G;
      if (i >= n) break;
      const Z vi = lds.v[i - k - 1];
      const Z wi = zadd(zmul(t, lds.staged[r]), zmul(a2, vi));
      Z* row = lds.rows + size_t(r) * n + (k + 1);
#pragma unroll
      for (int q = 0; q < KP; ++q) {
        const int j = tid + q * kThreads;
        if (j < m) row[j] = zsub(row[j], zadd(zmul(vi, wc[q]), zmul(wi, vc[q])));
      }
    }
    if (k + 2 == n) {
      if (g == out && tid == 0) d[n - 1] = cv[0].x;
      return;
    }
    column(cv, m);
    __builtin_amdgcn_s_waitcnt(kWaitStores);  // the refill, before the next publication
    __syncthreads();
    // ---- 3. next reflector and the products of step k + 1
    t = reflect(k + 1, vj);
  }
}

int max_lds() {
  static int bytes = [] {
    int dev = 0, v = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 65536;
    if (hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess) return 65536;
    return v;
  }();
  return bytes;
}

int device_cus() {
  static int cus = [] {
    int dev = 0, v = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 0;
    if (hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) return 0;
    return v;
  }();
  return cus;
}

// Target rows per workgroup: about 72 workgroups. More of them shorten a
// workgroup's own work but add pollers of every published row. Measured, us per
// column at n = 100 / 160 / 240 / 320 / 380 / 480 / 640: this rule 3.0 / 3.3 / 3.7 /
// 4.1 / 4.2 / 4.7 / 5.0, four rows 3.1 / 3.3 / 3.7 / 4.2 / 4.5 / 4.9 / 5.8, ten rows
// 3.6 / 3.9 / 4.2 / 4.5 / 4.6 / 4.9 / 5.1 (with arrival flags beside the values, two
// more round trips and nine workgroup barriers a column, four rows took 4.8 / 4.9 / 5.0
// / 5.1 / 5.2 / 5.4 / 5.7); SDFT_HIP_HETRD_ROWS overrides. More rows are used when the
// workgroups would outnumber the CUs.
int target_rows_per_group(int n) {
  static const int rows = [] {
    const char* e = std::getenv("SDFT_HIP_HETRD_ROWS");
    return e ? std::atoi(e) : 0;
  }();
  return rows > 0 ? std::min(rows, kThreads) : std::max(1, (n + 71) / 72);
}

// LDS the kernel declares statically (the workgroup reductions of the
// runtime included), which the dynamic slab must leave room for.
size_t static_lds() {
  static const size_t bytes = [] {
    hipFuncAttributes attr{};
    if (hipFuncGetAttributes(&attr, reinterpret_cast<const void*>(k_hetrd_lds<4>)) != hipSuccess) return size_t(4096);
    return size_t(attr.sharedSizeBytes);
  }();
  return bytes;
}
}  // namespace

bool hetrd_plan(int n, int* rows_per_group, int* groups) {
  if (n < 1 || n > kHetrdMaxOrder) return false;
  const int cus = device_cus();
  const size_t total = size_t(max_lds()), fixed = static_lds();
  if (fixed >= total) return false;
  const size_t budget = total - fixed;
  // the target rows per workgroup, as far as its LDS holds them, and at least so
  // many that there is at most one workgroup per CU
  const int least = cus > 0 ? (n + cus - 1) / cus : 1;
  int rpw = std::max(std::min(n, target_rows_per_group(n)), least);
  while (rpw > least && lds_bytes(n, rpw) > budget) --rpw;
  if (lds_bytes(n, rpw) > budget) return false;
  const int g = (n + rpw - 1) / rpw;
  if (cus > 0 && g > cus) return false;
  // every workgroup must be resident at once (each waits for all)
  int per_cu = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, reinterpret_cast<const void*>(k_hetrd_lds<4>), kThreads,
                                                   lds_bytes(n, rpw)) != hipSuccess ||
      per_cu < 1 || (cus > 0 && long(per_cu) * cus < g))
    return false;
  *rows_per_group = rpw;
  *groups = g;
  return true;
}

// the abort flag's line, then the published rows
constexpr size_t kFlagBytes = 64;
size_t hetrd_workspace_bytes(int n) { return kFlagBytes + kHetrdBuffers * kWords * size_t(n) * sizeof(unsigned long long); }

hipError_t launch_hetrd(const double* a, long lda, int n, double* refl, long ldr, double* d, double* e, double* tau,
                        void* workspace, hipStream_t s, bool force_expiry) {
  int rpw = 0, groups = 0;
  if (!hetrd_plan(n, &rpw, &groups)) return hipErrorInvalidValue;
  if (n == 1) {
    // d = Re a; nothing to reduce
    return hipMemcpyAsync(d, a, sizeof(double), hipMemcpyDeviceToDevice, s);
  }
  int* abort_flag = reinterpret_cast<int*>(workspace);
  auto* pub = reinterpret_cast<unsigned long long*>(static_cast<char*>(workspace) + kFlagBytes);
  // one fill: nothing published, nobody gave up (kHetrdRunning)
  hipError_t err = hipMemsetAsync(workspace, 0xFF, hetrd_workspace_bytes(n), s);
  if (err != hipSuccess) return err;
  // host-forced expiry (fault injection): the abort flag is raised before the
  // launch, so workgroups leave at their waits and the result is discarded
  if (force_expiry && (err = hipMemsetAsync(abort_flag, 1, 1, s)) != hipSuccess) return err;
  const Z* az = reinterpret_cast<const Z*>(a);
  Z* rz = reinterpret_cast<Z*>(refl);
  Z* tz = reinterpret_cast<Z*>(tau);
  // A plain launch: the plan keeps the grid within one workgroup per CU, so
  // on an idle device every workgroup is resident; when other work (another
  // stream or process) holds CUs, the bounded wait expires and the caller
  // redoes the solve by divide and conquer. A cooperative launch would
  // instead serialise the device for the reduction, and it is refused when
  // several processes share the device.
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(groups), dim3(kThreads), lds_bytes(n, rpw), s, az, lda, n, rpw, rz, ldr, d, e, tz, pub,
                       abort_flag);
  };
  if (n <= kThreads) go(k_hetrd_lds<1>);
  else if (n <= 2 * kThreads) go(k_hetrd_lds<2>);
  else go(k_hetrd_lds<4>);
  return hipGetLastError();
}

const int* hetrd_abort_flag(const void* workspace, int) { return reinterpret_cast<const int*>(workspace); }

// Loads this file's code object on the calling thread (see module_prime.hpp).
hipError_t prime_module_tridiag() {
  hipFuncAttributes a{};
  return hipFuncGetAttributes(&a, reinterpret_cast<const void*>(k_hetrd_lds<4>));
}

}  // namespace sdft_hip
