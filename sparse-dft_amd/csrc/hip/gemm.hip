// Complex GEMM on CDNA4 matrix cores, column-major with explicit leading
// dimensions (the semantics of src/compute_backend.hpp:21-27):
//   C = op(A) op(B) + beta * D,  op in {Normal, Adjoint},  D may alias C.
// Complex products use three real MFMAs per 16x16x4 block (Gauss form, 25 % fewer
// MFMA cycles than four):
//   P1 = Ar Br, P2 = Ai Bi, P3 = (Ar + Ai)(Br + Bi); re = P1 - P2, im = P3 - P1 - P2.
// FP64 uses v_mfma_f64_16x16x4_f64, FP32 uses v_mfma_f32_16x16x4_f32 (inputs
// stored in FP64 or FP32 are converted while staging into LDS).
// Long contractions (K >> M, N: projections B X, Galerkin slabs) are split
// along K into a workspace and reduced in a fixed order (deterministic).
#include <hip/hip_runtime.h>

#include "gemm.hpp"
#include "gemm_plan.hpp"
#include "lds_barrier.hpp"

#include <algorithm>
#include <type_traits>
#include <vector>

namespace sdft_hip {

namespace {
constexpr int BK = kGemmSlab;  // K of one slab
typedef double d4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));

template <typename T>
struct Acc;
template <>
struct Acc<double> {
  using type = d4;
  static __device__ __forceinline__ d4 mfma(double a, double b, d4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
};
template <>
struct Acc<float> {
  using type = f4;
  static __device__ __forceinline__ f4 mfma(float a, float b, f4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
};

// XCD-aware tile order. Workgroups are dispatched round-robin over the eight
// XCDs (linear id L runs on XCD L % 8), each with its own L2. The bijection
// below hands every XCD a contiguous range of tiles in (split, m, n) order
// with n fastest, so the tiles that share an A panel (and, for a few M tiles,
// a B panel) run on the same XCD and reuse it from that XCD's L2.
constexpr int kXcds = 8;
struct TileId {
  int m, n, split;
};
__device__ __forceinline__ TileId xcd_tile(int mt, int nt, int splits) {
  const int total = mt * nt * splits;
  const int lin = blockIdx.x + mt * (blockIdx.y + nt * blockIdx.z);
  const int xcd = lin % kXcds, slot = lin / kXcds;
  const int per = (total + kXcds - 1) / kXcds;  // tiles of the fuller XCDs
  const int full = total - (per - 1) * kXcds;   // number of XCDs holding `per` tiles
  const int t = xcd < full ? xcd * per + slot : full * per + (xcd - full) * (per - 1) + slot;
  return {(t / nt) % mt, t % nt, t / (nt * mt)};
}

template <typename T>
struct alignas(2 * sizeof(T)) Pair {
  T re, im;
};

// One operand's K slab: TM lines (rows of op(A), columns of op(B)) by BK of K, on
// its way from memory through registers to LDS. ALONG_K: contiguous along K in
// memory, kept [line][k] with an odd stride; otherwise contiguous along the
// lines, kept [k][line]. A thread's elements keep their byte offsets for the
// whole product while the slab's base advances as a scalar. Lines past the edge
// and k past the end read zeros: past the buffer by the hardware's bounds check.
// FAR (a leading dimension over kFarStride): 64-bit offsets and a test instead.
constexpr long kFarStride = 1L << 20;
template <typename T, typename S, bool ALONG_K, int TM, bool FAR>
struct Slab {
  static constexpr int E = TM * BK / 256;
  static_assert(E * 256 == TM * BK, "staging must tile the workgroup");
  static constexpr int STRIDE = ALONG_K ? BK + 1 : TM + (sizeof(T) == 8 ? 2 : 16);
  static constexpr int SIZE = ALONG_K ? TM * STRIDE : BK * STRIDE;
  using Value = typename std::conditional<sizeof(S) == 8, double2, float2>::type;
  using Offset = typename std::conditional<FAR, long, int>::type;
  static constexpr Offset kOut = -16;
  Value reg[E];
  Offset off[E];
  static __device__ __forceinline__ int line_of(int tid, int it) {
    const int e = tid + it * 256;
    return ALONG_K ? e / BK : e % TM;
  }
  static __device__ __forceinline__ int k_of(int tid, int it) {
    const int e = tid + it * 256;
    return ALONG_K ? e % BK : e / TM;
  }
  static __device__ __forceinline__ int at(int line, int k) { return ALONG_K ? line * STRIDE + k : k * STRIDE + line; }
  __device__ __forceinline__ void init(int tid, int lines, long ld) {
#pragma unroll
    for (int it = 0; it < E; ++it) {
      const int l = line_of(tid, it), k = k_of(tid, it);
      off[it] = l < lines ? Offset((ALONG_K ? l * ld + k : k * ld + l) * long(sizeof(Value))) : kOut;
    }
  }
  static __device__ __forceinline__ Value fetch(const S* base, Offset o) {
    if constexpr (FAR) {
      return o >= 0 ? *reinterpret_cast<const Value*>(reinterpret_cast<const char*>(base) + o) : Value{0, 0};
    } else {
      const __amdgpu_buffer_rsrc_t r =
          __builtin_amdgcn_make_buffer_rsrc(const_cast<S*>(base), 0, 0x7fffffff, 0x00027000);
      if constexpr (sizeof(S) == 8)
        return __builtin_bit_cast(Value, __builtin_amdgcn_raw_buffer_load_b128(r, o, 0, 0));
      else
        return __builtin_bit_cast(Value, __builtin_amdgcn_raw_buffer_load_b64(r, o, 0, 0));
    }
  }
  // `rest`: K left from the slab's start
  __device__ __forceinline__ void load(const S* base, int tid, int rest) {
    if (rest >= BK) {
#pragma unroll
      for (int it = 0; it < E; ++it) reg[it] = fetch(base, off[it]);
    } else {
#pragma unroll
      for (int it = 0; it < E; ++it) reg[it] = fetch(base, k_of(tid, it) < rest ? off[it] : kOut);
    }
  }
  template <bool CONJ>
  __device__ __forceinline__ void store(Pair<T>* lds, int tid) {
#pragma unroll
    for (int it = 0; it < E; ++it)
      lds[at(line_of(tid, it), k_of(tid, it))] = Pair<T>{T(reg[it].x), CONJ ? -T(reg[it].y) : T(reg[it].y)};
  }
};

// One TBM x TBN output tile per 256-thread workgroup (2 x 2 waves), K range
// [k0, k1) of this split. Each wave computes (TBM/2) x (TBN/2) as 16 x 16 blocks:
// per 4-deep K step one LDS read an operand block (re and im together) and three
// MFMAs a block pair, independent accumulators first. Two LDS slabs: while one is
// multiplied, the next travels from memory to registers and then into the other,
// with one barrier a slab. The MFMA takes the operands exchanged (C^T = B^T A^T),
// so that a lane's results lie along M: stores of 256 contiguous bytes.
// Bound: FP64 by the MFMA rate at the clock that FP64 MFMA load leaves (near
// 2.0 GHz; the matrix cores are busy in 72 to 77 % of the cycles of the 64-atom
// products, 67 % in FP32). WAVES: at least that many waves per SIMD.
template <typename T, typename TA, typename TB, bool ADJ_A, bool ADJ_B, int TBM, int TBN, bool FAR, int WAVES>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(WAVES))) void k_zgemm(
    int M, int N, int K, const TA* __restrict__ A, long lda, const TB* __restrict__ B, long ldb, GemmOutput first,
    GemmOutput second, int n_first, double alpha, int kps, double* __restrict__ work) {
  constexpr int IM = TBM / 32, JN = TBN / 32;
  using V = typename Acc<T>::type;
  using SlabA = Slab<T, TA, ADJ_A, TBM, FAR>;
  using SlabB = Slab<T, TB, !ADJ_B, TBN, FAR>;
  __shared__ Pair<T> lds_a[2][SlabA::SIZE];
  __shared__ Pair<T> lds_b[2][SlabB::SIZE];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const TileId tile = xcd_tile(gridDim.x, gridDim.y, gridDim.z);
  const int m0 = tile.m * TBM, n0 = tile.n * TBN;
  const int k0 = tile.split * kps, k1 = min(K, k0 + kps);
  const int wm = (wave & 1) * IM * 16, wn = (wave >> 1) * JN * 16;
  // acc_re = sum Ar Br, acc_x = sum Ai Bi, acc_im = sum (Ar + Ai)(Br + Bi)
  V acc_re[IM][JN], acc_im[IM][JN], acc_x[IM][JN];
#pragma unroll
  for (int i = 0; i < IM; ++i)
#pragma unroll
    for (int j = 0; j < JN; ++j) acc_re[i][j] = acc_im[i][j] = acc_x[i][j] = V{0, 0, 0, 0};
  SlabA sa;
  SlabB sb;
  sa.init(tid, M - m0, lda);
  sb.init(tid, N - n0, ldb);
  const TA* pa = A + 2 * (ADJ_A ? (long)m0 * lda + k0 : m0 + (long)k0 * lda);
  const TB* pb = B + 2 * (ADJ_B ? n0 + (long)k0 * ldb : (long)n0 * ldb + k0);
  const long step_a = 2 * (ADJ_A ? (long)BK : BK * lda), step_b = 2 * (ADJ_B ? BK * ldb : (long)BK);
  sa.load(pa, tid, k1 - k0);
  sb.load(pb, tid, k1 - k0);
  sa.template store<ADJ_A>(lds_a[0], tid);
  sb.template store<ADJ_B>(lds_b[0], tid);
  lds_barrier();
  int buffer = 0;
  for (int kb = k0; kb < k1; kb += BK) {
    const bool more = kb + BK < k1;
    if (more) {
      pa += step_a;
      pb += step_b;
      sa.load(pa, tid, k1 - kb - BK);
      sb.load(pb, tid, k1 - kb - BK);
    }
    const Pair<T>* la = lds_a[buffer];
    const Pair<T>* lb = lds_b[buffer];
#pragma unroll
    for (int ks = 0; ks < BK; ks += 4) {
      const int kr = ks + (lane >> 4), c = lane & 15;
      Pair<T> a[IM], b[JN];
#pragma unroll
      for (int i = 0; i < IM; ++i) a[i] = la[SlabA::at(wm + 16 * i + c, kr)];
#pragma unroll
      for (int j = 0; j < JN; ++j) b[j] = lb[SlabB::at(wn + 16 * j + c, kr)];
#pragma unroll
      for (int i = 0; i < IM; ++i)
#pragma unroll
        for (int j = 0; j < JN; ++j) {
          acc_re[i][j] = Acc<T>::mfma(b[j].re, a[i].re, acc_re[i][j]);
          acc_x[i][j] = Acc<T>::mfma(b[j].im, a[i].im, acc_x[i][j]);
        }
#pragma unroll
      for (int i = 0; i < IM; ++i)
#pragma unroll
        for (int j = 0; j < JN; ++j)
          acc_im[i][j] = Acc<T>::mfma(b[j].re + b[j].im, a[i].re + a[i].im, acc_im[i][j]);
    }
    if (more) {
      buffer ^= 1;
      sa.template store<ADJ_A>(lds_a[buffer], tid);
      sb.template store<ADJ_B>(lds_b[buffer], tid);
      lds_barrier();
    }
  }
  // Accumulator layout of each 16x16 block (columns of C^T = rows of C along the
  // lanes, lane % 16): f32 register r holds column 4*(lane/16) + r of C, f64
  // column 4*r + lane/16
#pragma unroll
  for (int i = 0; i < IM; ++i)
#pragma unroll
    for (int j = 0; j < JN; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = m0 + wm + 16 * i + (lane & 15);
        const int n = n0 + wn + 16 * j + (sizeof(T) == 8 ? 4 * r + (lane >> 4) : 4 * (lane >> 4) + r);
        if (m >= M || n >= N) continue;
        const double p1 = double(acc_re[i][j][r]), p2 = double(acc_x[i][j][r]);
        double re = (p1 - p2) * alpha, im = (double(acc_im[i][j][r]) - p1 - p2) * alpha;
        if (work) {
          *reinterpret_cast<double2*>(work + 2 * ((long)tile.split * M * N + m + (long)n * M)) = double2{re, im};
        } else {
          const bool one = n < n_first;
          const GemmOutput& o = one ? first : second;
          const long column = one ? n : n - n_first;
          if (o.beta != 0.0) {
            const double2 d = *reinterpret_cast<const double2*>(o.D + 2 * (m + column * o.ldd));
            re += o.beta * d.x;
            im += o.beta * d.y;
          }
          *reinterpret_cast<double2*>(o.C + 2 * (m + column * o.ldc)) = double2{re, im};
        }
      }
}

__global__ void k_splitk_reduce(int M, int N, int splits, const double* __restrict__ work, GemmOutput first,
                                GemmOutput second, int n_first) {
  // partials already carry alpha
  const long total = (long)M * N;
  for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < total; e += (long)gridDim.x * blockDim.x) {
    const int m = int(e % M);
    const long n = e / M;
    // partials summed in split order (deterministic); eight loads issued
    // ahead of their additions
    double re = 0, im = 0;
    int s = 0;
    for (; s + 8 <= splits; s += 8) {
      double2 v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = *reinterpret_cast<const double2*>(work + 2 * ((long)(s + u) * total + e));
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        re += v[u].x;
        im += v[u].y;
      }
    }
    for (; s < splits; ++s) {
      const double* w = work + 2 * ((long)s * total + e);
      re += w[0];
      im += w[1];
    }
    const bool one = n < n_first;
    const GemmOutput& o = one ? first : second;
    const long column = one ? n : n - n_first;
    if (o.beta != 0.0) {
      const double* d = o.D + 2 * (m + column * o.ldd);
      re += o.beta * d[0];
      im += o.beta * d[1];
    }
    double* c = o.C + 2 * (m + column * o.ldc);
    c[0] = re;
    c[1] = im;
  }
}

// Per-atom onsite products W[:, 0:m] = D_a P_a, W[:, m:2m] = Q_a P_a.
// FP64: compensated (TwoSum of FMA-exact products) in the scalar order of
// src/paw_compensated_product.hpp:41-56; FP32: plain products.
__global__ void k_atom_blocks_comp(int np, int columns, int atoms, const int* __restrict__ atom_offset,
                                   const int* __restrict__ atom_rows, const long* __restrict__ block_offset,
                                   const double* __restrict__ dblk, const double* __restrict__ qblk,
                                   const double* __restrict__ P, long ldp, double* __restrict__ W, long ldw,
                                   int which_mask) {
#pragma clang fp contract(off)
  const long total = (long)np * columns * 2;
  for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < total; e += (long)gridDim.x * blockDim.x) {
    const int row = int(e % np);
    const long rest = e / np;
    const int col = int(rest % columns);
    const int which = int(rest / columns);  // 0: D, 1: Q
    if (!((which_mask >> which) & 1)) continue;
    // find the atom of this row (atoms are few; linear scan over offsets)
    int a = 0;
    while (a + 1 < atoms && atom_offset[a + 1] <= row) ++a;
    const int r = atom_rows[a], o = atom_offset[a], i = row - o;
    const double* blk = (which ? qblk : dblk) + 2 * block_offset[a];  // column-major r x r
    double rs = 0, rc = 0, is = 0, ic = 0;
    auto add = [](double v, double& s, double& c) {
      const double next = s + v;
      const double back = next - s;
      c += (s - (next - back)) + (v - back);
      s = next;
    };
    auto product = [&](double x, double y, double& s, double& c) {
      const double rounded = x * y;
      add(rounded, s, c);
      add(__builtin_fma(x, y, -rounded), s, c);
    };
    const double* pc = P + 2 * (o + (long)col * ldp);
    for (int k = 0; k < r; ++k) {
      const double lr = blk[2 * (i + k * r)], li = blk[2 * (i + k * r) + 1];
      const double pr = pc[2 * k], pi = pc[2 * k + 1];
      product(lr, pr, rs, rc);
      product(-li, pi, rs, rc);
      product(lr, pi, is, ic);
      product(li, pr, is, ic);
    }
    double* w = W + 2 * (row + ((long)which * columns + col) * ldw);
    w[0] = rs + rc;
    w[1] = is + ic;
  }
}

__global__ void k_atom_blocks_f32(int np, int columns, int atoms, const int* __restrict__ atom_offset,
                                  const int* __restrict__ atom_rows, const long* __restrict__ block_offset,
                                  const double* __restrict__ dblk, const double* __restrict__ qblk,
                                  const double* __restrict__ P, long ldp, double* __restrict__ W, long ldw,
                                  int which_mask) {
  const long total = (long)np * columns * 2;
  for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < total; e += (long)gridDim.x * blockDim.x) {
    const int row = int(e % np);
    const long rest = e / np;
    const int col = int(rest % columns);
    const int which = int(rest / columns);
    if (!((which_mask >> which) & 1)) continue;
    int a = 0;
    while (a + 1 < atoms && atom_offset[a + 1] <= row) ++a;
    const int r = atom_rows[a], o = atom_offset[a], i = row - o;
    const double* blk = (which ? qblk : dblk) + 2 * block_offset[a];
    const double* pc = P + 2 * (o + (long)col * ldp);
    float re = 0.f, im = 0.f;
    for (int k = 0; k < r; ++k) {
      const float lr = float(blk[2 * (i + k * r)]), li = float(blk[2 * (i + k * r) + 1]);
      const float pr = float(pc[2 * k]), pi = float(pc[2 * k + 1]);
      re += lr * pr - li * pi;
      im += lr * pi + li * pr;
    }
    double* w = W + 2 * (row + ((long)which * columns + col) * ldw);
    w[0] = re;
    w[1] = im;
  }
}

unsigned reduce_blocks(int M, int N) { return unsigned(std::min<long>(1024, (long(M) * N + 255) / 256)); }

template <typename T, typename TA, typename TB, int CFG, bool FAR>
hipError_t launch_cfg(int aop, int bop, dim3 grid, int M, int N, int K, const TA* A, long lda, const TB* B, long ldb,
                      const GemmOutput& first, const GemmOutput& second, int n_first, double alpha, int kps,
                      double* work, hipStream_t s) {
  constexpr int TBM = kTiles[CFG].bm, TBN = kTiles[CFG].bn;
  constexpr int WAVES = sizeof(T) == 4 && CFG == 0 ? 3 : 2;
#define SDFT_LAUNCH(AA, BB)                                                                                         \
  hipLaunchKernelGGL((k_zgemm<T, TA, TB, AA, BB, TBM, TBN, FAR, WAVES>), grid, dim3(256), 0, s, M, N, K, A, lda, B, \
                     ldb, first, second, n_first, alpha, kps, work)
  if (!aop && !bop) SDFT_LAUNCH(false, false);
  else if (aop && !bop) SDFT_LAUNCH(true, false);
  else if (!aop && bop) SDFT_LAUNCH(false, true);
  else SDFT_LAUNCH(true, true);
#undef SDFT_LAUNCH
  return hipGetLastError();
}

template <typename T, typename TA, typename TB>
hipError_t dispatch_ops(int cfg, int aop, int bop, dim3 grid, int M, int N, int K, const TA* A, long lda, const TB* B,
                        long ldb, const GemmOutput& first, const GemmOutput& second, int n_first, double alpha, int kps,
                        double* work, hipStream_t s, const LaunchEvents* ev) {
  if (ev && ev->begin) {
    const hipError_t e = hipEventRecord(ev->begin, s);
    if (e != hipSuccess) return e;
  }
  hipError_t e;
  if (lda > kFarStride || ldb > kFarStride) {
    // 32-bit byte offsets do not reach a tile's last line: 64-bit ones, 32 x 32
    const dim3 far((M + 31) / 32, (N + 31) / 32, grid.z);
    e = launch_cfg<T, TA, TB, 0, true>(aop, bop, far, M, N, K, A, lda, B, ldb, first, second, n_first, alpha, kps, work, s);
  } else if (cfg == 2) {
    e = launch_cfg<T, TA, TB, 2, false>(aop, bop, grid, M, N, K, A, lda, B, ldb, first, second, n_first, alpha, kps, work, s);
  } else if (cfg == 1) {
    e = launch_cfg<T, TA, TB, 1, false>(aop, bop, grid, M, N, K, A, lda, B, ldb, first, second, n_first, alpha, kps, work, s);
  } else {
    e = launch_cfg<T, TA, TB, 0, false>(aop, bop, grid, M, N, K, A, lda, B, ldb, first, second, n_first, alpha, kps, work, s);
  }
  if (e != hipSuccess || !ev || !ev->end) return e;
  return hipEventRecord(ev->end, s);
}

// The launch of a plan; without a workspace the product is not split.
struct Launch {
  int cfg, splits, kps;
  dim3 grid;
};
Launch launch_for(const GemmPlan& plan, int M, int N, int K, bool have_work) {
  Launch p{};
  p.cfg = plan.cfg;
  p.kps = have_work ? plan.kps : gemm_k_per_split(K, 1);
  p.splits = (K + p.kps - 1) / p.kps;
  p.grid = dim3((M + kTiles[p.cfg].bm - 1) / kTiles[p.cfg].bm, (N + kTiles[p.cfg].bn - 1) / kTiles[p.cfg].bn,
                p.splits);
  return p;
}
}  // namespace

int zgemm_real_products(Precision) { return 3; }

std::size_t zgemm_workspace_bytes(int M, int N, int K) {
  const int splits = zgemm_splits(M, N, K);
  return splits > 1 ? std::size_t(splits) * M * N * 16 : 0;
}

// FP64 splits at least as often as FP32
int zgemm_splits(int M, int N, int K) { return K > 0 ? gemm_plan(true, M, N, K).splits : 1; }

namespace {
template <typename T, typename TA>
hipError_t run(int aop, int bop, int M, int N, int K, double alpha, const TA* A, long lda, const double* B, long ldb,
               const GemmOutput& first, const GemmOutput& second, int n_first, double* work, std::size_t work_bytes,
               hipStream_t s, const LaunchEvents* ev, int* partials) {
  const bool room = work != nullptr && work_bytes >= zgemm_workspace_bytes(M, N, K);
  const Launch pl = launch_for(gemm_plan(sizeof(T) == 8, M, N, K), M, N, K, room);
  double* wk = pl.splits > 1 ? work : nullptr;
  const hipError_t e = dispatch_ops<T, TA, double>(pl.cfg, aop, bop, pl.grid, M, N, K, A, lda, B, ldb, first, second,
                                                   n_first, alpha, pl.kps, wk, s, ev);
  if (partials) *partials = pl.splits;
  if (e != hipSuccess || pl.splits == 1 || partials) return e;
  hipLaunchKernelGGL(k_splitk_reduce, dim3(reduce_blocks(M, N)), dim3(256), 0, s, M, N, pl.splits, work, first, second,
                     n_first);
  return hipGetLastError();
}
}  // namespace

hipError_t zgemm(Precision prec, int aop, int bop, int M, int N, int K, double alpha, const double* A, long lda,
                 const double* B, long ldb, double* C, long ldc, const double* D, long ldd, double beta, double* work,
                 std::size_t work_bytes, hipStream_t s, const LaunchEvents* ev, int* partials) {
  if (M <= 0 || N <= 0) return hipSuccess;
  if (K <= 0) {
    // C = beta * D
    if (partials) *partials = 1;
    return launch_zaxpby(M, N, 0.0, nullptr, 0, beta, D, ldd, C, ldc, s);
  }
  const GemmOutput o{C, ldc, D, ldd, beta};
  return prec == Precision::FP64
             ? run<double, double>(aop, bop, M, N, K, alpha, A, lda, B, ldb, o, o, N, work, work_bytes, s, ev, partials)
             : run<float, double>(aop, bop, M, N, K, alpha, A, lda, B, ldb, o, o, N, work, work_bytes, s, ev, partials);
}

hipError_t zgemm_f32_storage(int aop, int bop, int M, int N, int K, double alpha, const float* A, long lda,
                             const double* B, long ldb, double* C, long ldc, const double* D, long ldd, double beta,
                             double* work, std::size_t work_bytes, hipStream_t s, const LaunchEvents* ev,
                             int* partials) {
  if (M <= 0 || N <= 0 || K <= 0) return hipSuccess;
  const GemmOutput o{C, ldc, D, ldd, beta};
  return run<float, float>(aop, bop, M, N, K, alpha, A, lda, B, ldb, o, o, N, work, work_bytes, s, ev, partials);
}

hipError_t zgemm_two_outputs(int aop, int M, int n_first, int n_second, int K, const double* A, long lda,
                             const double* B, long ldb, const GemmOutput& first, const GemmOutput& second, double* work,
                             std::size_t work_bytes, hipStream_t s, const LaunchEvents* ev) {
  if (M <= 0 || n_first <= 0 || n_second <= 0 || K <= 0) return hipErrorInvalidValue;
  return run<double, double>(aop, 0, M, n_first + n_second, K, 1.0, A, lda, B, ldb, first, second, n_first, work,
                             work_bytes, s, ev, nullptr);
}
hipError_t zgemm_two_outputs(int aop, int M, int n_first, int n_second, int K, const float* A, long lda,
                             const double* B, long ldb, const GemmOutput& first, const GemmOutput& second, double* work,
                             std::size_t work_bytes, hipStream_t s, const LaunchEvents* ev) {
  if (M <= 0 || n_first <= 0 || n_second <= 0 || K <= 0) return hipErrorInvalidValue;
  return run<float, float>(aop, 0, M, n_first + n_second, K, 1.0, A, lda, B, ldb, first, second, n_first, work,
                           work_bytes, s, ev, nullptr);
}

// ---- BF16 projector products (search arithmetic) ----
// C = alpha op(A) B + beta D with A the projector block stored as BF16 complex
// pairs (real part in the low 16 bits), B and C / D stored in FP64, products on
// v_mfma_f32_16x16x32_bf16 with FP32 accumulation. Lane l of that instruction
// holds 8 consecutive k of row (A) / column (B) l % 16, starting at
// k = 8 (l / 16); its accumulators are laid out as the f32 16x16 ones
// (register r: row 4 (l / 16) + r, column l % 16). Four real products per
// complex block: at BF16 precision the sums of the three-product form would
// lose the imaginary part to cancellation. One 128 x 32 tile per 256-thread
// workgroup, 4 waves of 32 x 32 along M, K slabs of 32 staged in LDS as
// [row][k] with a row stride of 40 elements (80 bytes, so the 8-element
// operand reads are aligned 16-byte LDS reads), the next slab prefetched into
// registers.
namespace {
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef short s8v __attribute__((ext_vector_type(8)));
constexpr int BKH = 32, SHB = BKH + 8, HTBM = 128, HTBN = 32;

__device__ __forceinline__ __bf16 bf16_from_bits(unsigned short b) { return __builtin_bit_cast(__bf16, b); }
__device__ __forceinline__ bf8 bf8_negate(bf8 v) {
  s8v bits = __builtin_bit_cast(s8v, v);
  bits ^= s8v{short(0x8000), short(0x8000), short(0x8000), short(0x8000), short(0x8000), short(0x8000),
              short(0x8000), short(0x8000)};
  return __builtin_bit_cast(bf8, bits);
}

template <bool ADJ_A>
__global__ __launch_bounds__(256) void k_zgemm_bf16(int M, int N, int K, const unsigned* __restrict__ A, long lda,
                                                    const double* __restrict__ B, long ldb, double* __restrict__ C,
                                                    long ldc, const double* __restrict__ D, long ldd, double alpha,
                                                    double beta, int kps, double* __restrict__ work) {
  constexpr int WGM = 4, WM = HTBM / WGM, WN = HTBN, IM = WM / 16, JN = WN / 16;
  constexpr int EA = HTBM * BKH / 256, EB = HTBN * BKH / 256;
  __shared__ __attribute__((aligned(16))) __bf16 as_re[HTBM * SHB];
  __shared__ __attribute__((aligned(16))) __bf16 as_im[HTBM * SHB];
  __shared__ __attribute__((aligned(16))) __bf16 bs_re[HTBN * SHB];
  __shared__ __attribute__((aligned(16))) __bf16 bs_im[HTBN * SHB];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const TileId tile = xcd_tile(gridDim.x, gridDim.y, gridDim.z);
  const int m0 = tile.m * HTBM, n0 = tile.n * HTBN;
  const int k0 = tile.split * kps, k1 = min(K, k0 + kps);
  const int wm = wave * WM;
  f4 acc_re[IM][JN], acc_im[IM][JN];
#pragma unroll
  for (int i = 0; i < IM; ++i)
#pragma unroll
    for (int j = 0; j < JN; ++j) {
      acc_re[i][j] = f4{0, 0, 0, 0};
      acc_im[i][j] = f4{0, 0, 0, 0};
    }
  unsigned pa[EA];
  double2 pb[EB];
  auto load = [&](int kb) {
#pragma unroll
    for (int it = 0; it < EA; ++it) {
      const int e = tid + it * 256;
      int mm, kk;
      if (!ADJ_A) { mm = e % HTBM; kk = e / HTBM; } else { kk = e % BKH; mm = e / BKH; }
      const int m = m0 + mm, k = kb + kk;
      pa[it] = (m < M && k < k1) ? (ADJ_A ? A[k + (long)m * lda] : A[m + (long)k * lda]) : 0u;
    }
#pragma unroll
    for (int it = 0; it < EB; ++it) {
      const int e = tid + it * 256;
      const int kk = e % BKH, nn = e / BKH;
      const int n = n0 + nn, k = kb + kk;
      pb[it] = (n < N && k < k1) ? *reinterpret_cast<const double2*>(B + 2 * (k + (long)n * ldb)) : double2{0, 0};
    }
  };
  auto store = [&]() {
#pragma unroll
    for (int it = 0; it < EA; ++it) {
      const int e = tid + it * 256;
      int mm, kk;
      if (!ADJ_A) { mm = e % HTBM; kk = e / HTBM; } else { kk = e % BKH; mm = e / BKH; }
      // op(A) = A^H conjugates: flip the sign bit of the imaginary part
      const unsigned short re = (unsigned short)(pa[it] & 0xffffu);
      const unsigned short im = (unsigned short)((pa[it] >> 16) ^ (ADJ_A ? 0x8000u : 0u));
      as_re[mm * SHB + kk] = bf16_from_bits(re);
      as_im[mm * SHB + kk] = bf16_from_bits(im);
    }
#pragma unroll
    for (int it = 0; it < EB; ++it) {
      const int e = tid + it * 256;
      const int kk = e % BKH, nn = e / BKH;
      bs_re[nn * SHB + kk] = __bf16(float(pb[it].x));
      bs_im[nn * SHB + kk] = __bf16(float(pb[it].y));
    }
  };
  if (k0 < k1) load(k0);
  for (int kb = k0; kb < k1; kb += BKH) {
    store();
    __syncthreads();
    if (kb + BKH < k1) load(kb + BKH);
    const int r = lane & 15, ko = 8 * (lane >> 4);
    bf8 ar[IM], ai[IM], br[JN], bi[JN], nbi[JN];
#pragma unroll
    for (int i = 0; i < IM; ++i) {
      ar[i] = *reinterpret_cast<const bf8*>(&as_re[(wm + 16 * i + r) * SHB + ko]);
      ai[i] = *reinterpret_cast<const bf8*>(&as_im[(wm + 16 * i + r) * SHB + ko]);
    }
#pragma unroll
    for (int j = 0; j < JN; ++j) {
      br[j] = *reinterpret_cast<const bf8*>(&bs_re[(16 * j + r) * SHB + ko]);
      bi[j] = *reinterpret_cast<const bf8*>(&bs_im[(16 * j + r) * SHB + ko]);
      nbi[j] = bf8_negate(bi[j]);
    }
#pragma unroll
    for (int i = 0; i < IM; ++i)
#pragma unroll
      for (int j = 0; j < JN; ++j) {
        acc_re[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ar[i], br[j], acc_re[i][j], 0, 0, 0);
        acc_im[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ar[i], bi[j], acc_im[i][j], 0, 0, 0);
      }
#pragma unroll
    for (int i = 0; i < IM; ++i)
#pragma unroll
      for (int j = 0; j < JN; ++j) {
        acc_re[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ai[i], nbi[j], acc_re[i][j], 0, 0, 0);
        acc_im[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ai[i], br[j], acc_im[i][j], 0, 0, 0);
      }
    __syncthreads();
  }
  const bool split = work != nullptr;
#pragma unroll
  for (int i = 0; i < IM; ++i)
#pragma unroll
    for (int j = 0; j < JN; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = m0 + wm + 16 * i + 4 * (lane >> 4) + r;
        const int n = n0 + 16 * j + (lane & 15);
        if (m >= M || n >= N) continue;
        double re = alpha * double(acc_re[i][j][r]), im = alpha * double(acc_im[i][j][r]);
        if (split) {
          double* w = work + 2 * ((long)tile.split * M * N + m + (long)n * M);
          w[0] = re;
          w[1] = im;
        } else {
          if (beta != 0.0) {
            const double* d = D + 2 * (m + (long)n * ldd);
            re += beta * d[0];
            im += beta * d[1];
          }
          double* c = C + 2 * (m + (long)n * ldc);
          c[0] = re;
          c[1] = im;
        }
      }
}

// FP32 / FP64 complex pairs -> BF16 pairs (round to nearest even)
template <typename S>
__global__ void k_to_bf16_pairs(const S* __restrict__ x, long count, unsigned* __restrict__ out) {
  for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < count; e += (long)gridDim.x * blockDim.x) {
    const unsigned short re = __builtin_bit_cast(unsigned short, __bf16(float(x[2 * e])));
    const unsigned short im = __builtin_bit_cast(unsigned short, __bf16(float(x[2 * e + 1])));
    out[e] = unsigned(re) | (unsigned(im) << 16);
  }
}
}  // namespace

hipError_t zgemm_bf16_storage(int aop, int M, int N, int K, double alpha, const unsigned* A, long lda,
                              const double* B, long ldb, double* C, long ldc, const double* D, long ldd, double beta,
                              double* work, std::size_t work_bytes, hipStream_t s, const LaunchEvents* ev,
                              int* partials) {
  if (M <= 0 || N <= 0 || K <= 0) return hipSuccess;
  const long tiles = long((M + HTBM - 1) / HTBM) * ((N + HTBN - 1) / HTBN);
  // long contractions split along K to >= 512 workgroups, within the workspace
  int splits = 1;
  while (tiles * splits < 512 && long(K) / (2 * splits) >= 256 && splits < 64) splits *= 2;
  while (splits > 1 && (!work || std::size_t(splits) * M * N * 16 > work_bytes)) splits /= 2;
  int kps = (K + splits - 1) / splits;
  kps = ((kps + BKH - 1) / BKH) * BKH;
  splits = (K + kps - 1) / kps;
  const dim3 grid((M + HTBM - 1) / HTBM, (N + HTBN - 1) / HTBN, splits);
  double* wk = splits > 1 ? work : nullptr;
  if (ev && ev->begin) {
    const hipError_t e = hipEventRecord(ev->begin, s);
    if (e != hipSuccess) return e;
  }
  if (aop)
    hipLaunchKernelGGL(k_zgemm_bf16<true>, grid, dim3(256), 0, s, M, N, K, A, lda, B, ldb, C, ldc, D, ldd, alpha,
                       beta, kps, wk);
  else
    hipLaunchKernelGGL(k_zgemm_bf16<false>, grid, dim3(256), 0, s, M, N, K, A, lda, B, ldb, C, ldc, D, ldd, alpha,
                       beta, kps, wk);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess && ev && ev->end) e = hipEventRecord(ev->end, s);
  if (partials) *partials = splits;
  if (e != hipSuccess || splits == 1 || partials) return e;
  const GemmOutput o{C, ldc, D, ldd, beta};
  hipLaunchKernelGGL(k_splitk_reduce, dim3(reduce_blocks(M, N)), dim3(256), 0, s, M, N, splits, work, o, o, N);
  return hipGetLastError();
}

hipError_t launch_to_bf16_pairs(const float* x, long count, unsigned* out, hipStream_t s) {
  if (count <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_to_bf16_pairs<float>, dim3(2048), dim3(256), 0, s, x, count, out);
  return hipGetLastError();
}
hipError_t launch_to_bf16_pairs(const double* x, long count, unsigned* out, hipStream_t s) {
  if (count <= 0) return hipSuccess;
  hipLaunchKernelGGL(k_to_bf16_pairs<double>, dim3(2048), dim3(256), 0, s, x, count, out);
  return hipGetLastError();
}

namespace {
constexpr int kOnsiteRows = 64;  // projector rows of one workgroup

// Onsite products straight from the projection's split-K partials: P (the quarters of
// a column's partials each summed in split order, then the four sums in theirs, which
// rounds unlike k_splitk_reduce's single chain) lives in LDS only, then per atom
// W(:, 0:m) = D P and W(:, m:2m) = Q P, or with `shift` W(:, 0:m) = (D - shift_j Q) P in
// one pass. Workgroup (g, j): atoms [group_atom[g], group_atom[g + 1]) (at most
// kOnsiteRows rows, or one larger atom), column j. Bound: latency of the partials
// (each read once). FP64 keeps the compensated scalar order of k_atom_blocks_comp.
template <typename T>
__global__ __launch_bounds__(256) void k_onsite_partials(int np, int columns, int splits,
                                                         const double* __restrict__ partial,
                                                         const int* __restrict__ group_atom,
                                                         const int* __restrict__ atom_offset,
                                                         const int* __restrict__ atom_rows,
                                                         const long* __restrict__ block_offset,
                                                         const double* __restrict__ dblk,
                                                         const double* __restrict__ qblk,
                                                         const double* __restrict__ shift, double* __restrict__ W,
                                                         int which_mask) {
#pragma clang fp contract(off)
  extern __shared__ __attribute__((aligned(16))) unsigned char onsite_lds[];
  double2* P = reinterpret_cast<double2*>(onsite_lds);
  const int j = blockIdx.y, tid = threadIdx.x;
  const int a0 = group_atom[blockIdx.x], a1 = group_atom[blockIdx.x + 1];
  const int row0 = atom_offset[a0], rows = atom_offset[a1 - 1] + atom_rows[a1 - 1] - row0;
  double2* sums = P + rows;  // three further quarters of the split sum
  const long total = (long)np * columns;
  const double2* src = reinterpret_cast<const double2*>(partial) + (long)j * np + row0;
  // four threads a row: each sums a quarter of the splits in order
  for (int e = tid; e < 4 * rows; e += 256) {
    const int r = e % rows, q = e / rows;
    const int s0 = splits * q / 4, s1 = splits * (q + 1) / 4;
    double re = 0, im = 0;
    int s = s0;
    for (; s + 4 <= s1; s += 4) {
      double2 v[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) v[u] = src[(s + u) * total + r];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        re += v[u].x;
        im += v[u].y;
      }
    }
    for (; s < s1; ++s) {
      const double2 v = src[s * total + r];
      re += v.x;
      im += v.y;
    }
    (q ? sums + (q - 1) * rows : P)[r] = double2{re, im};
  }
  __syncthreads();
  for (int r = tid; r < rows; r += 256) {
    double2 v = P[r];
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      v.x += sums[q * rows + r].x;
      v.y += sums[q * rows + r].y;
    }
    P[r] = v;
  }
  __syncthreads();
  auto product = [&](const double* blk, int r, int i, const double2* p, double& re, double& im) {
    if constexpr (sizeof(T) == 8) {
      double rs = 0, rc = 0, is = 0, ic = 0;
      auto add = [](double v, double& s, double& c) {
        const double next = s + v;
        const double back = next - s;
        c += (s - (next - back)) + (v - back);
        s = next;
      };
      auto term = [&](double x, double y, double& s, double& c) {
        const double rounded = x * y;
        add(rounded, s, c);
        add(__builtin_fma(x, y, -rounded), s, c);
      };
      for (int k = 0; k < r; ++k) {
        const double lr = blk[2 * (i + k * r)], li = blk[2 * (i + k * r) + 1];
        term(lr, p[k].x, rs, rc);
        term(-li, p[k].y, rs, rc);
        term(lr, p[k].y, is, ic);
        term(li, p[k].x, is, ic);
      }
      re = rs + rc;
      im = is + ic;
    } else {
      float fr = 0.f, fi = 0.f;
      for (int k = 0; k < r; ++k) {
        const float lr = float(blk[2 * (i + k * r)]), li = float(blk[2 * (i + k * r) + 1]);
        const float pr = float(p[k].x), pi = float(p[k].y);
        fr += lr * pr - li * pi;
        fi += lr * pi + li * pr;
      }
      re = fr;
      im = fi;
    }
  };
  double2* out = reinterpret_cast<double2*>(W) + (long)j * np + row0;
  for (int e = tid; e < (shift ? 1 : 2) * rows; e += 256) {
    const int row = e % rows, which = e / rows;
    if (!shift && !((which_mask >> which) & 1)) continue;
    int a = a0;
    while (a + 1 < a1 && atom_offset[a + 1] - row0 <= row) ++a;
    const int r = atom_rows[a], o = atom_offset[a] - row0;
    const double2* p = P + o;
    double re, im;
    product((which ? qblk : dblk) + 2 * block_offset[a], r, row - o, p, re, im);
    if (shift) {
      double qr, qi;
      product(qblk + 2 * block_offset[a], r, row - o, p, qr, qi);
      re -= shift[j] * qr;
      im -= shift[j] * qi;
    }
    out[(long)which * total + row] = double2{re, im};
  }
}
}  // namespace

std::vector<int> onsite_groups(const std::vector<int>& atom_rows) {
  std::vector<int> first{0};
  int rows = 0;
  for (std::size_t a = 0; a < atom_rows.size(); ++a) {
    if (rows && rows + atom_rows[a] > kOnsiteRows) {
      first.push_back(int(a));
      rows = 0;
    }
    rows += atom_rows[a];
  }
  first.push_back(int(atom_rows.size()));
  return first;
}

int onsite_group_rows(const std::vector<int>& atom_rows, const std::vector<int>& groups) {
  int most = 0;
  for (std::size_t g = 0; g + 1 < groups.size(); ++g) {
    int rows = 0;
    for (int a = groups[g]; a < groups[g + 1]; ++a) rows += atom_rows[std::size_t(a)];
    most = std::max(most, rows);
  }
  return most;
}

hipError_t launch_onsite_partials(Precision prec, int np, int columns, int splits, const double* partial,
                                  const int* group_atom, int groups, int group_rows, const int* atom_offset,
                                  const int* atom_rows, const long* block_offset, const double* dblk,
                                  const double* qblk, const double* shift, double* W, int which_mask, hipStream_t s) {
  const std::size_t lds = 4 * std::size_t(group_rows) * 16;
  if (columns > 65535 || group_rows > kOnsiteGroupRows) return hipErrorInvalidValue;
  if (prec == Precision::FP64)
    hipLaunchKernelGGL(k_onsite_partials<double>, dim3(groups, columns), dim3(256), lds, s, np, columns, splits,
                       partial, group_atom, atom_offset, atom_rows, block_offset, dblk, qblk, shift, W, which_mask);
  else
    hipLaunchKernelGGL(k_onsite_partials<float>, dim3(groups, columns), dim3(256), lds, s, np, columns, splits,
                       partial, group_atom, atom_offset, atom_rows, block_offset, dblk, qblk, shift, W, which_mask);
  return hipGetLastError();
}

hipError_t launch_atom_blocks(Precision prec, int np, int columns, int atoms, const int* atom_offset,
                              const int* atom_rows, const long* block_offset, const double* dblk, const double* qblk,
                              const double* P, long ldp, double* W, long ldw, int which_mask, hipStream_t s) {
  const long total = long(np) * columns * 2;
  const int blocks = int(std::min<long>((total + 255) / 256, 4096));
  if (prec == Precision::FP64)
    hipLaunchKernelGGL(k_atom_blocks_comp, dim3(blocks), dim3(256), 0, s, np, columns, atoms, atom_offset, atom_rows,
                       block_offset, dblk, qblk, P, ldp, W, ldw, which_mask);
  else
    hipLaunchKernelGGL(k_atom_blocks_f32, dim3(blocks), dim3(256), 0, s, np, columns, atoms, atom_offset, atom_rows,
                       block_offset, dblk, qblk, P, ldp, W, ldw, which_mask);
  return hipGetLastError();
}

// C = alpha * X + beta * D (complex, column-major, real scalars)
__global__ void k_zaxpby(int M, int N, double alpha, const double* __restrict__ X, long ldx, double beta,
                         const double* __restrict__ D, long ldd, double* __restrict__ C, long ldc) {
  const long total = (long)M * N;
  for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < total; e += (long)gridDim.x * blockDim.x) {
    const int m = int(e % M);
    const long n = e / M;
    double re = 0, im = 0;
    if (alpha != 0.0) { re = alpha * X[2 * (m + n * ldx)]; im = alpha * X[2 * (m + n * ldx) + 1]; }
    if (beta != 0.0) { re += beta * D[2 * (m + n * ldd)]; im += beta * D[2 * (m + n * ldd) + 1]; }
    C[2 * (m + n * ldc)] = re;
    C[2 * (m + n * ldc) + 1] = im;
  }
}

hipError_t launch_zaxpby(int M, int N, double alpha, const double* X, long ldx, double beta, const double* D, long ldd,
                         double* C, long ldc, hipStream_t s) {
  if (M <= 0 || N <= 0) return hipSuccess;
  const long total = long(M) * N;
  const int blocks = int(std::min<long>((total + 255) / 256, 8192));
  hipLaunchKernelGGL(k_zaxpby, dim3(blocks), dim3(256), 0, s, M, N, alpha, X, ldx, beta, D, ldd, C, ldc);
  return hipGetLastError();
}


// Loads this file's code object on the calling thread (see module_prime.hpp).
hipError_t prime_module_gemm() {
  hipFuncAttributes a{};
  return hipFuncGetAttributes(&a, reinterpret_cast<const void*>(k_splitk_reduce));
}

}  // namespace sdft_hip
