// Complex GEMM and PAW onsite-block launchers (MFMA, column-major, interleaved
// complex storage in FP64 unless stated otherwise).
#pragma once
#include <hip/hip_runtime_api.h>

#include <cstddef>
#include <vector>

namespace sdft_hip {

enum class Precision { FP64 = 0, FP32 = 1 };

// Optional events recorded on the launch stream immediately before and after
// the MFMA kernel of one GEMM (the split-K reduction is outside the pair).
struct LaunchEvents {
  hipEvent_t begin = nullptr, end = nullptr;
};

// One result block of a product: C = ... + beta * D.
struct GemmOutput {
  double* C = nullptr;
  long ldc = 0;
  const double* D = nullptr;
  long ldd = 0;
  double beta = 0;
};

int zgemm_splits(int M, int N, int K);
std::size_t zgemm_workspace_bytes(int M, int N, int K);

// C = alpha op(A) op(B) + beta * D; aop/bop: 0 = Normal, 1 = Adjoint. D may
// alias C. `prec` selects the arithmetic (FP64 or FP32 MFMA); storage is FP64.
// With `partials` a product split along K is left as *partials blocks of M x N (M
// the leading dimension) in `work` for the caller to sum (1: complete, in C).
hipError_t zgemm(Precision prec, int aop, int bop, int M, int N, int K, double alpha, const double* A, long lda,
                 const double* B, long ldb, double* C, long ldc, const double* D, long ldd, double beta, double* work,
                 std::size_t work_bytes, hipStream_t s, const LaunchEvents* ev = nullptr, int* partials = nullptr);
// Real MFMA products per complex multiply-add of the kernels: 3 (Gauss form). The conventional 8 m n k flop count of a complex GEMM corresponds to 4.
int zgemm_real_products(Precision prec);
// Same with A stored in FP32 (resident search copy of the projectors).
hipError_t zgemm_f32_storage(int aop, int bop, int M, int N, int K, double alpha, const float* A, long lda,
                             const double* B, long ldb, double* C, long ldc, const double* D, long ldd, double beta,
                             double* work, std::size_t work_bytes, hipStream_t s, const LaunchEvents* ev = nullptr, int* partials = nullptr);

// op(A) B with the first n_first columns of the result going to one output and the
// n_second others to another, in one launch that reads A once.
hipError_t zgemm_two_outputs(int aop, int M, int n_first, int n_second, int K, const double* A, long lda,
                             const double* B, long ldb, const GemmOutput& first, const GemmOutput& second, double* work,
                             std::size_t work_bytes, hipStream_t s, const LaunchEvents* ev);
hipError_t zgemm_two_outputs(int aop, int M, int n_first, int n_second, int K, const float* A, long lda,
                             const double* B, long ldb, const GemmOutput& first, const GemmOutput& second, double* work,
                             std::size_t work_bytes, hipStream_t s, const LaunchEvents* ev);

// C = alpha op(A) B + beta D (aop 0 = Normal, 1 = Adjoint) with A stored as BF16
// complex pairs (real part in the low 16 bits of each 32-bit word), B, C, D
// in FP64: BF16 MFMA products with FP32 accumulation (search arithmetic).
hipError_t zgemm_bf16_storage(int aop, int M, int N, int K, double alpha, const unsigned* A, long lda,
                              const double* B, long ldb, double* C, long ldc, const double* D, long ldd, double beta,
                              double* work, std::size_t work_bytes, hipStream_t s, const LaunchEvents* ev = nullptr, int* partials = nullptr);
// count complex values (FP32 or FP64 pairs) -> BF16 pairs, round to nearest even
hipError_t launch_to_bf16_pairs(const float* x, long count, unsigned* out, hipStream_t s);
hipError_t launch_to_bf16_pairs(const double* x, long count, unsigned* out, hipStream_t s);

// W(:, 0:m) = D_a P_a and W(:, m:2m) = Q_a P_a per atom block (which_mask bit
// 0: D, bit 1: Q). FP64 uses the compensated scalar order of the reference.
hipError_t launch_atom_blocks(Precision prec, int np, int columns, int atoms, const int* atom_offset,
                              const int* atom_rows, const long* block_offset, const double* dblk, const double* qblk,
                              const double* P, long ldp, double* W, long ldw, int which_mask, hipStream_t s);

// The same from the projection's split-K partials (`splits` blocks np x columns, P
// their sum): W(:, 0:m) = D P, W(:, m:2m) = Q P, or with `shift` (columns values on
// the device) W(:, 0:m) = (D - shift_j Q) P. group_atom (groups + 1 entries on the
// device): onsite_groups of the atoms; group_rows: rows of the largest group, at
// most kOnsiteGroupRows.
constexpr int kOnsiteGroupRows = 1024;
std::vector<int> onsite_groups(const std::vector<int>& atom_rows);
// rows of the largest group
int onsite_group_rows(const std::vector<int>& atom_rows, const std::vector<int>& groups);
hipError_t launch_onsite_partials(Precision prec, int np, int columns, int splits, const double* partial,
                                  const int* group_atom, int groups, int group_rows, const int* atom_offset,
                                  const int* atom_rows, const long* block_offset, const double* dblk,
                                  const double* qblk, const double* shift, double* W, int which_mask, hipStream_t s);

// C = alpha X + beta D
hipError_t launch_zaxpby(int M, int N, double alpha, const double* X, long ldx, double beta, const double* D, long ldd,
                         double* C, long ldc, hipStream_t s);

}  // namespace sdft_hip
