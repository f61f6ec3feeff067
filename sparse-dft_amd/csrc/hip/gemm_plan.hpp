// Launch plan of the complex GEMM (gemm.hip): tile and split along K of a shape.
// Free of HIP so that a host program can walk the rules.
#pragma once

#include <algorithm>

namespace sdft_hip {

constexpr int kGemmSlab = 16;  // K of one slab: splits are whole slabs

// Tiles: 0 = 32 x 32, 1 = 64 x 32, 2 = 64 x 64.
struct GemmTile {
  int bm, bn;
};
constexpr GemmTile kTiles[3] = {{32, 32}, {64, 32}, {64, 64}};

inline long gemm_tiles(int M, int N, int cfg) {
  return long((M + kTiles[cfg].bm - 1) / kTiles[cfg].bm) * ((N + kTiles[cfg].bn - 1) / kTiles[cfg].bn);
}
// Splits along K for about 1200 workgroups (a little over four a CU; 512 x 160 x n took
// 213 us with 1280, 230 and more with 640), at least 256 of K each, or 128 while that
// leaves CUs without a workgroup (128 x 37 x 4573 in 32 splits of 143), or 64 while half
// of them have none: a slab of K is then a round trip to memory, and the reduction of
// more partials costs less (120 x 20 x 1647 in 12 / 26 splits 12.6 / 9.7 us, 20 x 20 x 1647
// 13.6 / 9.2, 64 x 4 x 1647 11.8 / 8.8, 160 x 160 x 160 in 1 / 2 10.2 / 8.6); 48 at most
// to fill the chip.
inline int gemm_fill_splits(long tiles, int K) {
  const long most = std::min<long>(48, (1200 + tiles - 1) / tiles);
  long splits = std::min<long>(most, K / 256);
  if (tiles * splits < 256) splits = std::min<long>(most, K / 128);
  if (tiles * splits < 128) splits = std::min<long>({most, K / 64, (256 + tiles - 1) / tiles});
  return int(std::max<long>(1, splits));
}
// Fewest splits: powers of two to 2048 (FP32: 1024) workgroups of 32 x 32, 64 splits at
// most, 256 of K each at least. They bound the chain of additions behind a partial sum,
// whose rounding error grows with the root of its length, where the rule above alone
// cuts a wide or a small result too coarsely. Relative error against long double
// without / with the bound: 512 x 480 x 23847 FP64 2.35e-15 / 1.80e-15, 480 x 240 x 23847
// FP64 1.72e-15 / 1.32e-15, 64 x 480 x 23847 FP32 6.4e-7 / 4.9e-7. It costs no time: S of
// 480 columns of 64 atoms 1361 / 1353 us, the 64-atom solve 114.2 / 114.1 ms.
inline int gemm_least_splits(bool fp64, int M, int N, int K) {
  const long tiles = gemm_tiles(M, N, 0), target = fp64 ? 2048 : 1024;
  int splits = 1;
  while (tiles * splits < target && K / (2 * splits) >= 256 && splits < 64) splits *= 2;
  return splits;
}
// The tile of a shape, for both precisions: 64 x 64 where the result is wide (256
// columns, at most a tenth of them padding) and has 1200 such tiles, 64 x 32 where
// 768 workgroups are reached with splits, else 32 x 32. Measured, us, 64 x 64 /
// 64 x 32 / 32 x 32 at their best splits (n = 23847): n x 480 x 512 adjoint FP64
// 687 / 749 / 777, FP32 373 / 433 / 494; 512 x 160 x n FP64 268 / 213 / 225, FP32
// 140 / 126 / 133; 640 x 160 x n FP64 331 / 299 / 299, FP32 183 / 176 / 197; n x 220 x
// 380 FP64 279 / 260 / 267; 160 x 160 x n FP64 116 / 95 / 85; 128 x 37 x 4573 FP64
// 25 / 17 / 13; 9141 x 80 x 256 adjoint FP64 57 / 38 / 37. Against the single-buffered
// kernels (32 x 32 and 128 x 32 tiles, two barriers and per-element addresses and
// bounds in every slab): 512 x 160 x n FP64 287, FP32 164; 640 x 160 x n 391, 236;
// n x 480 x 512 823, 562; 160 x 160 x n 101, 69; 128 x 37 x 4573 19, 16.
struct GemmPlan {
  int cfg, splits, kps;  // tile, splits along K, K of a split
};
// K of a split (whole slabs) for at most `splits` of them
inline int gemm_k_per_split(int K, int splits) {
  return ((K + splits - 1) / splits + kGemmSlab - 1) / kGemmSlab * kGemmSlab;
}
inline GemmPlan gemm_plan(bool fp64, int M, int N, int K) {
  GemmPlan p{};
  p.cfg = 0;
  if (N >= 256 && (N + 63) / 64 * 64 <= N + N / 10 && gemm_tiles(M, N, 2) >= 1200) {
    p.cfg = 2;
  } else {
    const long tiles = gemm_tiles(M, N, 1);
    if (tiles * gemm_fill_splits(tiles, K) >= 768) p.cfg = 1;
  }
  p.splits = std::max(gemm_fill_splits(gemm_tiles(M, N, p.cfg), K), gemm_least_splits(fp64, M, N, K));
  p.kps = gemm_k_per_split(K, p.splits);
  return p;
}

}  // namespace sdft_hip
