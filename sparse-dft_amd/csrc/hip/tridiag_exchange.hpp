// Who takes part in which step of the one-launch tridiagonalisation's exchange
// (tridiag.hip); free of HIP so that a host program can walk the same rules.
#pragma once

namespace sdft_hip {

constexpr int kHetrdBuffers = 3;  // published steps in flight: step k uses buffer k % 3

// Workgroup g of `groups` keeps the rows g + r groups < n; the first r whose row
// is at least `row`.
constexpr int hetrd_first_row(int groups, int g, int row) { return row <= g ? 0 : (row - g + groups - 1) / groups; }

// The workgroup of the last row, which stays to the end and writes the outputs.
constexpr int hetrd_last_group(int n, int groups) { return (n - 1) % groups; }

// Whether workgroup g reads step k. Its rows at k + 2 and beyond need it, and those
// it publishes in step k + 1; row k + 1 does not, it is reduced. A reader (but the
// last row's workgroup, which in the end reads alone) is thus a publisher of the
// next step, so a workgroup that has received every row of step k knows that
// nobody reads step k - 1.
constexpr bool hetrd_reads(int n, int groups, int g, int k) {
  return g == hetrd_last_group(n, groups) || g + hetrd_first_row(groups, g, k + 2) * groups < n;
}

}  // namespace sdft_hip
