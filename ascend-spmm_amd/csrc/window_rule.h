// Which matrices the window-by-window pipeline (preprocess_windows.hip) takes
// and which go to the sorting pipeline (preprocess.hip), by their sizes.  Host
// arithmetic only.
#pragma once

#include <cmath>
#include <cstdint>

namespace spmm {
namespace win {

// A window's column set is a bitmap in LDS, one bit per column: 2^20 columns
// are 128 KB, beside 16 KB of prefix counts.
constexpr int64_t kMaxColumns = int64_t(1) << 20;
// One work-group of at most 1024 threads per window, and a grid holds fewer
// than 2^32 threads.
constexpr int64_t kMaxWindows = (int64_t(1) << 22) - 1;

enum class Op { kBlocks, kSplit, kTask, kTaskLayout };  // kBlocks: csr_to_bcsr and csr_to_ascend_cube

// Time of a conversion on each pipeline (ns).  The sorting pipeline pays for
// its launches and per nonzero.  The window pipeline pays little per nonzero
// but for every window, however empty: about 5.5 ns to schedule and set up its
// work-groups, and the clears and sweeps of its bitmaps, which grow with the
// columns and faster than them, as large bitmaps leave few work-groups on a CU
// (2^12, 2^16, 2^18, 2^19, 2^20 columns: 6, 7, 11, 21, 47 ns per window).
//
// Fitted to 681 matrices of random columns, 2^12 to 2^20 rows and columns, 1/4
// to 64 nonzeros per row, windows of 1, 4, 8 and 16 rows.  Both sides, us
// (sorting / windows): csr_to_bcsr of 2^20 rows and columns, 16.8M nonzeros,
// 2289 / 3225, of 1.0M 381 / 3065, in windows of one row 365 / 48000; of 2^18
// and 1.0M, 370 / 206; of 2^20 rows, 2^12 columns, 4.2M, 647 / 441 and 0.3M,
// 264 / 417; preprocess of 2^20, 4.2M, 1280 / 2011, of 2^19, 8.4M, 1816 / 588.
struct Cost {
  double sort_call, sort_nnz, sort_row;             // ns
  double call, nnz, window, wide;                   // wide: a window's bitmaps at 2^20 columns
};
constexpr Cost kCosts[] = {
    {180e3, 0.116, 0.05, 35e3, 0.0125, 5.6, 39.2},  // kBlocks
    {320e3, 0.207, 0.08, 45e3, 0.022, 5.0, 38.5},   // kSplit
    {440e3, 0.141, 0.14, 112e3, 0.006, 6.6, 20.2},  // kTask
    {850e3, 0.420, 0.45, 182e3, 0.089, 12.4, 56.3}, // kTaskLayout
};

// The window pipeline is tried where it is faster by the fit with a margin of
// 15%: none of the 681 matrices is then slower than with the sorting pipeline,
// and 24 of them, by up to 1.6 times, would have been faster window by window.
inline bool faster(Op op, int64_t rows, int64_t cols, int64_t nnz, int64_t W) {
  const Cost& c = kCosts[static_cast<int>(op)];
  const double windows = static_cast<double>((rows + W - 1) / W), z = static_cast<double>(nnz);
  const double share = static_cast<double>(cols) / static_cast<double>(kMaxColumns);
  return c.call + c.nnz * z + windows * (c.window + c.wide * share * std::sqrt(share)) <=
         0.85 * (c.sort_call + c.sort_nnz * z + c.sort_row * static_cast<double>(rows));
}

// kTaskLayout: a square matrix, whose transpose in packed rows (whole windows)
// goes the same way.  The plan kernels look at what sizes do not show.
inline bool eligible(Op op, int64_t rows, int64_t cols, int64_t nnz, int64_t W) {
  if (W < 1 || W > 16 || rows < 1 || cols < 1 || nnz < 1 || nnz >= (int64_t(1) << 31)) return false;
  if ((rows + W - 1) / W > kMaxWindows || cols > kMaxColumns) return false;
  if (op == Op::kTaskLayout && (rows + 15) / 16 * 16 > kMaxColumns) return false;
  return faster(op, rows, cols, nnz, W);
}

}  // namespace win
}  // namespace spmm
