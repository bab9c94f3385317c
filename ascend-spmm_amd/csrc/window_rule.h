// Which matrices the window-by-window pipeline (preprocess_windows.hip) takes
// and which go to the sorting pipeline (preprocess.hip), by their sizes.  Host
// arithmetic only.
#pragma once

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

// kTaskLayout: a square matrix, whose transpose in packed rows (whole windows)
// goes the same way.  The plan kernels look at what sizes do not show.
inline bool eligible(Op op, int64_t rows, int64_t cols, int64_t nnz, int64_t W) {
  if (W < 1 || W > 16 || rows < 1 || cols < 1 || nnz < 1 || nnz >= (int64_t(1) << 31)) return false;
  if ((rows + W - 1) / W > kMaxWindows || cols > kMaxColumns) return false;
  if (op == Op::kTaskLayout && (rows + 15) / 16 * 16 > kMaxColumns) return false;
  return true;
}

}  // namespace win
}  // namespace spmm
