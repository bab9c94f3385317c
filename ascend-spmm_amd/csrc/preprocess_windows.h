// Window-by-window preprocessing (preprocess_windows.hip): host interface used
// by the pipelines of preprocess.hip.
//
// Applies to matrices whose rows hold strictly ascending column ids, with at
// most kMaxColumns columns, fewer than 2^31 nonzeros and windows of at most 16
// rows (eligible() checks the sizes; the plan kernels check the rest and set
// WindowState::err otherwise, and the caller then takes the sorting pipeline,
// which also reports every input error).
#pragma once

#include "common.h"

namespace spmm {
namespace win {

// A window's column set is a bitmap in LDS, one bit per column: 2^20 columns
// are 128 KB, beside 16 KB of prefix counts.
constexpr int64_t kMaxColumns = int64_t(1) << 20;

struct Matrix {
  int64_t rows, cols, nnz;
  int32_t index_type, value_type;
  const void* rowptr;
  const void* col;
  const void* value;
};

inline bool eligible(const Matrix& m, int64_t W) {
  return W >= 1 && W <= 16 && m.rows >= 1 && m.cols >= 1 && m.cols <= kMaxColumns && m.nnz >= 1 &&
         m.nnz < (int64_t(1) << 31) && m.rows < (int64_t(1) << 31) - 64;
}

// Device record of a plan, read back by the host in one copy.
struct WindowState {
  int64_t err;             // nonzero: not for this path (or an input error)
  int64_t p_begin, n;      // first position, nonzeros
  int64_t total;           // bcsr: blocks; cube: tiles; split: kept blocks
  int64_t vnnz;            // split: nonzeros of the CSR part
};

// csr_to_bcsr / csr_to_ascend_cube.
struct BlockArrays {
  WindowState* state;
  uint32_t* nb;   // [nwin] blocks (tiles) per window
  uint32_t* ptr;  // [nwin + 1] exclusive sums
};

spmm_status plan_blocks(const Matrix& m, int64_t W, bool tiles, const BlockArrays& a, hipStream_t s);
spmm_status fill_blocks(const Matrix& m, int64_t W, bool tiles, const BlockArrays& a, void* crow, void* uniq,
                        void* val, hipStream_t s);

}  // namespace win
}  // namespace spmm
