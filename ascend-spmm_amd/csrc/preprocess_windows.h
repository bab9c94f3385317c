// Window-by-window preprocessing (preprocess_windows.hip): host interface used
// by the pipelines of preprocess.hip.
//
// Applies to matrices whose rows hold strictly ascending column ids, of the
// sizes that window_rule.h takes (the plan kernels check the rest and set the
// record's error word otherwise, and the caller then takes the sorting
// pipeline, which also reports every input error).
#pragma once

#include "common.h"
#include "window_rule.h"

namespace spmm {
namespace win {

struct Matrix {
  int64_t rows, cols, nnz;
  int32_t index_type, value_type;
  const void* rowptr;
  const void* col;
  const void* value;
};

inline bool eligible(Op op, const Matrix& m, int64_t W) { return eligible(op, m.rows, m.cols, m.nnz, W); }

// A plan's record holds p_begin and n, whatever else err says (not of a row
// pointer that is not monotone inside [0, nnz]).
bool ends_known(int64_t err);

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

// preprocess (16-row windows).  Device record of its plan.
struct TaskRecord {
  int64_t err;
  int64_t p_begin, n;
  int64_t bpos;            // sorted position of the marginal window, -1: none
  int64_t bwin, bblocks;   // the marginal window and its blocks
  int64_t baic, shared;    // its blocks on the block part; both parts hold some
  int64_t naic;            // windows of the block part
  int64_t aic_blocks, vnnz, shared_nnz;
  int64_t last_pos;        // sorted position of the last (perhaps shorter) window
  int64_t out_rows;
  double est_aic, est_aiv, est_max;
  int64_t t_kept, t_vnnz;  // graph layout: the transpose's split
  int64_t t_err;           // its error word (err is read, so not written, by its kernels)
};

// block_level_split, and the graph layout's transpose.
struct SplitArrays {
  uint32_t* nb;     // [nwin] blocks per window
  uint32_t* hist;   // [16][nwin] blocks by occupancy
  uint32_t* total;  // [kHistCopies][16] sums of hist over the windows, in copies
  uint32_t* moved;  // [nwin] blocks of the boundary occupancy that move
  uint32_t* kptr;   // [nwin + 1] kept blocks before
  uint32_t* vptr;   // [nwin + 1] moved nonzeros before
  uint32_t* occ;    // [nnz] occupancies of windows too wide for LDS
  uint32_t* first;  // [min(nnz, cols)] first nonzeros of the boundary window's blocks
  uint32_t* rule;   // [1] boundary occupancy
};
constexpr int kHistCopies = 64;

spmm_status plan_split(const Matrix& m, double a, int64_t W, const SplitArrays& x, WindowState* state, hipStream_t s);
spmm_status fill_split(const Matrix& m, int64_t W, const SplitArrays& x, void* crow, void* uniq, void* val, void* vrow,
                       void* vcol, void* vval, hipStream_t s);

struct TaskArrays {
  TaskRecord* record;
  uint32_t* nb;        // [nwin]
  uint64_t *dkey, *sdkey;
  uint32_t *wid, *rank, *swin;  // windows, their ranks and order by density
  uint64_t* sbz;         // [nwin] blocks << 32 | nonzeros, in that order
  uint32_t *pnb, *pnnz;  // [nwin + 1] blocks and nonzeros before, in that order
  uint32_t *mocc, *mfirst, *midx;  // [min(nnz, cols)] marginal window's blocks
  uint32_t* mrow;                  // [17]
  void* temp;
  size_t temp_bytes;
  // graph layout
  uint32_t* inv;               // [rows]
  uint32_t *tkey, *stkey;      // [nnz] packed row of each transposed entry
  uint64_t *tword, *stword;    // [nnz] packed column << 32 | value bits (or entry)
  uint32_t* rp;                // [16 nwin + 1] transposed row pointer
  SplitArrays split;
};

// Temporary bytes of the device sorts.
size_t task_temp_bytes(const Matrix& m, bool layout);
// handed_over: the counts have found the matrix not to be for this pipeline,
// and the plan has ended there.
spmm_status plan_task(const Matrix& m, bool layout, const TaskArrays& x, bool* handed_over, hipStream_t s);
// naic: the plan's TaskRecord::naic.
spmm_status fill_task(const Matrix& m, bool layout, int64_t naic, const TaskArrays& x, const spmm_taskmap_out* o,
                      hipStream_t s);

spmm_status plan_blocks(const Matrix& m, int64_t W, bool tiles, const BlockArrays& a, hipStream_t s);
spmm_status fill_blocks(const Matrix& m, int64_t W, bool tiles, const BlockArrays& a, void* crow, void* uniq,
                        void* val, hipStream_t s);

}  // namespace win
}  // namespace spmm
