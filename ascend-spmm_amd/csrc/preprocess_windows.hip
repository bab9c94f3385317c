// Window-by-window preprocessing: the layout converters without a sort.
//
// A window's rows are contiguous in the CSR arrays, so one work-group can find
// its distinct columns by itself: a bitmap over the columns in LDS, one bit
// per column, set by the window's nonzeros.  The popcount of the bitmap is the
// window's number of 16x1 blocks, and a column's rank among the set bits is
// its block (columns ascend, as the layouts ask).  Plans count (or rank)
// blocks per window and scan a few words per window; fills build the bitmap
// again and write every output straight from the CSR arrays.  So the column
// ids are read twice, the values once, and no per-nonzero array is ever
// written, where the sorting pipeline moves about 20 words of 8 bytes per
// nonzero through memory (csr_to_bcsr of 14.4M nonzeros in 4096 banded windows:
// 1380 us there, 144 us here: counting 30 us, writing 78 us, the read-back
// that sizes the outputs and launches the rest).
//
// Bound: vector instructions per nonzero on long windows (about 130 in
// write_blocks, 60 in count_windows), and on short ones the latency of a
// window's steps (row pointers, columns, LDS atomics, scan), which the other
// windows resident on the CU cover: a bitmap of 100,000 columns is 12.5 KB,
// and work-groups are sized so that a CU holds 1024-2048 threads of them.
#include "preprocess_windows.h"

#include <type_traits>

namespace spmm {
namespace win {
namespace {

typedef unsigned int u2_t __attribute__((ext_vector_type(2)));
typedef unsigned int u4_t __attribute__((ext_vector_type(4)));

enum : int { kGeneral = 1 };  // WindowState::err: take the sorting pipeline

// ------------------------------------------------------------- bitmap sizes

// Words per prefix group (1 << gshift: 2, 4 or 8) and LDS layout: bitmap words
// (padded to whole quads), then one prefix count per group.  Two words per
// group make a rank one 8-byte read and two popcounts; larger bitmaps take
// longer groups so that more of them stay resident.
struct BitmapShape {
  uint32_t words, groups;
  int gshift;
  int threads;
  size_t lds() const { return (static_cast<size_t>(words) + groups) * sizeof(uint32_t); }
  explicit BitmapShape(int64_t cols) {
    uint32_t w = static_cast<uint32_t>((cols + 31) / 32);
    gshift = w > 16384 ? 3 : (w > 4096 ? 2 : 1);
    const uint32_t gw = gshift == 3 ? 8 : 4;
    words = (w + gw - 1) / gw * gw;
    groups = ((words >> gshift) + 3u) & ~3u;  // what follows stays 16-byte aligned
    // 8 work-groups of 256 threads fit a CU's LDS up to 20 KB each, 4 of 512
    // up to 40 KB, 2 of 1024 up to 80 KB.
    threads = lds() <= 18 * 1024 ? 256 : (lds() <= 38 * 1024 ? 512 : 1024);
  }
};

// ----------------------------------------------------------- device helpers

// The window's rows: offsets of its W rows' starts (and end) from its first
// position.  Returns false (n = 0) when the row pointer is not monotone inside
// [0, nnz].  All threads call it; a barrier inside.
struct WindowRows {
  uint32_t off[17];  // off[r]: first nonzero of row r, off[W] .. off[16] = n
  uint32_t n;
  uint32_t ok;
  int64_t base;
};

template <typename P>
__device__ inline void load_window(const P* __restrict__ rowptr, int64_t rows, int64_t nnz, int64_t w, int W,
                                   WindowRows* s) {
  if (threadIdx.x < 64) {
    const int t = threadIdx.x <= static_cast<unsigned>(W) ? threadIdx.x : W;
    const int64_t r = w * W + t;
    const int64_t v = static_cast<int64_t>(rowptr[r < rows ? r : rows]);
    const int64_t up = __shfl_up(v, 1);
    const bool bad = v < 0 || v > nnz || (threadIdx.x > 0 && v < up);
    const int64_t v0 = __shfl(v, 0);
    const bool any = __ballot(bad) != 0;
    const int64_t vw = __shfl(v, W);
    if (threadIdx.x <= 16) s->off[threadIdx.x] = any ? 0u : static_cast<uint32_t>(v - v0);
    if (threadIdx.x == 0) {
      s->base = any ? 0 : v0;
      s->n = any ? 0u : static_cast<uint32_t>(vw - v0);
      s->ok = any ? 0u : 1u;
    }
  }
  __syncthreads();
}

// The rows' first offsets in scalar registers (the LDS copy would be read
// again for every nonzero, behind the LDS writes in between).
struct RowStarts {
  uint32_t off[16];
  __device__ inline explicit RowStarts(const WindowRows& s) {
#pragma unroll
    for (int t = 0; t < 16; ++t) off[t] = __builtin_amdgcn_readfirstlane(s.off[t]);
  }
  // Row (inside the window) of offset i: the last row that starts at or before it.
  __device__ inline uint32_t row(uint32_t i) const {
    uint32_t r = 0;
#pragma unroll
    for (int t = 1; t < 16; ++t) r += i >= off[t] ? 1u : 0u;
    return r;
  }
  __device__ inline bool starts(uint32_t i) const {
    bool any = false;
#pragma unroll
    for (int t = 1; t < 16; ++t) any = any || off[t] == i;
    return any;
  }
};

__device__ inline void clear_words(uint32_t* p, uint32_t words) {  // words % 4 == 0, p 16-byte aligned
  u4_t* q = reinterpret_cast<u4_t*>(p);
  for (uint32_t i = threadIdx.x; i < words / 4; i += blockDim.x) q[i] = u4_t{0u, 0u, 0u, 0u};
}

// Exclusive scan of one value per thread over the work-group; total in
// *sum (all threads).  s_wave: 17 words of LDS.  Two barriers.
__device__ inline uint32_t block_exclusive(uint32_t v, uint32_t* s_wave, uint32_t* sum) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
  uint32_t x = v;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t y = __shfl_up(x, o);
    x += lane >= o ? y : 0u;
  }
  __syncthreads();  // an earlier scan's sums have been read
  if (lane == 63) s_wave[wave] = x;
  __syncthreads();
  uint32_t before = 0, all = 0;
  for (int i = 0; i < waves; ++i) {
    const uint32_t t = s_wave[i];
    before += i < wave ? t : 0u;
    all += t;
  }
  *sum = all;
  return before + x - v;
}

// Prefix counts of the bitmap's groups; returns the number of set bits.  A
// thread takes whole quads of words.
__device__ inline uint32_t bitmap_prefix(const uint32_t* bm, uint32_t* prefix, uint32_t words, int gshift,
                                         uint32_t* s_wave) {
  const uint32_t quads = words / 4;
  uint32_t per = (quads + blockDim.x - 1) / blockDim.x;
  if (gshift == 3) per += per & 1u;  // whole groups
  const uint32_t q0 = threadIdx.x * per, q1 = q0 + per < quads ? q0 + per : quads;
  const u4_t* q = reinterpret_cast<const u4_t*>(bm);
  uint32_t sum = 0;
  for (uint32_t i = q0; i < q1; ++i) {
    const u4_t b = q[i];
    sum += __popc(b[0]) + __popc(b[1]) + __popc(b[2]) + __popc(b[3]);
  }
  uint32_t total;
  uint32_t at = block_exclusive(sum, s_wave, &total);
  for (uint32_t i = q0; i < q1; ++i) {
    const u4_t b = q[i];
    const uint32_t lo = __popc(b[0]) + __popc(b[1]);
    if (gshift == 1) {
      prefix[2 * i] = at;
      prefix[2 * i + 1] = at + lo;
    } else if (gshift == 2) {
      prefix[i] = at;
    } else if ((i & 1u) == 0) {
      prefix[i >> 1] = at;
    }
    at += lo + __popc(b[2]) + __popc(b[3]);
  }
  __syncthreads();
  return total;
}

// Set bits of this wavefront's share of the bitmap.
__device__ inline uint32_t count_bits(const uint32_t* bm, uint32_t words) {
  const u4_t* q = reinterpret_cast<const u4_t*>(bm);
  uint32_t c = 0;
  for (uint32_t i = threadIdx.x; i < words / 4; i += blockDim.x) {
    const u4_t b = q[i];
    c += __popc(b[0]) + __popc(b[1]) + __popc(b[2]) + __popc(b[3]);
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o);
  return c;
}

// Rank of a set column among the bitmap's set bits.
__device__ inline uint32_t bitmap_rank(const uint32_t* bm, const uint32_t* prefix, int gshift, uint32_t c) {
  const uint32_t wi = c >> 5, g = wi >> gshift;
  const uint32_t in = wi & ((1u << gshift) - 1u);
  const uint32_t below = (1u << (c & 31u)) - 1u;
  uint32_t r = prefix[g];
  if (gshift == 1) {
    const u2_t b = reinterpret_cast<const u2_t*>(bm)[g];
    return r + __popc(b[0] & (in ? 0xFFFFFFFFu : below)) + __popc(b[1] & (in ? below : 0u));
  }
  const u4_t* q = reinterpret_cast<const u4_t*>(bm + (g << gshift));
  const int quads = 1 << (gshift - 2);
  for (int k = 0; k < quads; ++k) {
    const u4_t b = q[k];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t idx = 4u * k + j;
      const uint32_t mask = idx < in ? 0xFFFFFFFFu : (idx == in ? below : 0u);
      r += __popc(b[j] & mask);
    }
  }
  return r;
}

// Columns of a window, kHold per thread in registers: windows of at most
// kHold * blockDim.x nonzeros read their columns once per kernel.
constexpr int kHold = 16;

// v of the lane below, across the wavefront; `first` for lane 0.
template <typename C>
__device__ inline C lane_below(C v, C first) {
  if constexpr (sizeof(C) == 4) {
    return static_cast<C>(
        __builtin_amdgcn_update_dpp(static_cast<int>(first), static_cast<int>(v), 0x138, 0xF, 0xF, false));
  } else {
    const uint64_t f = static_cast<uint64_t>(first), u = static_cast<uint64_t>(v);
    const uint32_t lo = __builtin_amdgcn_update_dpp(static_cast<int>(f), static_cast<int>(u), 0x138, 0xF, 0xF, false);
    const uint32_t hi =
        __builtin_amdgcn_update_dpp(static_cast<int>(f >> 32), static_cast<int>(u >> 32), 0x138, 0xF, 0xF, false);
    return static_cast<C>(static_cast<uint64_t>(hi) << 32 | lo);
  }
}

// ORs in the bits of the lane kShift below in the same row of 16 lanes when
// it has the same word.  Both moves run in every lane, outside the selection:
// a DPP move reads nothing from a lane that is switched off.
template <int kShift>
__device__ inline void combine(uint32_t word, uint32_t& bit) {
  const int w = __builtin_amdgcn_update_dpp(-2, static_cast<int>(word), 0x110 + kShift, 0xF, 0xF, false);
  const int b = __builtin_amdgcn_update_dpp(0, static_cast<int>(bit), 0x110 + kShift, 0xF, 0xF, false);
  bit |= static_cast<uint32_t>(w) == word ? static_cast<uint32_t>(b) : 0u;
}

// ORs each lane's bit into its bitmap word.  Neighbouring nonzeros of a dense
// row share words, and same-word LDS atomics of a wavefront run one after
// another, so a lane first takes in the bits of up to three lanes below it
// with the same word (DPP moves), and only the last lane of such a run, or of
// its quad, does the atomic: every bit is covered, and ORing one twice does
// no harm (counting 14.4M nonzeros at 13 per word: 30 us, 41 us with an
// atomic per nonzero).  A lane without a column passes word ~0.
__device__ inline void or_bits(uint32_t* bm, uint32_t word, uint32_t bit) {
  const uint32_t next = static_cast<uint32_t>(
      __builtin_amdgcn_update_dpp(-2, static_cast<int>(word), 0x101, 0xF, 0xF, false));  // lane above; -2 past the row
  bool last = true;
  if (__ballot(next == word && word != ~0u) != 0) {
    combine<1>(word, bit);
    combine<2>(word, bit);
    last = next != word || (threadIdx.x & 3) == 3;
  }
  if (last && word != ~0u) atomicOr(&bm[word], bit);
}

// Sets the window's bits and leaves its columns in `held` when they fit the
// registers (windows of at most kHold * blockDim.x nonzeros).  *bad collects
// what the path does not take: columns outside [0, cols) and rows that do not
// ascend strictly.
template <bool kCheck, typename Cols>
__device__ inline void set_bits(const Cols& col, const WindowRows& s, int64_t cols, uint32_t* bm,
                                uint32_t (&held)[kHold], int* bad) {
  const uint32_t T = blockDim.x, n = s.n;
  const RowStarts starts(s);
  for (uint32_t i0 = 0; i0 < n; i0 += kHold * T) {
    using C = typename Cols::Id;
    C c[kHold];
#pragma unroll
    for (int k = 0; k < kHold; ++k) {
      const uint32_t i = i0 + k * T + threadIdx.x;
      c[k] = i < n ? col(s.base + i) : static_cast<C>(-1);
    }
#pragma unroll
    for (int k = 0; k < kHold; ++k) {
      if (i0 + k * T < n) {  // uniform
        const uint32_t i = i0 + k * T + threadIdx.x;
        bool in = i < n;
        if constexpr (kCheck) {
          C before = static_cast<C>(-1);  // lane 0: the nonzero before the wavefront's
          if ((threadIdx.x & 63) == 0 && in && i > 0) before = col(s.base + i - 1);
          const C prev = lane_below(c[k], before);
          if (in && i > 0 && c[k] <= prev) {  // allowed at a row's first nonzero only
            if (!starts.starts(i)) *bad = 1;
          }
          if (in && (c[k] < 0 || static_cast<int64_t>(c[k]) >= cols)) {
            *bad = 1;
            in = false;
          }
        }
        const uint32_t u = static_cast<uint32_t>(c[k]);
        or_bits(bm, in ? u >> 5 : ~0u, 1u << (u & 31u));
        held[k] = u;
      }
    }
  }
}

template <typename I>
struct CsrColumns {
  using Id = I;
  const I* p;
  __device__ inline I operator()(int64_t i) const { return p[i]; }
};

// ------------------------------------------------------------------ kernels

__global__ void state_init(WindowState* __restrict__ st) {
  if (threadIdx.x == 0) *st = WindowState{0, 0, 0, 0, 0};
}

// Blocks (kTiles: 16-block tiles) of every window, one work-group each.
template <typename I, bool kTiles>
__global__ __launch_bounds__(1024) void count_windows(const I* __restrict__ rowptr, const I* __restrict__ col,
                                                      int64_t rows, int64_t cols, int64_t nnz, int W,
                                                      uint32_t words, uint32_t* __restrict__ nb,
                                                      WindowState* __restrict__ st) {
  extern __shared__ __align__(16) uint32_t bm[];
  __shared__ WindowRows s;
  __shared__ uint32_t s_count;
  const int64_t w = blockIdx.x;
  clear_words(bm, words);
  if (threadIdx.x == 0) s_count = 0;
  load_window(rowptr, rows, nnz, w, W, &s);
  uint32_t held[kHold];
  int bad = s.ok ? 0 : 1;
  set_bits<true>(CsrColumns<I>{col}, s, cols, bm, held, &bad);
  if (bad) st->err = kGeneral;
  __syncthreads();
  uint32_t c = count_bits(bm, words);
  if ((threadIdx.x & 63) == 0 && c != 0) atomicAdd(&s_count, c);
  __syncthreads();
  if (threadIdx.x == 0) nb[w] = kTiles ? (s_count + 15u) / 16u : s_count;
}

// Exclusive sums of nb over the windows, and the plan's record: one
// work-group, kScanPer windows per thread and round.
constexpr int kScanPer = 8;

template <typename I>
__global__ __launch_bounds__(1024) void scan_windows(const uint32_t* __restrict__ nb, int64_t nwin,
                                                     uint32_t* __restrict__ ptr, const I* __restrict__ rowptr,
                                                     int64_t rows, WindowState* __restrict__ st) {
  __shared__ uint32_t s_wave[17];
  uint32_t carry = 0;
  for (int64_t i0 = 0; i0 < nwin; i0 += 1024 * kScanPer) {
    const int64_t a = i0 + static_cast<int64_t>(threadIdx.x) * kScanPer;
    uint32_t v[kScanPer], sum = 0, total;
#pragma unroll
    for (int k = 0; k < kScanPer; ++k) v[k] = a + k < nwin ? nb[a + k] : 0u;
#pragma unroll
    for (int k = 0; k < kScanPer; ++k) sum += v[k];
    uint32_t at = carry + block_exclusive(sum, s_wave, &total);
#pragma unroll
    for (int k = 0; k < kScanPer; ++k) {
      if (a + k < nwin) ptr[a + k] = at;
      at += v[k];
    }
    carry += total;
  }
  if (threadIdx.x == 0) {
    ptr[nwin] = carry;
    st->p_begin = static_cast<int64_t>(rowptr[0]);
    st->n = static_cast<int64_t>(rowptr[rows]) - st->p_begin;
    st->total = carry;
  }
}

// Zeroes n values of a window's output: 16-byte stores where p is aligned.
template <typename U>
__device__ inline void zero_values(U* p, int64_t n) {
  constexpr int kPer = 16 / sizeof(U);
  if (reinterpret_cast<uintptr_t>(p) % 16 == 0) {
    u4_t* q = reinterpret_cast<u4_t*>(p);
    for (int64_t i = threadIdx.x; i < n / kPer; i += blockDim.x) q[i] = u4_t{0u, 0u, 0u, 0u};
    for (int64_t i = n / kPer * kPer + threadIdx.x; i < n; i += blockDim.x) p[i] = static_cast<U>(0);
  } else {
    for (int64_t i = threadIdx.x; i < n; i += blockDim.x) p[i] = static_cast<U>(0);
  }
}

// The work-group's earlier global stores are performed (in its XCD's L2)
// before any of its later ones are issued: its zeros never overtake its
// values.
__device__ inline void stores_done() {
  __asm__ volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
}

// Blocks of 16 values gathered in LDS and written out whole.  A wavefront's
// values go to consecutive blocks at one row, 16 values apart, so block b is
// rotated by b / (blocks per 256 bytes): the 64 lanes then fall on 64 banks.
// Unit: 4 bytes (8 for 8-byte values).
constexpr size_t kTileBytes = 20 * 1024;

template <typename U>
struct ValueTile {
  using Unit = typename std::conditional<sizeof(U) == 8, uint64_t, uint32_t>::type;
  static constexpr uint32_t kPerUnit = sizeof(Unit) / sizeof(U);
  static constexpr uint32_t kUnits = 16 / kPerUnit;  // per block
  static constexpr uint32_t kShift = sizeof(U) == 2 ? 3 : (sizeof(U) == 4 ? 2 : 1);
  static constexpr uint32_t kBlocks = kTileBytes / (16 * sizeof(U));
  Unit* p;
  uint32_t* col;  // [kBlocks]: the blocks' columns
  __device__ inline explicit ValueTile(uint32_t* lds) : p(reinterpret_cast<Unit*>(lds)), col(lds + kTileBytes / 4) {}
  static constexpr size_t kLds = kTileBytes + kBlocks * sizeof(uint32_t);
  __device__ inline uint32_t unit(uint32_t b, uint32_t j) const { return b * kUnits + ((j + (b >> kShift)) & (kUnits - 1)); }
  __device__ inline void set(uint32_t b, uint32_t rr, U v) const {
    reinterpret_cast<U*>(p)[unit(b, rr / kPerUnit) * kPerUnit + rr % kPerUnit] = v;
  }
  template <typename I>
  __device__ inline void write(I* uniq, U* out, uint32_t blocks) const {  // out aligned to a unit
    Unit* q = reinterpret_cast<Unit*>(out);
    for (uint32_t b = threadIdx.x; b < blocks; b += blockDim.x) uniq[b] = static_cast<I>(col[b]);
    for (uint32_t t = threadIdx.x; t < blocks * kUnits; t += blockDim.x) q[t] = p[unit(t / kUnits, t % kUnits)];
  }
};

// csr_to_bcsr / csr_to_ascend_cube outputs of every window, one work-group
// each.  Every nonzero writes its block's column (the same one).
template <typename I, typename U, bool kTiles>
__global__ __launch_bounds__(1024) void write_blocks(const I* __restrict__ rowptr, const I* __restrict__ col,
                                                     const U* __restrict__ val, int64_t rows, int64_t cols,
                                                     int64_t nnz, int W, int64_t nwin, uint32_t words,
                                                     uint32_t groups, int gshift, uint32_t tile_blocks,
                                                     const uint32_t* __restrict__ ptr, I* __restrict__ crow,
                                                     I* __restrict__ uniq, U* __restrict__ out) {
  extern __shared__ __align__(16) uint32_t bm[];
  uint32_t* const prefix = bm + words;
  __shared__ WindowRows s;
  __shared__ uint32_t s_wave[17];
  const int64_t w = blockIdx.x;
  clear_words(bm, words);
  load_window(rowptr, rows, nnz, w, W, &s);
  const uint32_t p0 = ptr[w], p1 = ptr[w + 1];
  if (threadIdx.x == 0) {
    crow[w] = static_cast<I>(p0);
    if (w == nwin - 1) crow[nwin] = static_cast<I>(p1);
  }
  constexpr int64_t kUnit = kTiles ? 256 : 16;  // values per block or tile
  // Windows whose blocks fit the LDS tile are put together there; longer ones
  // (and tile outputs) are zeroed and scattered into in memory.
  const ValueTile<U> tile(prefix + groups);
  const bool staged = !kTiles && p1 - p0 <= tile_blocks &&
                      reinterpret_cast<uintptr_t>(out) % sizeof(typename ValueTile<U>::Unit) == 0;
  if (staged)
    clear_words(reinterpret_cast<uint32_t*>(tile.p), (p1 - p0) * 16 * sizeof(U) / 4);
  else
    zero_values(out + kUnit * p0, kUnit * (p1 - p0));
  if (kTiles)
    for (uint32_t i = threadIdx.x; i < 16u * (p1 - p0); i += blockDim.x) uniq[16 * static_cast<int64_t>(p0) + i] = 0;
  uint32_t held[kHold];
  int bad = 0;
  set_bits<false>(CsrColumns<I>{col}, s, cols, bm, held, &bad);
  const uint32_t T = blockDim.x, n = s.n;
  const bool once = n <= kHold * T;
  U v[kHold];  // windows held in registers load their values ahead of the scan
  if (once) {
#pragma unroll
    for (int k = 0; k < kHold; ++k) {
      const uint32_t i = k * T + threadIdx.x;
      if (i < n) v[k] = val[s.base + i];
    }
  }
  if (staged)
    __syncthreads();  // the bits and the cleared tile are complete
  else
    stores_done();
  bitmap_prefix(bm, prefix, words, gshift, s_wave);
  const RowStarts starts(s);
  U* const out_w = out + kUnit * p0;
  I* const uniq_w = uniq + (kTiles ? 16 : 1) * static_cast<int64_t>(p0);
  for (uint32_t i0 = 0; i0 < n; i0 += kHold * T) {
    if (!once) {
#pragma unroll
      for (int k = 0; k < kHold; ++k) {
        const uint32_t i = i0 + k * T + threadIdx.x;
        if (i < n) {
          v[k] = val[s.base + i];
          held[k] = static_cast<uint32_t>(col[s.base + i]);
        }
      }
    }
#pragma unroll
    for (int k = 0; k < kHold; ++k) {
      const uint32_t i = i0 + k * T + threadIdx.x;
      if (i < n) {
        const uint32_t b = bitmap_rank(bm, prefix, gshift, held[k]);
        const uint32_t rr = starts.row(i);
        if (staged) {
          tile.col[b] = held[k];
          tile.set(b, rr, v[k]);
        } else {
          uniq_w[b] = static_cast<I>(held[k]);
          out_w[kTiles ? 256 * static_cast<int64_t>(b / 16) + 16 * rr + b % 16 : 16 * static_cast<int64_t>(b) + rr] =
              v[k];
        }
      }
    }
  }
  if (staged) {
    __syncthreads();
    tile.write(uniq_w, out_w, p1 - p0);
  }
}

// --------------------------------------------------------------------- host

template <typename F>
spmm_status by_index(int32_t it, F f) {
  if (it == SPMM_INDEX_I32) return f(int32_t{});
  return f(int64_t{});
}

template <typename F>
spmm_status by_value(int32_t vt, F f) {
  if (vt == SPMM_VALUE_F16) return f(uint16_t{});
  if (vt == SPMM_VALUE_F32) return f(uint32_t{});
  return f(uint64_t{});
}

}  // namespace

spmm_status plan_blocks(const Matrix& m, int64_t W, bool tiles, const BlockArrays& a, hipStream_t s) {
  const int64_t nwin = ceil_div(m.rows, W);
  const BitmapShape b(m.cols);
  return by_index(m.index_type, [&](auto i) {
    using I = decltype(i);
    const I* rowptr = static_cast<const I*>(m.rowptr);
    hipLaunchKernelGGL(state_init, dim3(1), dim3(64), 0, s, a.state);
    auto count = tiles ? count_windows<I, true> : count_windows<I, false>;
    hipLaunchKernelGGL(count, dim3(static_cast<unsigned>(nwin)), dim3(b.threads), b.words * sizeof(uint32_t), s, rowptr,
                       static_cast<const I*>(m.col), m.rows, m.cols, m.nnz, static_cast<int>(W), b.words, a.nb,
                       a.state);
    hipLaunchKernelGGL(scan_windows<I>, dim3(1), dim3(1024), 0, s, a.nb, nwin, a.ptr, rowptr, m.rows, a.state);
    return check_launch("window counts");
  });
}

spmm_status fill_blocks(const Matrix& m, int64_t W, bool tiles, const BlockArrays& a, void* crow, void* uniq,
                        void* val, hipStream_t s) {
  const int64_t nwin = ceil_div(m.rows, W);
  const BitmapShape b(m.cols);
  return by_index(m.index_type, [&](auto i) {
    using I = decltype(i);
    return by_value(m.value_type, [&](auto u) {
      using U = decltype(u);
      auto write = tiles ? write_blocks<I, U, true> : write_blocks<I, U, false>;
      // The tile goes beside bitmaps of up to 20 KB (655,000 columns would leave
      // one work-group per CU).
      const uint32_t tile_blocks = !tiles && b.lds() <= 20 * 1024 ? ValueTile<U>::kBlocks : 0;
      const size_t lds = b.lds() + (tile_blocks ? ValueTile<U>::kLds : 0);
      hipLaunchKernelGGL(write, dim3(static_cast<unsigned>(nwin)), dim3(b.threads), lds, s,
                         static_cast<const I*>(m.rowptr), static_cast<const I*>(m.col), static_cast<const U*>(m.value),
                         m.rows, m.cols, m.nnz, static_cast<int>(W), nwin, b.words, b.groups, b.gshift, tile_blocks,
                         a.ptr, static_cast<I*>(crow), static_cast<I*>(uniq), static_cast<U*>(val));
      return check_launch("window blocks");
    });
  });
}

}  // namespace win
}  // namespace spmm
