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
// 1380 us there, 148 us here: counting 31 us, writing 85 us, the read-back
// that sizes the outputs and launches the rest; preprocess of 2.0M power-law
// nonzeros 762 -> 146 us, of a 7.2M-nonzero graph with its packed transpose
// 4079 -> 1109 us).  The splits need no sort of the blocks either: they take
// blocks in order of occupancy, then first nonzero, so counts per occupancy
// give every prefix, and only one window's blocks of one occupancy are ranked.
//
// Bound: vector instructions per nonzero on long windows (about 130 in
// write_blocks, 60 in count_windows).  On short ones each window's own cost:
// the latency of its steps (row pointers, columns, LDS atomics, scan), which the
// other windows resident on the CU cover, and the clears and sweeps of its
// bitmap, one word per 32 columns however few nonzeros there are.  At 262,144
// columns a window of 480 nonzeros clears 8192 words in every kernel and sweeps
// them once to count and twice to rank, about as many wavefront instructions as
// its nonzeros take.  Past some width the sorting pipeline is the faster one
// (window_rule.h).  Work-groups are sized so that a CU holds 1024-2048 threads
// of them: a bitmap of 100,000 columns is 12.5 KB.
#include <rocprim/device/device_radix_sort.hpp>

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "preprocess_windows.h"

namespace spmm {
namespace win {
namespace {

typedef unsigned int u2_t __attribute__((ext_vector_type(2)));
typedef unsigned int u4_t __attribute__((ext_vector_type(4)));

// A plan's error word: take the sorting pipeline; kBadRows: the row pointer
// is not monotone inside [0, nnz].
enum : unsigned long long { kGeneral = 1, kBadRows = 2 };

// Raises err's bits (its kernel's other work-groups may read it meanwhile); by
// one thread of a work-group, as same-address atomics run one after another.
__device__ inline void raise_error(int64_t* err, unsigned long long bits) {
  atomicOr(reinterpret_cast<unsigned long long*>(err), bits);
}

// Plan kernels, at entry, by a thread outside the wavefront that loads the
// window's rows: the plan's first position and nonzeros (window 0; ends may be
// null), and *stop, an LDS word complete at the next barrier: whether err is
// raised already.  One thread reads it, as wavefronts must not each read a word
// that their own launch raises, and only in grids of more work-groups than run
// at once (a load past the L2s: 0.6 us of a conversion of 42).
template <typename P, typename State>
__device__ inline void enter_plan(const P* __restrict__ rowptr, int64_t rows, State* ends, const int64_t* err,
                                  uint32_t* stop) {
  if (threadIdx.x != 64) return;
  *stop = gridDim.x > 4096 && __hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0 ? 1u : 0u;
  if (blockIdx.x == 0 && ends != nullptr) {
    ends->p_begin = static_cast<int64_t>(rowptr[0]);
    ends->n = static_cast<int64_t>(rowptr[rows]) - static_cast<int64_t>(rowptr[0]);
  }
}

// ------------------------------------------------------------- bitmap sizes

// Words per prefix group (1 << gshift: 2 or 8) and LDS layout: bitmap words
// (padded to whole quads), then one prefix count per group.  Two words per
// group make a rank one 8-byte read and two popcounts; larger bitmaps take
// longer groups so that more of them stay resident.
struct BitmapShape {
  uint32_t words, groups;
  int gshift;
  int64_t mean;
  size_t lds() const { return (static_cast<size_t>(words) + groups) * sizeof(uint32_t); }
  BitmapShape(int64_t cols, int64_t nnz, int64_t windows) {
    uint32_t w = static_cast<uint32_t>((cols + 31) / 32);
    gshift = w > 4096 ? 3 : 1;
    const uint32_t gw = gshift == 3 ? 8 : 4;
    words = (w + gw - 1) / gw * gw;
    groups = ((words >> gshift) + 3u) & ~3u;  // what follows stays 16-byte aligned
    mean = nnz / windows;
  }
  // Enough threads that the work-groups a CU's 160 KB of LDS holds keep 16
  // wavefronts on it; windows of a thousand nonzeros or more take at least
  // 512, so that their columns fit registers.
  int threads(size_t lds_bytes) const {
    const size_t fit = 160 * 1024 / (lds_bytes + 512);
    const int t = fit >= 4 ? 256 : (fit >= 2 ? 512 : 1024);
    return t == 256 && mean > 1024 ? 512 : t;
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

// The same in scalar registers: the LDS copy would be read again for every
// nonzero, behind the LDS writes in between, and a scalar base keeps the
// loads' addresses to 32-bit offsets.
struct RowStarts {
  uint32_t off[16];
  uint32_t n;
  int64_t base;
  __device__ inline explicit RowStarts(const WindowRows& s) {
#pragma unroll
    for (int t = 0; t < 16; ++t) off[t] = __builtin_amdgcn_readfirstlane(s.off[t]);
    n = __builtin_amdgcn_readfirstlane(s.n);
    const uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(s.base));
    const uint32_t hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(s.base >> 32));
    base = static_cast<int64_t>(static_cast<uint64_t>(hi) << 32 | lo);
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

// Inclusive sum over the wavefront: DPP moves, which leave the LDS pipe (a
// shuffle's) to the bitmaps.  Whole wavefronts only.
template <int kCtrl, int kRows>
__device__ inline uint32_t dpp_add(uint32_t v) {
  return v + static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), kCtrl, kRows, 0xF, true));
}
__device__ inline uint32_t wave_inclusive(uint32_t v) {
  v = dpp_add<0x111, 0xF>(v);  // lanes 1, 2, 4 and 8 below in the row of 16
  v = dpp_add<0x112, 0xF>(v);
  v = dpp_add<0x114, 0xF>(v);
  v = dpp_add<0x118, 0xF>(v);
  v = dpp_add<0x142, 0xA>(v);  // row ends to the next row, then to the upper half
  v = dpp_add<0x143, 0xC>(v);
  return v;
}
__device__ inline uint64_t wave_inclusive(uint64_t v) {
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint64_t y = __shfl_up(v, o);
    v += lane >= o ? y : 0u;
  }
  return v;
}

// Exclusive scan of one value per thread over the work-group; total in
// *sum (all threads).  s_wave: 17 values of LDS.  Two barriers.
template <typename V>
__device__ inline V block_exclusive(V v, V* s_wave, V* sum) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
  const V x = wave_inclusive(v);
  __syncthreads();  // an earlier scan's sums have been read
  if (lane == 63) s_wave[wave] = x;
  __syncthreads();
  V before = 0, all = 0;
  for (int i = 0; i < waves; ++i) {
    const V t = s_wave[i];
    before += i < wave ? t : V(0);
    all += t;
  }
  *sum = all;
  return before + x - v;
}

// Prefix counts of the bitmap's groups; returns the number of set bits.  Each
// wavefront takes consecutive quads of words, 64 at a time, so that its reads
// meet no bank conflict: a first sweep counts its bits, a second one writes
// the counts before each group.
__device__ inline uint32_t quad_bits(const u4_t& b) {
  return __popc(b[0]) + __popc(b[1]) + __popc(b[2]) + __popc(b[3]);
}

__device__ inline uint32_t bitmap_prefix(const uint32_t* bm, uint32_t* prefix, uint32_t words, int gshift,
                                         uint32_t* s_wave) {
  const uint32_t quads = words / 4, lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
  const uint32_t rounds = (quads + blockDim.x - 1) / blockDim.x;
  const uint32_t first = wave * rounds * 64 + lane;
  const u4_t* q = reinterpret_cast<const u4_t*>(bm);
  uint32_t mine = 0;
  for (uint32_t t = 0; t < rounds; ++t) {
    const uint32_t i = first + t * 64;
    if (i < quads) mine += quad_bits(q[i]);
  }
  const uint32_t sum = wave_inclusive(mine);
  __syncthreads();  // an earlier scan's sums have been read
  if (lane == 63) s_wave[wave] = sum;
  __syncthreads();
  uint32_t at = 0, total = 0;
  for (uint32_t i = 0; i < waves; ++i) {
    const uint32_t t = s_wave[i];
    at += i < wave ? t : 0u;
    total += t;
  }
  for (uint32_t t = 0; t < rounds; ++t) {
    const uint32_t i = first + t * 64;
    const u4_t b = i < quads ? q[i] : u4_t{0u, 0u, 0u, 0u};
    const uint32_t lo = __popc(b[0]) + __popc(b[1]);
    const uint32_t c = lo + __popc(b[2]) + __popc(b[3]);
    const uint32_t in = wave_inclusive(c);
    const uint32_t before = at + in - c;
    if (i < quads) {
      if (gshift == 1) {
        prefix[2 * i] = before;
        prefix[2 * i + 1] = before + lo;
      } else if (gshift == 2) {
        prefix[i] = before;
      } else if ((i & 1u) == 0) {
        prefix[i >> 1] = before;
      }
    }
    at += static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(in), 63));
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

// A window is one work-group's work, so plans hand matrices with a longer
// window than this to the sorting pipeline, which spreads its nonzeros over
// the chip.  One window alone: preprocess 346 us at 32,768 nonzeros and 592 us
// at 65,536, against 472 and 487 us there (block_level_split 292 and 535
// against 360); in a matrix of many nonzeros the sorts cost more (100 windows
// of 64,000: block_level_split 816 us here, 1400 us there; 16 of 131,072: 1097
// against 721 us).
__device__ inline bool long_window(uint32_t n, int64_t nnz) { return n > 32768u && n > nnz / 64; }

// Columns of a window, kHold per thread in registers: windows of at most
// kHold * blockDim.x nonzeros read their columns once per kernel.
constexpr int kHold = 8;

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
__device__ inline void set_bits(const Cols& cols_at, const RowStarts& s, int64_t cols, uint32_t* bm,
                                uint32_t (&held)[kHold], int* bad) {
  using C = typename Cols::Id;
  const Cols col = cols_at.at(s.base);
  const uint32_t n = s.n;
  for (uint32_t i0 = 0; i0 < n; i0 += kHold * blockDim.x) {
    // Through an empty asm: offsets are made per element, not held for all.
    uint32_t T = __builtin_amdgcn_readfirstlane(blockDim.x);
    __asm__ volatile("" : "+s"(T));
    C c[kHold];
#pragma unroll
    for (int k = 0; k < kHold; ++k) {
      const uint32_t i = i0 + k * T + threadIdx.x;
      c[k] = i < n ? col(i) : static_cast<C>(-1);
    }
#pragma unroll
    for (int k = 0; k < kHold; ++k) {
      if (i0 + k * T < n) {  // uniform
        const uint32_t i = i0 + k * T + threadIdx.x;
        bool in = i < n;
        if constexpr (kCheck) {
          C before = static_cast<C>(-1);  // lane 0: the nonzero before the wavefront's
          if ((threadIdx.x & 63) == 0 && in && i > 0) before = col(i - 1);
          const C prev = lane_below(c[k], before);
          if (in && i > 0 && c[k] <= prev) {  // allowed at a row's first nonzero only
            if (!s.starts(i)) *bad = 1;
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

// Columns (values) of a window's nonzeros by offset: at(base) moves to a
// window's first one.
template <typename I>
struct CsrColumns {
  using Id = I;
  const I* __restrict__ p;
  __device__ inline CsrColumns at(int64_t base) const { return CsrColumns{p + base}; }
  __device__ inline I operator()(uint32_t i) const { return p[i]; }
};

// ------------------------------------------------------------------ kernels

// Zeroes a plan's record and n more words.
__global__ void state_init(uint32_t* __restrict__ st, int words, uint32_t* __restrict__ more, int n) {
  for (int i = threadIdx.x; i < words; i += blockDim.x) st[i] = 0u;
  for (int i = threadIdx.x; i < n; i += blockDim.x) more[i] = 0u;
}

template <typename State>
void init_state(State* st, uint32_t* more, int n, hipStream_t s) {
  hipLaunchKernelGGL(state_init, dim3(1), dim3(256), 0, s, reinterpret_cast<uint32_t*>(st),
                     static_cast<int>(sizeof(State) / 4), more, n);
}

// Blocks (kTiles: 16-block tiles) of every window, one work-group each; with
// dkey, also the window's sort key for descending density (the complement of
// the bits of nonzeros / blocks, a non-negative double), its id, and a zeroed
// rank.
template <typename I, bool kTiles, typename State>
__global__ __launch_bounds__(1024) void count_windows(const I* __restrict__ rowptr, const I* __restrict__ col,
                                                      int64_t rows, int64_t cols, int64_t nnz, int W,
                                                      uint32_t words, uint32_t* __restrict__ nb,
                                                      uint64_t* __restrict__ dkey, uint32_t* __restrict__ wid,
                                                      uint32_t* __restrict__ rank, State* __restrict__ st) {
  extern __shared__ __align__(16) uint32_t bm[];
  __shared__ WindowRows s;
  __shared__ uint32_t s_count, s_stop, s_bad;
  const int64_t w = blockIdx.x;
  enter_plan(rowptr, rows, st, &st->err, &s_stop);
  clear_words(bm, words);
  if (threadIdx.x == 0) s_count = s_bad = 0;
  load_window(rowptr, rows, nnz, w, W, &s);
  uint32_t held[kHold];
  int bad = s.ok && !long_window(s.n, nnz) ? 0 : 1;
  // Once a window is bad the counts are of no use: the rest only leave values
  // that the next kernels can go through.  Uniform.
  if (!bad && !s_stop) set_bits<true>(CsrColumns<I>{col}, RowStarts(s), cols, bm, held, &bad);
  if (bad) s_bad = 1;
  __syncthreads();
  uint32_t c = count_bits(bm, words);
  if ((threadIdx.x & 63) == 0 && c != 0) atomicAdd(&s_count, c);
  __syncthreads();
  if (threadIdx.x == 0) {
    if (s_bad) raise_error(&st->err, s.ok ? kGeneral : kGeneral | kBadRows);
    nb[w] = kTiles ? (s_count + 15u) / 16u : s_count;
    if (dkey != nullptr) {
      const double density = s_count ? static_cast<double>(s.n) / static_cast<double>(s_count) : 0.0;
      dkey[w] = ~static_cast<uint64_t>(__double_as_longlong(density));
      wid[w] = static_cast<uint32_t>(w);
      rank[w] = 0u;
    }
  }
}

// Exclusive sums of nb over the windows, and the plan's record: one
// work-group, kScanPer windows per thread and round.
constexpr int kScanPer = 8;

__global__ __launch_bounds__(1024) void scan_windows(const uint32_t* __restrict__ nb, int64_t nwin,
                                                     uint32_t* __restrict__ ptr, WindowState* __restrict__ st) {
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
  __device__ inline uint32_t unit(uint32_t b, uint32_t j) const {
    return b * kUnits + ((j + (b >> kShift)) & (kUnits - 1));
  }
  __device__ inline void set(uint32_t b, uint32_t rr, U v) const {
    reinterpret_cast<U*>(p)[unit(b, rr / kPerUnit) * kPerUnit + rr % kPerUnit] = v;
  }
  template <typename I>
  __device__ inline void write(I* uniq, U* out, uint32_t blocks) const {
    Unit* q = reinterpret_cast<Unit*>(out);  // out is aligned to a unit
    for (uint32_t b = threadIdx.x; b < blocks; b += blockDim.x) uniq[b] = static_cast<I>(col[b]);
    for (uint32_t t = threadIdx.x; t < blocks * kUnits; t += blockDim.x) q[t] = p[unit(t / kUnits, t % kUnits)];
  }
};

// One window's blocks, whole: columns to uniq (and, with packed, the columns'
// packed ids, by position, to renumbered), values to out.  Called by all threads after load_window, with
// the bitmap cleared; `blocks` is their number (kTiles: 16-block tiles).
// Every nonzero writes its block's column (the same one).
template <bool kTiles, typename I, typename U>
__device__ inline void emit_blocks(const WindowRows& s, const I* __restrict__ col, const U* __restrict__ val,
                                   int64_t cols, uint32_t* bm, uint32_t words, uint32_t groups, int gshift,
                                   uint32_t* s_wave, uint32_t tile_blocks, uint32_t blocks, I* __restrict__ uniq,
                                   U* __restrict__ out, const uint32_t* __restrict__ packed,
                                   I* __restrict__ renumbered) {
  uint32_t* const prefix = bm + words;
  constexpr int64_t kUnit = kTiles ? 256 : 16;  // values per block or tile
  // Windows whose blocks fit the LDS tile are put together there; longer ones
  // (and tile outputs) are zeroed and scattered into in memory.
  const ValueTile<U> tile(prefix + groups);
  const bool staged = !kTiles && blocks <= tile_blocks &&
                      reinterpret_cast<uintptr_t>(out) % sizeof(typename ValueTile<U>::Unit) == 0;
  if (staged)
    clear_words(reinterpret_cast<uint32_t*>(tile.p), blocks * 16 * sizeof(U) / 4);
  else
    zero_values(out, kUnit * blocks);
  if (kTiles)
    for (uint32_t i = threadIdx.x; i < 16u * blocks; i += blockDim.x) uniq[i] = 0;
  const RowStarts starts(s);
  const I* const col_w = col + starts.base;
  const U* const val_w = val + starts.base;
  uint32_t held[kHold];
  int bad = 0;
  set_bits<false>(CsrColumns<I>{col}, starts, cols, bm, held, &bad);
  const uint32_t n = starts.n;
  const bool once = n <= kHold * blockDim.x;
  U v[kHold];  // windows held in registers load their values ahead of the scan
  if (once) {
#pragma unroll
    for (int k = 0; k < kHold; ++k) {
      const uint32_t i = k * blockDim.x + threadIdx.x;
      if (i < n) v[k] = val_w[i];
    }
  }
  if (staged)
    __syncthreads();  // the bits and the cleared tile are complete
  else
    stores_done();
  bitmap_prefix(bm, prefix, words, gshift, s_wave);
  for (uint32_t i0 = 0; i0 < n; i0 += kHold * blockDim.x) {
    uint32_t T = __builtin_amdgcn_readfirstlane(blockDim.x);
    __asm__ volatile("" : "+s"(T));
    if (!once) {
#pragma unroll
      for (int k = 0; k < kHold; ++k) {
        const uint32_t i = i0 + k * T + threadIdx.x;
        if (i < n) {
          v[k] = val_w[i];
          held[k] = static_cast<uint32_t>(col_w[i]);
        }
      }
    }
    if (staged) {
#pragma unroll
      for (int k = 0; k < kHold; ++k) {
        const uint32_t i = i0 + k * T + threadIdx.x;
        if (i < n) {
          const uint32_t b = bitmap_rank(bm, prefix, gshift, held[k]);
          tile.col[b] = held[k];
          if (packed != nullptr) renumbered[b] = static_cast<I>(packed[starts.base + i]);
          tile.set(b, starts.row(i), v[k]);
        }
      }
    } else {
#pragma unroll
      for (int k = 0; k < kHold; ++k) {
        const uint32_t i = i0 + k * T + threadIdx.x;
        if (i < n) {
          const uint32_t b = bitmap_rank(bm, prefix, gshift, held[k]);
          const uint32_t rr = starts.row(i);
          uniq[b] = static_cast<I>(held[k]);
          if (packed != nullptr) renumbered[b] = static_cast<I>(packed[starts.base + i]);
          out[kTiles ? 256 * static_cast<int64_t>(b / 16) + 16 * rr + b % 16 : 16 * static_cast<int64_t>(b) + rr] =
              v[k];
        }
      }
    }
  }
  if (staged) {
    __syncthreads();
    tile.write(uniq, out, blocks);
  }
}

// csr_to_bcsr / csr_to_ascend_cube outputs of every window, one work-group each.
template <typename I, typename U, bool kTiles>
__global__ __launch_bounds__(1024) void write_blocks(const I* __restrict__ rowptr, const I* __restrict__ col,
                                                     const U* __restrict__ val, int64_t rows, int64_t cols,
                                                     int64_t nnz, int W, int64_t nwin, uint32_t words,
                                                     uint32_t groups, int gshift, uint32_t tile_blocks,
                                                     const uint32_t* __restrict__ ptr, I* __restrict__ crow,
                                                     I* __restrict__ uniq, U* __restrict__ out) {
  extern __shared__ __align__(16) uint32_t bm[];
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
  emit_blocks<kTiles>(s, col, val, cols, bm, words, groups, gshift, s_wave, tile_blocks, p1 - p0,
                      uniq + (kTiles ? 16 : 1) * static_cast<int64_t>(p0),
                      out + (kTiles ? 256 : 16) * static_cast<int64_t>(p0),
                      static_cast<const uint32_t*>(nullptr), static_cast<I*>(nullptr));
}

// ------------------------------------------------------------------ preprocess

// First i in [lo, hi) with pred(i), hi if none, for a predicate that stays
// true; by one whole wavefront, 64 places a round.
template <typename F>
__device__ inline int64_t first_true(int64_t lo, int64_t hi, F pred) {
  const int lane = threadIdx.x & 63;
  while (lo < hi) {
    const int64_t step = (hi - lo + 64) / 65;
    const int64_t i = lo + (lane + 1) * step - 1;
    const unsigned long long in = __ballot(i < hi);
    const unsigned long long yes = __ballot(i < hi && pred(i));
    if (yes == 0) {
      lo += __popcll(in) * step;
    } else {
      const int f = __ffsll(static_cast<long long>(yes)) - 1;
      hi = lo + (f + 1) * step - 1;
      lo += f * step;
    }
  }
  return hi;
}

// Loads that see other threads' device-scope atomics of the same work-group.
__device__ inline uint32_t fresh(const uint32_t* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <typename P>
__device__ inline uint32_t window_nnz(const P* __restrict__ rowptr, int64_t rows, int64_t w) {
  const int64_t r0 = 16 * w, r1 = r0 + 16 < rows ? r0 + 16 : rows;
  return static_cast<uint32_t>(rowptr[r1] - rowptr[r0]);
}

// The windows in descending density, ties by id: swin[position] = window and
// sbz[position] = blocks << 32 | nonzeros.
//
// rank_windows counts, for 64 windows per wavefront, those that come before
// each among 64 * kRankBlocks of the keys, which it loads 64 at a time and
// hands round by lane reads; place_windows writes the windows to their ranks.
// nwin^2 comparisons, but two launches; past kRankWindows windows the device
// radix sort takes over (six launches, 33 us for 6250 windows) and
// place_windows only fetches the pairs.  Fetching them here spreads the
// gathers over the CUs (one work-group alone took about 2 ns for each).
constexpr int64_t kRankWindows = 8192;
constexpr int64_t kRankBlocks = 2;

__global__ __launch_bounds__(64) void rank_windows(const uint64_t* __restrict__ key, int64_t nwin,
                                                   uint32_t* __restrict__ rank) {
  const int lane = threadIdx.x;
  const int64_t own = blockIdx.x, i = 64 * own + lane;
  auto load = [&](int64_t block) {  // keys past the end come after everything
    const int64_t j = 64 * block + lane;
    return j < nwin ? key[j] : ~uint64_t(0);
  };
  const uint64_t mine = load(own);
  const uint32_t lo = static_cast<uint32_t>(mine), hi = static_cast<uint32_t>(mine >> 32);
  const int64_t blocks = (nwin + 63) / 64;
  const int64_t b0 = blockIdx.y * kRankBlocks, b1 = b0 + kRankBlocks < blocks ? b0 + kRankBlocks : blocks;
  uint32_t before = 0;
  uint64_t keys = load(b0);
  for (int64_t b = b0; b < b1; ++b) {
    const uint64_t next = b + 1 < b1 ? load(b + 1) : 0u;
    const int klo = static_cast<int>(keys), khi = static_cast<int>(keys >> 32);
    // Keys of lower windows count when equal too: less-or-equal, as not (mine < key).
    if (b < own) {
#pragma unroll 16
      for (int u = 0; u < 64; ++u) {
        const uint32_t l = __builtin_amdgcn_readlane(klo, u), h = __builtin_amdgcn_readlane(khi, u);
        before += hi < h || (hi == h && lo < l) ? 0u : 1u;
      }
    } else if (b > own) {
#pragma unroll 16
      for (int u = 0; u < 64; ++u) {
        const uint32_t l = __builtin_amdgcn_readlane(klo, u), h = __builtin_amdgcn_readlane(khi, u);
        before += h < hi || (h == hi && l < lo) ? 1u : 0u;
      }
    } else {
      for (int u = 0; u < 64; ++u) {
        const uint32_t l = __builtin_amdgcn_readlane(klo, u), h = __builtin_amdgcn_readlane(khi, u);
        before += h < hi || (h == hi && (l < lo || (l == lo && u < lane))) ? 1u : 0u;
      }
    }
    keys = next;
  }
  if (i < nwin) atomicAdd(rank + i, before);
}

// rank (of every window), or with rank null swin as the sort left it.
template <typename P>
__global__ __launch_bounds__(256) void place_windows(const uint32_t* __restrict__ rank, int64_t nwin,
                                                     const P* __restrict__ rowptr, int64_t rows,
                                                     const uint32_t* __restrict__ nb, uint32_t* __restrict__ swin,
                                                     uint64_t* __restrict__ sbz, TaskRecord* __restrict__ st) {
  const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t >= nwin) return;
  const int64_t i = rank != nullptr ? t : static_cast<int64_t>(swin[t]), r = rank != nullptr ? rank[t] : t;
  if (rank != nullptr) swin[r] = static_cast<uint32_t>(i);
  sbz[r] = static_cast<uint64_t>(nb[i]) << 32 | (st->err == 0 ? window_nnz(rowptr, rows, i) : 0u);
  if (i == nwin - 1) st->last_pos = r;
}

// The cost model's decisions, by one work-group: prefix sums of blocks and
// nonzeros over the windows in density order, the marginal window (first
// position with (blocks so far) / 295 >= (nonzeros left) / 505), the split of
// its blocks that minimises max(block cost, vector cost), and the sizes.
//
// The marginal window's blocks are taken in order of occupancy (descending),
// then first nonzero, so the nonzeros of the first q blocks follow from the
// 16 occupancy counts, and only the boundary occupancy's blocks need their
// first nonzeros ranked: no sort.
// host_err (or null): a host word that takes the plan's errors so far.
constexpr int kDecidePer = 8;

// blocks / 295 >= nonzeros / 505 in double precision (custom_op.cpp:813-826).
// Where the exact products differ by more than 2^-40 of their sum, the two
// rounded quotients (off by 2^-53 each) compare as they do.
__device__ inline bool block_cost_reaches(int64_t blocks, int64_t nonzeros) {
  const int64_t x = blocks * 505, y = nonzeros * 295, gap = x > y ? x - y : y - x;
  if (gap > (x + y) >> 40) return x > y;
  return static_cast<double>(blocks) / 295.0 >= static_cast<double>(nonzeros) / 505.0;
}

template <typename I>
__global__ __launch_bounds__(1024) void task_decide(const I* __restrict__ rowptr, const I* __restrict__ col,
                                                    int64_t rows, int64_t cols, int64_t nnz, int64_t nwin,
                                                    uint32_t words, uint32_t groups, int gshift, int layout,
                                                    const uint32_t* __restrict__ nb, const uint32_t* __restrict__ swin,
                                                    const uint64_t* __restrict__ sbz, uint32_t* pnb, uint32_t* pnnz,
                                                    uint32_t near_blocks, uint32_t* far_occ, uint32_t* far_first,
                                                    uint32_t* midx, uint32_t* mrow, TaskRecord* st,
                                                    int64_t* host_err) {
  extern __shared__ __align__(16) uint32_t bm[];
  uint32_t* const prefix = bm + words;
  __shared__ WindowRows s;
  __shared__ uint32_t s_wave[17];
  __shared__ int64_t s_q;
  __shared__ uint32_t s_bpos, h[17], cb[17], cn[17], s_rows[17];
  const uint32_t tid = threadIdx.x;
  const int64_t p_begin = st->p_begin, n = st->n;
  const bool part = layout && (p_begin != 0 || n != nnz);
  const int64_t err = st->err;  // raised below only: a wavefront that reads it then leaves as well
  if (tid == 0) {
    if (part) raise_error(&st->err, kGeneral);
    if (host_err != nullptr)
      __hip_atomic_store(host_err, part ? static_cast<int64_t>(kGeneral) : err, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_SYSTEM);
  }
  if (part || err != 0) return;  // uniform
  if (tid == 0) s_bpos = ~0u;
  uint32_t carry_b = 0, carry_z = 0;  // blocks, nonzeros
  __syncthreads();
  for (int64_t i0 = 0; i0 < nwin; i0 += 1024 * kDecidePer) {
    const int64_t a = i0 + static_cast<int64_t>(tid) * kDecidePer;
    uint32_t b[kDecidePer], z[kDecidePer], sum_b = 0, sum_z = 0, all_b, all_z;
    if (a + kDecidePer <= nwin) {  // whole 16-byte loads (sbz is 256-byte aligned)
#pragma unroll
      for (int k = 0; k < kDecidePer; k += 2) {
        const u4_t v = *reinterpret_cast<const u4_t*>(sbz + a + k);
        z[k] = v[0];
        b[k] = v[1];
        z[k + 1] = v[2];
        b[k + 1] = v[3];
      }
    } else {
#pragma unroll
      for (int k = 0; k < kDecidePer; ++k) {
        const uint64_t v = a + k < nwin ? sbz[a + k] : 0u;
        z[k] = static_cast<uint32_t>(v);
        b[k] = static_cast<uint32_t>(v >> 32);
      }
    }
#pragma unroll
    for (int k = 0; k < kDecidePer; ++k) {
      sum_b += b[k];
      sum_z += z[k];
    }
    uint32_t pb = carry_b + block_exclusive(sum_b, s_wave, &all_b);
    uint32_t pz = carry_z + block_exclusive(sum_z, s_wave, &all_z);
    uint32_t found = ~0u;
#pragma unroll
    for (int k = 0; k < kDecidePer; ++k) {
      if (a + k < nwin) {
        pnb[a + k] = pb;
        pnnz[a + k] = pz;
        pb += b[k];
        pz += z[k];
        if (found == ~0u && block_cost_reaches(pb, nnz - static_cast<int64_t>(pz)))
          found = static_cast<uint32_t>(a + k);
      }
    }
    if (found != ~0u) atomicMin(&s_bpos, found);
    carry_b += all_b;
    carry_z += all_z;
  }
  if (tid == 0) {
    pnb[nwin] = carry_b;
    pnnz[nwin] = carry_z;
  }
  stores_done();
  const bool none = s_bpos == ~0u;
  int64_t q = 0, c = 0, bwin = -1;
  uint32_t shared_nnz = 0;
  double est_aic = 0.0, est_aiv = 0.0, est_max = 0.0;
  if (!none) {
    bwin = swin[s_bpos];
    c = nb[bwin];
    // Occupancies, first nonzeros and places of its blocks: in LDS when they fit.
    const bool near = c <= near_blocks;
    uint32_t* const mocc = near ? prefix + groups : far_occ;
    uint32_t* const mfirst = near ? prefix + groups + near_blocks : far_first;
    uint32_t* const place = near ? prefix + groups + 2 * near_blocks : midx;
    auto load = [&](const uint32_t* p) { return near ? *p : fresh(p); };
    const int64_t prefix_blocks = fresh(pnb + s_bpos);
    const int64_t remaining = nnz - fresh(pnnz + s_bpos);
    clear_words(bm, words);
    load_window(rowptr, rows, nnz, bwin, 16, &s);
    uint32_t held[kHold];
    int bad = 0;
    const RowStarts starts(s);
    set_bits<false>(CsrColumns<I>{col}, starts, cols, bm, held, &bad);
    for (uint32_t k = tid; k < c; k += 1024) {
      mocc[k] = 0u;
      mfirst[k] = ~0u;
    }
    if (tid < 17) h[tid] = 0u;
    if (tid < 17) s_rows[tid] = 0u;
    stores_done();
    bitmap_prefix(bm, prefix, words, gshift, s_wave);
    auto block_of = [&](uint32_t i) {
      return bitmap_rank(bm, prefix, gshift, static_cast<uint32_t>(col[s.base + i]));
    };
    for (uint32_t i = tid; i < s.n; i += 1024) {
      const uint32_t k = block_of(i);
      atomicAdd(mocc + k, 1u);
      atomicMin(mfirst + k, i);
    }
    stores_done();
    for (uint32_t k = tid; k < c; k += 1024) atomicAdd(&h[load(mocc + k) & 31u], 1u);  // 1 .. 16: columns are distinct
    __syncthreads();
    if (tid == 0) {
      uint32_t blocks = 0, nz = 0;
      for (int o = 16; o >= 0; --o) {
        cb[o] = blocks;
        cn[o] = nz;
        blocks += h[o];
        nz += h[o] * o;
      }
    }
    __syncthreads();
    // max(block cost, vector cost) with the first k blocks on the block part.
    auto cost = [&](int64_t k, double& aic, double& aiv) {
      int o = 16;
      while (o > 1 && k > static_cast<int64_t>(cb[o]) + h[o]) --o;
      const int64_t assigned = cn[o] + (k - cb[o]) * o;
      aic = static_cast<double>(prefix_blocks + k) / 295.0;
      aiv = static_cast<double>(remaining - assigned) / 505.0;
      return (aic < aiv) ? aiv : aic;
    };
    // The block cost does not shrink with k and the vector cost does not grow,
    // also as computed, so their maximum has its minimum at the first k where
    // the block cost reaches the vector cost, or before it: then at the first
    // k whose vector cost is the least one.
    if (tid < 64) {
      double x, y;
      int64_t k = first_true(0, c + 1, [&](int64_t i) { return cost(i, x, y), x >= y; });
      if (k > 0) {
        const double left = cost(k - 1, x, y);  // its vector cost
        if (k > c || !(cost(k, x, y) < left))
          k = first_true(0, k - 1, [&](int64_t i) { return cost(i, x, y) <= left; });
      }
      if (tid == 0) s_q = k;
    }
    __syncthreads();
    q = s_q;
    est_max = cost(q, est_aic, est_aiv);
    if (q > 0 && q < c) {
      // Boundary occupancy `edge`: `take` of its blocks stay, in order of first nonzero.
      int edge = 16;
      while (edge > 1 && q >= static_cast<int64_t>(cb[edge]) + h[edge]) --edge;
      const uint32_t take = static_cast<uint32_t>(q - cb[edge]);
      for (uint32_t k = tid; k < c; k += 1024) place[k] = load(mocc + k) > static_cast<uint32_t>(edge) ? 1u : 0u;
      stores_done();
      uint32_t before = 0;
      for (uint32_t i0 = 0; i0 < s.n && before < take; i0 += 1024) {
        const uint32_t i = i0 + tid;
        uint32_t k = 0, flag = 0, total;
        if (i < s.n) {
          k = block_of(i);
          flag = load(mocc + k) == static_cast<uint32_t>(edge) && load(mfirst + k) == i ? 1u : 0u;
        }
        const uint32_t at = before + block_exclusive(flag, s_wave, &total);
        if (flag && at < take) place[k] = 1u;
        before += total;
      }
      stores_done();
      uint32_t kept = 0;
      for (uint32_t k0 = 0; k0 < c; k0 += 1024) {
        const uint32_t k = k0 + tid;
        uint32_t total;
        const uint32_t f = k < c ? load(place + k) : 0u;
        const uint32_t at = kept + block_exclusive(f, s_wave, &total);
        if (k < c) place[k] = midx[k] = f ? at : ~0u;
        kept += total;
      }
      stores_done();
      for (uint32_t i = tid; i < s.n; i += 1024)
        if (load(place + block_of(i)) == ~0u) atomicAdd(&s_rows[starts.row(i)], 1u);
      __syncthreads();
      for (int t = 0; t < 16; ++t) {
        if (tid == 0) mrow[t] = shared_nnz;
        shared_nnz += s_rows[t];
      }
      if (tid == 0) mrow[16] = shared_nnz;
    }
  }
  if (tid == 0) {
    const int64_t naic = none ? 0 : static_cast<int64_t>(s_bpos) + (q > 0 ? 1 : 0);
    const int64_t last_rows = rows - 16 * (nwin - 1);
    const int64_t aiv_rows = 16 * (nwin - naic) - (st->last_pos >= naic ? 16 - last_rows : 0);
    st->bpos = none ? -1 : static_cast<int64_t>(s_bpos);
    st->bwin = bwin;
    st->bblocks = c;
    st->baic = q;
    st->shared = q > 0 && q < c ? 1 : 0;
    st->naic = naic;
    st->aic_blocks = none ? 0 : static_cast<int64_t>(fresh(pnb + s_bpos)) + q;
    st->shared_nnz = shared_nnz;
    st->vnnz = shared_nnz + n - fresh(pnnz + naic);
    st->out_rows = layout ? 16 * nwin : 16 * naic + aiv_rows;
    st->est_aic = est_aic;
    st->est_aiv = est_aiv;
    st->est_max = est_max;
  }
}

// First packed row of the window at sorted position i: 16 rows per window,
// except a shorter last window among the vector windows.
__device__ inline int64_t packed_base(const TaskRecord* st, int64_t i, int64_t last_rows) {
  const int64_t last = st->last_pos;
  return 16 * i - (last >= st->naic && i > last ? 16 - last_rows : 0);
}

// inv[row] = packed row (the graph layout's plan needs it; one thread per
// window and row).
__global__ __launch_bounds__(256) void task_inverse(const uint32_t* __restrict__ swin, int64_t nwin, int64_t rows,
                                                    const TaskRecord* __restrict__ st, uint32_t* __restrict__ inv) {
  if (st->err != 0) return;
  const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  const int64_t i = t >> 4;
  if (i >= nwin) return;
  const int64_t r = 16 * static_cast<int64_t>(swin[i]) + (t & 15);
  if (r < rows) inv[r] = static_cast<uint32_t>(packed_base(st, i, rows - 16 * (nwin - 1)) + (t & 15));
}

struct TaskOut {
  void *crow, *uniq, *val, *vrow, *vcol, *vval, *runiq, *rvcol;
  int64_t *perm, *inv;
};

// Packed rows of the window at sorted position i: permutation both ways, row
// pointers (mrow: the shared window's; else v0 + the rows' own offsets, which
// a block window has none of).
template <typename I>
__device__ inline void write_rows(const WindowRows& s, const TaskRecord* st, int64_t i, int64_t w, int64_t nwin,
                                  int64_t rows, bool block_part, const uint32_t* mrow, int64_t v0, const TaskOut& o) {
  I* const vrow = static_cast<I*>(o.vrow);
  const uint32_t tid = threadIdx.x;
  const int64_t last_rows = rows - 16 * (nwin - 1);
  const int64_t row0 = packed_base(st, i, last_rows);
  const int64_t real = w == nwin - 1 ? last_rows : 16;
  if (tid < 16) {
    const int64_t r = 16 * w + tid;
    if (tid < real) {
      o.perm[row0 + tid] = r;
      o.inv[r] = row0 + tid;
    } else if (block_part) {
      o.perm[row0 + tid] = -1;
    }
    if (block_part)
      vrow[row0 + tid] = static_cast<I>(mrow != nullptr ? mrow[tid] : 0u);
    else if (tid < real)
      vrow[row0 + tid] = static_cast<I>(v0 + s.off[tid]);
  }
  if (i == nwin - 1) {
    // Packed rows past the last window's (the graph layout pads to whole windows).
    const int64_t out_rows = st->out_rows;
    for (int64_t r = row0 + (block_part ? 16 : real) + tid; r <= out_rows; r += blockDim.x) {
      vrow[r] = static_cast<I>(st->vnnz);
      if (r < out_rows) o.perm[r] = -1;
    }
  }
  if (i == 0 && tid == 0) static_cast<I*>(o.crow)[st->naic] = static_cast<I>(st->aic_blocks);
}

// Outputs of the vector part's windows (sorted positions from naic on), which
// keep their rows as they are: a copy, and no LDS that would hold back others.
template <typename I, typename U>
__global__ __launch_bounds__(256) void write_vector_rows(const I* __restrict__ rowptr, const I* __restrict__ col,
                                                         const U* __restrict__ val, int64_t rows, int64_t nnz,
                                                         int64_t nwin, int64_t naic,
                                                         const uint32_t* __restrict__ swin,
                                                         const uint32_t* __restrict__ pnnz,
                                                         const TaskRecord* __restrict__ st,
                                                         const uint32_t* __restrict__ packed, TaskOut o) {
  __shared__ WindowRows s;
  const int64_t i = naic + blockIdx.x;
  const int64_t w = swin[i];
  load_window(rowptr, rows, nnz, w, 16, &s);
  const RowStarts starts(s);
  const int64_t v0 = st->shared_nnz + pnnz[i] - pnnz[naic];
  write_rows<I>(s, st, i, w, nwin, rows, false, nullptr, v0, o);
  const I* const col_w = col + starts.base;
  const U* const val_w = val + starts.base;
  I* const vcol = static_cast<I*>(o.vcol) + v0;
  I* const rvcol = packed != nullptr ? static_cast<I*>(o.rvcol) + v0 : nullptr;
  U* const vval = static_cast<U*>(o.vval) + v0;
  constexpr int kU = 4;
  for (uint32_t i0 = 0; i0 < starts.n; i0 += kU * blockDim.x) {
    I c[kU];
    U v[kU];
    uint32_t r[kU];
#pragma unroll
    for (int k = 0; k < kU; ++k) {
      const uint32_t e = i0 + k * blockDim.x + threadIdx.x;
      c[k] = e < starts.n ? col_w[e] : static_cast<I>(0);
      v[k] = e < starts.n ? val_w[e] : static_cast<U>(0);
      r[k] = packed != nullptr && e < starts.n ? packed[starts.base + e] : 0u;
    }
#pragma unroll
    for (int k = 0; k < kU; ++k) {
      const uint32_t e = i0 + k * blockDim.x + threadIdx.x;
      if (e < starts.n) {
        vcol[e] = c[k];
        vval[e] = v[k];
        if (packed != nullptr) rvcol[e] = static_cast<I>(r[k]);
      }
    }
  }
}

// Outputs of the block part's windows (sorted positions below naic).
template <typename I, typename U>
__global__ __launch_bounds__(1024) void write_block_rows(const I* __restrict__ rowptr, const I* __restrict__ col,
                                                         const U* __restrict__ val, int64_t rows, int64_t cols,
                                                         int64_t nnz, int64_t nwin, uint32_t words, uint32_t groups,
                                                         int gshift, uint32_t tile_blocks,
                                                         const uint32_t* __restrict__ swin,
                                                         const uint32_t* __restrict__ nb,
                                                         const uint32_t* __restrict__ pnb,
                                                         const uint32_t* __restrict__ midx,
                                                         const uint32_t* __restrict__ mrow,
                                                         const TaskRecord* __restrict__ st,
                                                         const uint32_t* __restrict__ packed, TaskOut o) {
  extern __shared__ __align__(16) uint32_t bm[];
  __shared__ WindowRows s;
  __shared__ uint32_t s_wave[17];
  const int64_t i = blockIdx.x;
  const int64_t w = swin[i];
  const uint32_t T = blockDim.x, tid = threadIdx.x;
  const bool split = st->shared != 0 && i == st->bpos;
  clear_words(bm, words);
  load_window(rowptr, rows, nnz, w, 16, &s);
  write_rows<I>(s, st, i, w, nwin, rows, true, split ? mrow : nullptr, 0, o);
  const int64_t p0 = pnb[i];
  if (tid == 0) static_cast<I*>(o.crow)[i] = static_cast<I>(p0);
  I* const uniq = static_cast<I*>(o.uniq) + p0;
  I* const runiq = packed != nullptr ? static_cast<I*>(o.runiq) + p0 : nullptr;
  U* const out = static_cast<U*>(o.val) + 16 * p0;
  if (!split) {
    emit_blocks<false>(s, col, val, cols, bm, words, groups, gshift, s_wave, tile_blocks, nb[w], uniq, out, packed,
                       runiq);
    return;
  }
  // The marginal window, shared by both parts: kept blocks at midx, the other
  // nonzeros (the vector part's first) in their order.
  I* const vcol = static_cast<I*>(o.vcol);
  I* const rvcol = static_cast<I*>(o.rvcol);
  U* const vval = static_cast<U*>(o.vval);
  uint32_t* const prefix = bm + words;
  uint32_t held[kHold];
  int bad = 0;
  const RowStarts starts(s);
  zero_values(out, 16 * st->baic);
  set_bits<false>(CsrColumns<I>{col}, starts, cols, bm, held, &bad);
  stores_done();
  bitmap_prefix(bm, prefix, words, gshift, s_wave);
  uint32_t before = 0;
  for (uint32_t i0 = 0; i0 < s.n; i0 += T) {
    const uint32_t e = i0 + tid;
    uint32_t moved = 0, total;
    I c = 0;
    U v = 0;
    if (e < s.n) {
      c = col[s.base + e];
      v = val[s.base + e];
      const uint32_t b = midx[bitmap_rank(bm, prefix, gshift, static_cast<uint32_t>(c))];
      if (b != ~0u) {
        uniq[b] = c;
        if (packed != nullptr) runiq[b] = static_cast<I>(packed[s.base + e]);
        out[16 * static_cast<int64_t>(b) + starts.row(e)] = v;
      } else {
        moved = 1;
      }
    }
    const uint32_t at = before + block_exclusive(moved, s_wave, &total);
    if (moved) {
      vcol[at] = c;
      vval[at] = v;
      if (packed != nullptr) rvcol[at] = static_cast<I>(packed[s.base + e]);
    }
    before += total;
  }
}

// ------------------------------------------------------------------- splits

// Entries of P A^T P^T, in the order of A's nonzeros: key = packed row
// inv[column], word = packed column inv[row] << 32 | the value's bits (the
// nonzero's position for 8-byte values), so a stable sort by key yields the
// transposed arrays themselves.
template <typename I, typename U>
__global__ __launch_bounds__(256) void transpose_pairs(const I* __restrict__ rowptr, const I* __restrict__ col,
                                                       const U* __restrict__ val, int64_t rows, int64_t nnz,
                                                       const TaskRecord* __restrict__ st,
                                                       const uint32_t* __restrict__ inv, uint32_t* __restrict__ key,
                                                       uint64_t* __restrict__ word) {
  __shared__ WindowRows s;
  __shared__ uint32_t s_inv[16];
  if (st->err != 0) return;
  const int64_t w = blockIdx.x;
  if (threadIdx.x < 16) s_inv[threadIdx.x] = 16 * w + threadIdx.x < rows ? inv[16 * w + threadIdx.x] : 0u;
  load_window(rowptr, rows, nnz, w, 16, &s);
  const RowStarts starts(s);
  constexpr int kU = 4;  // nonzeros per thread and round, their loads in flight together
  const I* const col_w = col + starts.base;
  const U* const val_w = val + starts.base;
  for (uint32_t i0 = 0; i0 < starts.n; i0 += kU * blockDim.x) {
    uint32_t c[kU], low[kU];
#pragma unroll
    for (int k = 0; k < kU; ++k) {
      const uint32_t i = i0 + k * blockDim.x + threadIdx.x;
      c[k] = i < starts.n ? static_cast<uint32_t>(col_w[i]) : 0u;
      low[k] = i < starts.n && sizeof(U) < 8 ? static_cast<uint32_t>(val_w[i]) : static_cast<uint32_t>(starts.base) + i;
    }
#pragma unroll
    for (int k = 0; k < kU; ++k) c[k] = inv[c[k]];
#pragma unroll
    for (int k = 0; k < kU; ++k) {
      const uint32_t i = i0 + k * blockDim.x + threadIdx.x;
      if (i < starts.n) {
        key[starts.base + i] = c[k];
        word[starts.base + i] = static_cast<uint64_t>(s_inv[starts.row(i)]) << 32 | low[k];
      }
    }
  }
}

__global__ __launch_bounds__(256) void transpose_starts(const uint32_t* __restrict__ key, int64_t n, int64_t rows,
                                                        const TaskRecord* __restrict__ st, uint32_t* __restrict__ rp) {
  if (st->err != 0) return;
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i > n) return;
  const int64_t prev = i > 0 ? static_cast<int64_t>(key[i - 1]) : -1;
  const int64_t cur = i < n ? static_cast<int64_t>(key[i]) : rows;
  for (int64_t r = prev + 1; r <= cur; ++r) rp[r] = static_cast<uint32_t>(i);
}

struct WordColumns {
  using Id = uint32_t;
  const uint64_t* __restrict__ p;
  __device__ inline WordColumns at(int64_t base) const { return WordColumns{p + base}; }
  __device__ inline uint32_t operator()(uint32_t i) const { return static_cast<uint32_t>(p[i] >> 32); }
};

template <typename U>
struct CsrValues {
  const U* __restrict__ p;
  __device__ inline CsrValues at(int64_t base) const { return CsrValues{p + base}; }
  __device__ inline U operator()(uint32_t i) const { return p[i]; }
};

template <typename U>
struct WordValues {
  const uint64_t* __restrict__ p;
  const U* __restrict__ val;  // 8-byte values: the word holds the nonzero's position
  __device__ inline WordValues at(int64_t base) const { return WordValues{p + base, val}; }
  __device__ inline U operator()(uint32_t i) const {
    const uint32_t low = static_cast<uint32_t>(p[i]);
    if constexpr (sizeof(U) == 8) return val[low];
    else return static_cast<U>(low);
  }
};

// Occupancies of a window's blocks, in LDS up to kOccLds blocks, else in
// global memory; columns' ranks in `prefix`.  `occ` is cleared by the caller.
constexpr uint32_t kOccLds = 768;

template <typename Cols>
__device__ inline void count_occupancy(const Cols& cols_at, const RowStarts& s, const uint32_t* bm,
                                       const uint32_t* prefix, int gshift, uint32_t* occ) {
  const Cols col = cols_at.at(s.base);
  for (uint32_t i = threadIdx.x; i < s.n; i += blockDim.x)
    atomicAdd(occ + bitmap_rank(bm, prefix, gshift, static_cast<uint32_t>(col(i))), 1u);
}

// Blocks per window by occupancy, and their sums over all windows (spread over
// kHistCopies counters: same-address atomics run one after another).  `stop`
// (or null) is an error word of earlier kernels, which makes this one leave;
// it raises its own errors in `err`, a different word: were it the same one,
// the wavefronts of a work-group could read it before and after another
// work-group's store, and those that stayed would use the LDS of those that
// left, and write by it.  `ends` (or null) takes the first position and the
// number of nonzeros.
template <typename P, typename Cols, bool kCheck>
__global__ __launch_bounds__(1024) void split_counts(const P* __restrict__ rowptr, Cols col, int64_t rows,
                                                     int64_t cols, int64_t nnz, int W, uint32_t words, uint32_t groups,
                                                     int gshift, uint32_t* __restrict__ nb, uint32_t* __restrict__ hist,
                                                     uint32_t* __restrict__ total, uint32_t* occ_far,
                                                     const int64_t* stop, int64_t* err, WindowState* ends) {
  extern __shared__ __align__(16) uint32_t bm[];
  uint32_t* const prefix = bm + words;
  __shared__ WindowRows s;
  __shared__ uint32_t s_wave[17], s_hist[32], s_stop;
  if (stop != nullptr && *stop != 0) return;  // uniform: not written in this launch
  const int64_t w = blockIdx.x;
  if (kCheck) enter_plan(rowptr, rows, ends, err, &s_stop);  // the transpose's errors are a few long windows
  clear_words(bm, words);
  if (threadIdx.x < 32) s_hist[threadIdx.x] = 0u;
  load_window(rowptr, rows, nnz, w, W, &s);
  uint32_t held[kHold];
  int bad = s.ok && !long_window(s.n, nnz) ? 0 : 1;
  const RowStarts starts(s);
  if (!bad && !(kCheck && s_stop)) set_bits<kCheck>(col, starts, cols, bm, held, &bad);  // uniform
  if (__syncthreads_or(bad)) {
    if (threadIdx.x == 0) raise_error(err, s.ok ? kGeneral : kGeneral | kBadRows);
    return;
  }
  if (kCheck && s_stop) return;
  const uint32_t blocks = bitmap_prefix(bm, prefix, words, gshift, s_wave);
  const bool near = blocks <= kOccLds;
  uint32_t* const occ = near ? prefix + groups : occ_far + s.base;
  for (uint32_t k = threadIdx.x; k < blocks; k += blockDim.x) occ[k] = 0u;
  stores_done();
  count_occupancy(col, starts, bm, prefix, gshift, occ);
  stores_done();
  for (uint32_t k0 = 0; k0 < blocks; k0 += blockDim.x) {
    const uint32_t k = k0 + threadIdx.x;
    const uint32_t o = k < blocks ? (near ? occ[k] : fresh(occ + k)) : 0u;
    const unsigned long long ones = __ballot(o == 1u);  // most blocks of a scattered matrix
    if ((threadIdx.x & 63) == 0 && ones) atomicAdd(&s_hist[1], static_cast<uint32_t>(__popcll(ones)));
    if (o > 1u) atomicAdd(&s_hist[o & 31u], 1u);
  }
  __syncthreads();
  if (threadIdx.x < 16) {
    const uint32_t v = s_hist[threadIdx.x + 1];
    hist[threadIdx.x * static_cast<int64_t>(gridDim.x) + w] = v;
    if (v) atomicAdd(total + 16 * (w % kHistCopies) + threadIdx.x, v);
  }
  if (threadIdx.x == 0) nb[w] = blocks;
}

// |ratio(k) - a| of the split after its first k blocks, ratio = blocks left /
// nonzeros moved (custom_op.cpp:1207-1220), from the occupancy counts.
struct SplitCost {
  uint32_t below[18], moved[18];  // blocks and nonzeros of lower occupancies
  int64_t blocks;
  double a;
  __device__ inline double ratio(int64_t k) const {
    int o = 1;
    while (o < 16 && k > static_cast<int64_t>(below[o + 1])) ++o;
    const int64_t nz = moved[o] + (k - below[o]) * o;
    const int64_t rem = blocks - k;
    return nz == 0 ? (rem > 0 ? INFINITY : 0.0) : static_cast<double>(rem) / static_cast<double>(nz);
  }
  __device__ inline double diff(int64_t k) const { return fabs(ratio(k) - a); }
};

// Which blocks move to the CSR part: the first k of the order (occupancy,
// first nonzero), k the first minimum of SplitCost::diff.  ratio(k) does not
// grow with k, also as computed (one rounded division of exact integers), so
// diff does not grow up to the first k with ratio <= a and does not shrink
// after it: the minimum is at that k or before it, and binary searches find
// its first place.  Then, per window, its share of the boundary occupancy's
// blocks, and prefix sums of kept blocks and moved nonzeros.  One work-group.
// stop, err: as for split_counts, written by earlier kernels only.
__global__ __launch_bounds__(1024) void split_decide(int64_t nwin, double a,
                                                     const uint32_t* __restrict__ nb,
                                                     const uint32_t* __restrict__ hist,
                                                     const uint32_t* __restrict__ total, uint32_t* __restrict__ moved,
                                                     uint32_t* __restrict__ kptr, uint32_t* __restrict__ vptr,
                                                     uint32_t* __restrict__ rule, const int64_t* stop,
                                                     const int64_t* err, int64_t* kept_out, int64_t* vnnz_out) {
  __shared__ SplitCost f;
  __shared__ uint32_t s_wave[17], s_h[16], s_edge;
  __shared__ uint64_t s_wave64[17];
  __shared__ int64_t s_k;
  const uint32_t tid = threadIdx.x;
  if (*err != 0 || (stop != nullptr && *stop != 0)) return;
  if (tid < 16) s_h[tid] = 0u;
  __syncthreads();
  for (uint32_t t = tid; t < 16 * kHistCopies; t += 1024) {
    const uint32_t v = total[t];
    if (v) atomicAdd(&s_h[t & 15u], v);
  }
  __syncthreads();
  if (tid == 0) {
    uint32_t b = 0, z = 0;
    f.below[0] = f.moved[0] = 0u;
    for (int o = 1; o <= 16; ++o) {
      f.below[o] = b;
      f.moved[o] = z;
      b += s_h[o - 1];
      z += s_h[o - 1] * o;
    }
    f.below[17] = b;
    f.moved[17] = z;
    f.blocks = b;
    f.a = a;
  }
  __syncthreads();
  if (tid < 64) {
    int64_t k = 0;
    if (f.blocks > 0 && isfinite(a)) {  // else no finite minimum: nothing moves
      const int64_t at = first_true(1, f.blocks + 1, [&](int64_t i) { return f.ratio(i) <= a; });
      if (at == 1 || (at <= f.blocks && f.diff(at) < f.diff(at - 1))) {
        k = at;
      } else {
        const double least = f.diff(at - 1);
        k = first_true(1, at - 1, [&](int64_t i) { return f.diff(i) <= least; });
      }
    }
    int edge = 1;
    while (edge < 16 && k >= static_cast<int64_t>(f.below[edge + 1])) ++edge;
    if (tid == 0) {
      s_k = k - f.below[edge];  // blocks of occupancy `edge` that move
      s_edge = static_cast<uint32_t>(edge);
      *rule = static_cast<uint32_t>(edge);
    }
  }
  __syncthreads();
  const int edge = static_cast<int>(s_edge);
  const uint32_t take = static_cast<uint32_t>(s_k);
  constexpr int kPer = 4;
  uint32_t before = 0;
  uint64_t carry = 0;  // kept blocks << 32 | moved nonzeros
  for (int64_t w0 = 0; w0 < nwin; w0 += 1024 * kPer) {
    const int64_t i = w0 + static_cast<int64_t>(tid) * kPer;
    uint32_t at_edge[kPer], low_blocks[kPer], low_nnz[kPer], blocks[kPer], sum = 0, all;
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
      at_edge[k] = low_blocks[k] = low_nnz[k] = 0u;
      blocks[k] = i + k < nwin ? nb[i + k] : 0u;
    }
    for (int o = 1; o <= edge; ++o) {
      const uint32_t* const h = hist + (o - 1) * nwin;
#pragma unroll
      for (int k = 0; k < kPer; ++k) {
        const uint32_t v = i + k < nwin ? h[i + k] : 0u;
        low_blocks[k] += o < edge ? v : 0u;
        low_nnz[k] += o < edge ? v * o : 0u;
        at_edge[k] = v;
      }
    }
#pragma unroll
    for (int k = 0; k < kPer; ++k) sum += at_edge[k];
    uint32_t at = before + block_exclusive(sum, s_wave, &all);
    before += all;
    uint64_t mine = 0, whole;
    uint32_t kept[kPer], nz[kPer];
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
      const uint32_t m = at >= take ? 0u : (take - at < at_edge[k] ? take - at : at_edge[k]);
      at += at_edge[k];
      kept[k] = blocks[k] - low_blocks[k] - m;
      nz[k] = low_nnz[k] + m * static_cast<uint32_t>(edge);
      if (i + k < nwin) moved[i + k] = m;
      mine += static_cast<uint64_t>(kept[k]) << 32 | nz[k];
    }
    uint64_t pos = carry + block_exclusive(mine, s_wave64, &whole);
    carry += whole;
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
      if (i + k < nwin) {
        kptr[i + k] = static_cast<uint32_t>(pos >> 32);
        vptr[i + k] = static_cast<uint32_t>(pos);
      }
      pos += static_cast<uint64_t>(kept[k]) << 32 | nz[k];
    }
  }
  if (tid == 0) {
    kptr[nwin] = static_cast<uint32_t>(carry >> 32);
    vptr[nwin] = static_cast<uint32_t>(carry);
    *kept_out = static_cast<int64_t>(carry >> 32);
    *vnnz_out = static_cast<int64_t>(carry & 0xFFFFFFFFu);
  }
}

// A window's outputs of the split.
template <typename P, typename Cols, typename Vals, typename O, typename U>
__global__ __launch_bounds__(1024) void write_split(const P* __restrict__ rowptr, Cols cols_at, Vals vals_at,
                                                    int64_t rows, int64_t cols, int64_t nnz, int W, int64_t nwin,
                                                    uint32_t words, uint32_t groups, int gshift, SplitArrays x,
                                                    O* __restrict__ crow, O* __restrict__ uniq, U* __restrict__ out,
                                                    O* __restrict__ vrow, O* __restrict__ vcol, U* __restrict__ vval) {
  extern __shared__ __align__(16) uint32_t bm[];
  uint32_t* const prefix = bm + words;
  __shared__ WindowRows s;
  __shared__ uint32_t s_wave[17], s_vrow[17];
  const int64_t w = blockIdx.x;
  const uint32_t T = blockDim.x, tid = threadIdx.x;
  const uint32_t k0 = x.kptr[w], kept = x.kptr[w + 1] - k0, blocks = x.nb[w];
  const int64_t v0 = x.vptr[w];
  const uint32_t v_n = x.vptr[w + 1] - x.vptr[w];
  if (kept != 0) clear_words(bm, words);
  load_window(rowptr, rows, nnz, w, W, &s);
  if (tid == 0) {
    crow[w] = static_cast<O>(k0);
    if (w == nwin - 1) {
      crow[nwin] = static_cast<O>(k0 + kept);
      vrow[nwin * W] = static_cast<O>(v0 + v_n);
    }
  }
  const RowStarts starts(s);
  const Cols col = cols_at.at(starts.base);
  const Vals val = vals_at.at(starts.base);
  const uint32_t n = starts.n;
  if (kept == 0) {  // the rows as they are
    if (tid < static_cast<uint32_t>(W)) vrow[w * W + tid] = static_cast<O>(v0 + s.off[tid]);
    for (uint32_t i = tid; i < n; i += T) {
      vcol[v0 + i] = static_cast<O>(col(i));
      vval[v0 + i] = val(i);
    }
    return;
  }
  U* const out_w = out + static_cast<int64_t>(W) * k0;
  O* const uniq_w = uniq + k0;
  zero_values(out_w, static_cast<int64_t>(W) * kept);
  uint32_t held[kHold];
  int bad = 0;
  set_bits<false>(cols_at, starts, cols, bm, held, &bad);
  if (tid < 17) s_vrow[tid] = v_n;
  stores_done();
  bitmap_prefix(bm, prefix, words, gshift, s_wave);
  const bool mixed = v_n != 0;
  const bool near = blocks <= kOccLds;
  uint32_t* const occ = near ? prefix + groups : x.occ + s.base;
  if (mixed) {
    const uint32_t edge = *x.rule, m = x.moved[w], at_edge = x.hist[(edge - 1) * nwin + w];
    for (uint32_t k = tid; k < blocks; k += T) occ[k] = 0u;
    const bool part = m != 0 && m != at_edge;  // this window holds the boundary
    if (part)
      for (uint32_t k = tid; k < blocks; k += T) x.first[k] = ~0u;
    stores_done();
    count_occupancy(cols_at, starts, bm, prefix, gshift, occ);
    auto block_of = [&](uint32_t i) {
      return bitmap_rank(bm, prefix, gshift, static_cast<uint32_t>(col(i)));
    };
    auto load = [&](uint32_t k) { return near ? occ[k] : fresh(occ + k); };
    constexpr uint32_t kMoved = 0x80000000u;
    if (part) {
      for (uint32_t i = tid; i < n; i += T) atomicMin(x.first + block_of(i), i);
      stores_done();
      uint32_t before = 0;
      for (uint32_t i0 = 0; i0 < n && before < m; i0 += T) {
        const uint32_t i = i0 + tid;
        uint32_t k = 0, flag = 0, total;
        if (i < n) {
          k = block_of(i);
          flag = (load(k) & ~kMoved) == edge && fresh(x.first + k) == i ? 1u : 0u;
        }
        const uint32_t at = before + block_exclusive(flag, s_wave, &total);
        if (flag && at < m) occ[k] = edge | kMoved;
        before += total;
      }
    }
    stores_done();
    // Kept blocks' places, in column order.
    uint32_t before = 0;
    for (uint32_t b0 = 0; b0 < blocks; b0 += T) {
      const uint32_t k = b0 + tid;
      uint32_t total;
      const uint32_t o = k < blocks ? load(k) : 0u;
      const bool keep = k < blocks && (o & kMoved) == 0u && (o > edge || (o == edge && (part || m == 0)));
      const uint32_t at = before + block_exclusive(keep ? 1u : 0u, s_wave, &total);
      if (k < blocks) occ[k] = keep ? at : ~0u;
      before += total;
    }
    stores_done();
  }
  uint32_t before = 0;
  for (uint32_t i0 = 0; i0 < n; i0 += T) {
    const uint32_t i = i0 + tid;
    uint32_t c = 0, moved = 0;
    U v = 0;
    if (i < n) {
      c = static_cast<uint32_t>(col(i));
      v = val(i);
      uint32_t b = bitmap_rank(bm, prefix, gshift, c);
      if (mixed) b = near ? occ[b] : fresh(occ + b);
      if (b != ~0u) {
        uniq_w[b] = static_cast<O>(c);
        out_w[static_cast<int64_t>(W) * b + starts.row(i)] = v;
      } else {
        moved = 1;
      }
    }
    if (mixed) {  // uniform
      uint32_t total;
      const uint32_t at = before + block_exclusive(moved, s_wave, &total);
      if (moved) {
        vcol[v0 + at] = static_cast<O>(c);
        vval[v0 + at] = v;
      }
      if (i < n && (i == 0 || starts.starts(i)))  // first nonzero of one or more rows (empty ones share it)
        for (int t = 0; t < 16; ++t)
          if (s.off[t] == i) s_vrow[t] = at;
      before += total;
    }
  }
  __syncthreads();
  if (tid < static_cast<uint32_t>(W)) vrow[w * W + tid] = static_cast<O>(v0 + (mixed ? s_vrow[tid] : 0u));
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

namespace {
// The LDS tile goes beside bitmaps of up to 20 KB; larger ones leave too few
// work-groups per CU with it.
template <typename U>
uint32_t tile_capacity(const BitmapShape& b) {
  return b.lds() <= 20 * 1024 ? ValueTile<U>::kBlocks : 0;
}
}  // namespace

spmm_status plan_blocks(const Matrix& m, int64_t W, bool tiles, const BlockArrays& a, hipStream_t s) {
  const int64_t nwin = ceil_div(m.rows, W);
  const BitmapShape b(m.cols, m.nnz, nwin);
  return by_index(m.index_type, [&](auto i) {
    using I = decltype(i);
    const I* rowptr = static_cast<const I*>(m.rowptr);
    init_state(a.state, nullptr, 0, s);
    const size_t lds = b.words * sizeof(uint32_t);
    auto count = tiles ? count_windows<I, true, WindowState> : count_windows<I, false, WindowState>;
    hipLaunchKernelGGL(count, dim3(static_cast<unsigned>(nwin)), dim3(b.threads(lds)), lds, s, rowptr,
                       static_cast<const I*>(m.col), m.rows, m.cols, m.nnz, static_cast<int>(W), b.words, a.nb,
                       static_cast<uint64_t*>(nullptr), static_cast<uint32_t*>(nullptr),
                       static_cast<uint32_t*>(nullptr), a.state);
    hipLaunchKernelGGL(scan_windows, dim3(1), dim3(1024), 0, s, a.nb, nwin, a.ptr, a.state);
    return check_launch("window counts");
  });
}

spmm_status fill_blocks(const Matrix& m, int64_t W, bool tiles, const BlockArrays& a, void* crow, void* uniq,
                        void* val, hipStream_t s) {
  const int64_t nwin = ceil_div(m.rows, W);
  const BitmapShape b(m.cols, m.nnz, nwin);
  return by_index(m.index_type, [&](auto i) {
    using I = decltype(i);
    return by_value(m.value_type, [&](auto u) {
      using U = decltype(u);
      auto write = tiles ? write_blocks<I, U, true> : write_blocks<I, U, false>;
      const uint32_t tile_blocks = tiles ? 0 : tile_capacity<U>(b);
      const size_t lds = b.lds() + (tile_blocks ? ValueTile<U>::kLds : 0);
      hipLaunchKernelGGL(write, dim3(static_cast<unsigned>(nwin)), dim3(b.threads(lds)), lds, s,
                         static_cast<const I*>(m.rowptr), static_cast<const I*>(m.col), static_cast<const U*>(m.value),
                         m.rows, m.cols, m.nnz, static_cast<int>(W), nwin, b.words, b.groups, b.gshift, tile_blocks,
                         a.ptr, static_cast<I*>(crow), static_cast<I*>(uniq), static_cast<U*>(val));
      return check_launch("window blocks");
    });
  });
}

// ------------------------------------------------------------ split, host

namespace {

template <typename P, typename Cols, bool kCheck>
spmm_status run_split(const P* rowptr, Cols col, int64_t rows, int64_t cols, int64_t nnz, double a, int64_t W,
                      const SplitArrays& x, const int64_t* stop, int64_t* err, WindowState* ends, int64_t* kept,
                      int64_t* vnnz, hipStream_t s) {
  const int64_t nwin = ceil_div(rows, W);
  const BitmapShape b(cols, nnz, nwin);
  const size_t lds = b.lds() + kOccLds * sizeof(uint32_t);
  hipLaunchKernelGGL((split_counts<P, Cols, kCheck>), dim3(static_cast<unsigned>(nwin)), dim3(b.threads(lds)), lds, s,
                     rowptr, col, rows, cols, nnz, static_cast<int>(W), b.words, b.groups, b.gshift, x.nb, x.hist,
                     x.total, x.occ, stop, err, ends);
  hipLaunchKernelGGL(split_decide, dim3(1), dim3(1024), 0, s, nwin, a, x.nb, x.hist, x.total, x.moved, x.kptr, x.vptr,
                     x.rule, stop, static_cast<const int64_t*>(err), kept, vnnz);
  return check_launch("split counts");
}

template <typename P, typename Cols, typename Vals, typename O, typename U>
spmm_status launch_split_fill(const P* rowptr, Cols col, Vals val, int64_t rows, int64_t cols, int64_t nnz, int64_t W,
                              const SplitArrays& x, void* crow, void* uniq, U* out, void* vrow, void* vcol, U* vval,
                              hipStream_t s) {
  const int64_t nwin = ceil_div(rows, W);
  const BitmapShape b(cols, nnz, nwin);
  const size_t lds = b.lds() + kOccLds * sizeof(uint32_t);
  hipLaunchKernelGGL((write_split<P, Cols, Vals, O, U>), dim3(static_cast<unsigned>(nwin)), dim3(b.threads(lds)), lds,
                     s, rowptr, col, val, rows, cols, nnz, static_cast<int>(W), nwin, b.words, b.groups, b.gshift, x,
                     static_cast<O*>(crow), static_cast<O*>(uniq), out, static_cast<O*>(vrow), static_cast<O*>(vcol),
                     vval);
  return check_launch("split outputs");
}

}  // namespace

spmm_status plan_split(const Matrix& m, double a, int64_t W, const SplitArrays& x, WindowState* state, hipStream_t s) {
  return by_index(m.index_type, [&](auto i) {
    using I = decltype(i);
    init_state(state, x.total, 16 * kHistCopies, s);
    return run_split<I, CsrColumns<I>, true>(static_cast<const I*>(m.rowptr),
                                             CsrColumns<I>{static_cast<const I*>(m.col)}, m.rows, m.cols, m.nnz, a, W,
                                             x, nullptr, &state->err, state, &state->total, &state->vnnz, s);
  });
}

spmm_status fill_split(const Matrix& m, int64_t W, const SplitArrays& x, void* crow, void* uniq, void* val, void* vrow,
                       void* vcol, void* vval, hipStream_t s) {
  return by_index(m.index_type, [&](auto i) {
    using I = decltype(i);
    return by_value(m.value_type, [&](auto u) {
      using U = decltype(u);
      return launch_split_fill<I, CsrColumns<I>, CsrValues<U>, I, U>(
          static_cast<const I*>(m.rowptr), CsrColumns<I>{static_cast<const I*>(m.col)},
          CsrValues<U>{static_cast<const U*>(m.value)}, m.rows, m.cols, m.nnz, W, x, crow, uniq, static_cast<U*>(val),
          vrow, vcol, static_cast<U*>(vval), s);
    });
  });
}

// ------------------------------------------------------- preprocess, host

namespace {

int key_bits(uint64_t max_value) {
  int b = 1;
  while (b < 64 && (max_value >> b) != 0) ++b;
  return b;
}

}  // namespace

bool ends_known(int64_t err) { return (err & static_cast<int64_t>(kBadRows)) == 0; }

namespace {

// A pinned word per host thread, freed when the thread ends.
struct HostWord {
  int64_t* p = nullptr;
  ~HostWord() {
    if (p != nullptr) (void)hipHostFree(p);
  }
  int64_t* get() {
    if (p == nullptr &&
        hipHostMalloc(reinterpret_cast<void**>(&p), sizeof *p, hipHostMallocPortable | hipHostMallocCoherent) !=
            hipSuccess) {
      (void)hipGetLastError();
      p = nullptr;
    }
    return p;
  }
};
thread_local HostWord host_word;

// A value that a kernel of this call stores to the thread's word, which the
// host looks at while the stream goes on.
struct Awaited {
  static constexpr int64_t kPending = -1;
  int64_t* word;
  hipStream_t stream;
  bool due = false;  // the store has been launched and not been seen
  Awaited(bool wanted, hipStream_t s) : word(wanted ? host_word.get() : nullptr), stream(s) {
    if (word != nullptr) __atomic_store_n(word, kPending, __ATOMIC_SEQ_CST);
  }
  // The stored value; 0 without a word, or once the stream has run dry.
  spmm_status wait(int64_t* value) {
    *value = 0;
    if (!due) return SPMM_OK;
    for (uint32_t looks = 1;; ++looks) {
      int64_t v = __atomic_load_n(word, __ATOMIC_ACQUIRE);
      // Rarely, tenths of a second apart: the query puts a marker in the stream
      // (6 us between two kernels).
      if (v == kPending && looks % (1u << 27) == 0) {
        const hipError_t e = hipStreamQuery(stream);
        if (e != hipSuccess && e != hipErrorNotReady) return check_hip(e, "waiting for the counts");
        if (e == hipSuccess && (v = __atomic_load_n(word, __ATOMIC_ACQUIRE)) == kPending) v = 0;
      }
      if (v != kPending) {
        due = false;
        *value = v;
        return SPMM_OK;
      }
    }
  }
  ~Awaited() {  // after an error: no store may come once the word serves another call
    if (due) (void)hipStreamSynchronize(stream);
  }
};

}  // namespace

size_t task_temp_bytes(const Matrix& m, bool layout) {
  size_t a = 0, b = 0;
  const size_t nwin = static_cast<size_t>(ceil_div(m.rows, 16));
  (void)rocprim::radix_sort_pairs(nullptr, a, static_cast<const uint64_t*>(nullptr), static_cast<uint64_t*>(nullptr),
                                  static_cast<const uint32_t*>(nullptr), static_cast<uint32_t*>(nullptr), nwin, 0, 64);
  if (layout)
    (void)rocprim::radix_sort_pairs(nullptr, b, static_cast<const uint32_t*>(nullptr), static_cast<uint32_t*>(nullptr),
                                    static_cast<const uint64_t*>(nullptr), static_cast<uint64_t*>(nullptr),
                                    static_cast<size_t>(m.nnz), 0, 32);
  return a > b ? a : b;
}

spmm_status plan_task(const Matrix& m, bool layout, const TaskArrays& x, bool* handed_over, hipStream_t s) {
  *handed_over = false;
  const int64_t nwin = ceil_div(m.rows, 16);
  // The sort of the transposed entries, a fifth of the plan, is not started for
  // a matrix that the counts hand over: task_decide first stores their error
  // word to a host word, and the host launches the sort while the GPU is still at
  // work on the rest of task_decide.
  Awaited counts_err(layout, s);
  const BitmapShape b(m.cols, m.nnz, nwin);
  return by_index(m.index_type, [&](auto i) {
    using I = decltype(i);
    const I* rowptr = static_cast<const I*>(m.rowptr);
    const I* col = static_cast<const I*>(m.col);
    init_state(x.record, layout ? x.split.total : nullptr, layout ? 16 * kHistCopies : 0, s);
    const size_t count_lds = b.words * sizeof(uint32_t);
    hipLaunchKernelGGL((count_windows<I, false, TaskRecord>), dim3(static_cast<unsigned>(nwin)),
                       dim3(b.threads(count_lds)), count_lds, s, rowptr, col, m.rows, m.cols, m.nnz, 16, b.words, x.nb,
                       x.dkey, x.wid, x.rank, x.record);
    if (spmm_status st = check_launch("window counts")) return st;
    size_t bytes = x.temp_bytes;
    const bool ranked = nwin <= kRankWindows;
    if (ranked) {
      const int64_t key_blocks = ceil_div(nwin, 64);
      hipLaunchKernelGGL(rank_windows,
                         dim3(static_cast<unsigned>(key_blocks),
                              static_cast<unsigned>(ceil_div(key_blocks, kRankBlocks))),
                         dim3(64), 0, s, x.dkey, nwin, x.rank);
    } else if (hipError_t e = rocprim::radix_sort_pairs(x.temp, bytes, static_cast<const uint64_t*>(x.dkey), x.sdkey,
                                                        static_cast<const uint32_t*>(x.wid), x.swin,
                                                        static_cast<size_t>(nwin), 0, 64, s)) {
      return check_hip(e, "density sort");
    }
    hipLaunchKernelGGL(place_windows<I>, dim3(static_cast<unsigned>(ceil_div(nwin, 256))), dim3(256), 0, s,
                       ranked ? x.rank : static_cast<const uint32_t*>(nullptr), nwin, rowptr, m.rows, x.nb, x.swin,
                       x.sbz, x.record);
    const uint32_t near_blocks =
        b.lds() <= 100 * 1024 ? static_cast<uint32_t>((152 * 1024 - b.lds()) / (3 * sizeof(uint32_t)) / 4 * 4) : 0;
    hipLaunchKernelGGL(task_decide<I>, dim3(1), dim3(1024), b.lds() + 3 * near_blocks * sizeof(uint32_t), s, rowptr,
                       col, m.rows, m.cols, m.nnz, nwin, b.words, b.groups, b.gshift, layout ? 1 : 0, x.nb, x.swin,
                       x.sbz, x.pnb, x.pnnz, near_blocks, x.mocc, x.mfirst, x.midx, x.mrow, x.record, counts_err.word);
    if (spmm_status st = check_launch("task mapping")) return st;
    counts_err.due = counts_err.word != nullptr;
    if (!layout) return SPMM_OK;
    // P A^T P^T and its fixed 295/505 split.
    hipLaunchKernelGGL(task_inverse, dim3(static_cast<unsigned>(ceil_div(16 * nwin, 256))), dim3(256), 0, s, x.swin,
                       nwin, m.rows, x.record, x.inv);
    if (spmm_status st = by_value(m.value_type, [&](auto u) {
          using U = decltype(u);
          hipLaunchKernelGGL((transpose_pairs<I, U>), dim3(static_cast<unsigned>(nwin)), dim3(256), 0, s, rowptr, col,
                             static_cast<const U*>(m.value), m.rows, m.nnz, x.record, x.inv, x.tkey, x.tword);
          return check_launch("transpose keys");
        }))
      return st;
    int64_t err = 0;
    if (spmm_status st = counts_err.wait(&err)) return st;
    if (err != 0) {
      *handed_over = true;
      return SPMM_OK;
    }
    bytes = x.temp_bytes;
    if (hipError_t e = rocprim::radix_sort_pairs(x.temp, bytes, static_cast<const uint32_t*>(x.tkey), x.stkey,
                                                 static_cast<const uint64_t*>(x.tword), x.stword,
                                                 static_cast<size_t>(m.nnz), 0,
                                                 key_bits(static_cast<uint64_t>(16 * nwin)), s))
      return check_hip(e, "transpose sort");
    hipLaunchKernelGGL(transpose_starts, dim3(static_cast<unsigned>(ceil_div(m.nnz + 1, 256))), dim3(256), 0, s,
                       x.stkey, m.nnz, 16 * nwin, x.record, x.rp);
    return run_split<uint32_t, WordColumns, false>(x.rp, WordColumns{x.stword}, 16 * nwin, 16 * nwin, m.nnz,
                                                   295.0 / 505.0, 16, x.split, &x.record->err, &x.record->t_err,
                                                   nullptr, &x.record->t_kept, &x.record->t_vnnz, s);
  });
}

spmm_status fill_task(const Matrix& m, bool layout, int64_t naic, const TaskArrays& x, const spmm_taskmap_out* o,
                      hipStream_t s) {
  const int64_t nwin = ceil_div(m.rows, 16);
  const BitmapShape b(m.cols, m.nnz, nwin);
  return by_index(m.index_type, [&](auto i) {
    using I = decltype(i);
    return by_value(m.value_type, [&](auto u) -> spmm_status {
      using U = decltype(u);
      const uint32_t tile_blocks = tile_capacity<U>(b);
      const size_t lds = b.lds() + (tile_blocks ? ValueTile<U>::kLds : 0);
      const int block_threads = std::max(b.threads(lds), 512);  // block windows are the denser ones
      const U* val = static_cast<const U*>(m.value);
      // The transposed entries' keys, in the order of the nonzeros, are the
      // columns' packed ids: read in place of a gather from inv.
      const uint32_t* packed = layout ? x.tkey : nullptr;
      const TaskOut out{o->crow_window_ptr, o->unique_col_ids, o->value, o->vrow_window_ptr, o->vcol_indices, o->vvalue,
                        o->renumbered_unique_col_ids, o->renumbered_vcol_indices, o->permutation, o->inv_permutation};
      const I* rowptr = static_cast<const I*>(m.rowptr);
      const I* col = static_cast<const I*>(m.col);
      if (naic > 0)
        hipLaunchKernelGGL((write_block_rows<I, U>), dim3(static_cast<unsigned>(naic)), dim3(block_threads), lds, s,
                           rowptr, col, val, m.rows, m.cols, m.nnz, nwin, b.words, b.groups, b.gshift, tile_blocks,
                           x.swin, x.nb, x.pnb, x.midx, x.mrow, x.record, packed, out);
      if (nwin > naic)
        hipLaunchKernelGGL((write_vector_rows<I, U>), dim3(static_cast<unsigned>(nwin - naic)), dim3(256), 0, s, rowptr,
                           col, val, m.rows, m.nnz, nwin, naic, x.swin, x.pnnz, x.record, packed, out);
      if (spmm_status st = check_launch("task outputs")) return st;
      if (!layout) return SPMM_OK;
      return launch_split_fill<uint32_t, WordColumns, WordValues<U>, I, U>(
          x.rp, WordColumns{x.stword}, WordValues<U>{x.stword, val}, 16 * nwin, 16 * nwin, m.nnz, 16, x.split,
          o->transpose_crow_window_ptr, o->transpose_unique_col_ids, static_cast<U*>(o->transpose_value),
          o->transpose_vrow_window_ptr, o->transpose_vcol_indices, static_cast<U*>(o->transpose_vvalue), s);
    });
  });
}

}  // namespace win
}  // namespace spmm
