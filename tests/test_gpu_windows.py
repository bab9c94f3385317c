"""The window-by-window preprocessing kernels at the sizes where they change
behaviour (bitmap word and prefix-group edges, windows longer than the
registers hold, the LDS tile's edge, the column limit), bit for bit against
the CPU oracle; and the inputs they hand to the sorting pipeline instead."""

import concurrent.futures

import numpy as np
import pytest
import torch

import oracle as O
from test_gpu_preprocess import assert_same

pytestmark = pytest.mark.gpu

# 31 .. 129: words and prefix groups; 131072 / 131073: 2- and 4-word groups;
# 524288 / 524289: 4- and 8-word groups; 2^20: the limit; 2^20 + 1: past it.
COLS = [1, 31, 32, 33, 127, 128, 129, 4097, 131072, 131073, 524288, 524289, 1 << 20, (1 << 20) + 1]


def matrix(cols, rows=37, seed=0):
    """Random short rows, a run of adjacent columns, an empty row, the first
    and last columns, and one row longer than a work-group holds (4096 or
    more nonzeros, where there are so many columns)."""
    rng = np.random.default_rng(cols + seed)
    parts = [np.unique(rng.integers(0, cols, int(rng.integers(0, 40)))) for _ in range(rows)]
    parts[2] = np.arange(max(0, cols // 2 - 70), min(cols, cols // 2 + 70))
    parts[3] = np.zeros(0, np.int64)
    parts[4] = np.unique(np.array([0, cols - 1]))
    parts[20] = np.unique(rng.integers(0, cols, min(6 * cols, 9000)))
    crow = np.zeros(rows + 1, np.int64)
    crow[1:] = np.cumsum([p.size for p in parts])
    return crow, np.concatenate(parts).astype(np.int64)


def as_types(crow, col, index, value, seed=3):
    val = np.random.default_rng(seed).uniform(-1, 1, col.size).astype(value)
    return crow.astype(index), col.astype(index), val


def gpu(*arrays):
    return [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in arrays]


@pytest.mark.parametrize("cols", COLS)
@pytest.mark.parametrize("window", [1, 7, 16])
def test_blocks_and_tiles(spmm_npu, cols, window):
    crow, col = matrix(cols)
    for index, value in ((np.int32, np.float16), (np.int64, np.float32), (np.int32, np.float64)):
        args = as_types(crow, col, index, value)
        assert_same(spmm_npu.csr_to_bcsr(*gpu(*args), 37, cols, window), O.csr_to_bcsr(*args, 37, cols, window))
        assert_same(spmm_npu.csr_to_ascend_cube(*gpu(*args), 37, cols, window),
                    O.csr_to_ascend_cube(*args, 37, cols, window))


@pytest.mark.parametrize("extra", [-1, 0, 1])
@pytest.mark.parametrize("blocks,value", [(640, np.float16), (320, np.float32), (160, np.float64)])
def test_tile_edge(spmm_npu, blocks, value, extra):
    """A window of exactly as many blocks as the LDS tile holds, one less, one
    more (20 KB of 16-value blocks)."""
    n = blocks + extra
    crow = np.array([0, n, n + 1], np.int64)
    col = np.concatenate([np.arange(n), [n // 2]]).astype(np.int64)
    args = as_types(crow, col, np.int32, value)
    assert_same(spmm_npu.csr_to_bcsr(*gpu(*args), 2, 5000, 16), O.csr_to_bcsr(*args, 2, 5000, 16))


@pytest.mark.parametrize("threads,cols,others", [(256, 3000, 12), (512, 3000, 0), (1024, 1 << 20, 0)])
@pytest.mark.parametrize("extra", [-1, 0, 1])
def test_window_of_register_size(spmm_npu, threads, cols, others, extra):
    """A window of as many nonzeros as a work-group's threads hold in registers
    (8 each), one less, one more.  Work-groups have 256 threads where the
    windows average at most 1024 nonzeros (here among `others` short ones), 512
    where they hold more, and 1024 beside a bitmap that fills the LDS."""
    n = 8 * threads + extra
    rng = np.random.default_rng(n)
    rows = [np.sort(rng.choice(cols, k, replace=False)) for k in (n // 3, n - 2 * (n // 3), n // 3)]
    rows += [np.zeros(0, np.int64)] * 13
    for _ in range(16 * others):
        rows.append(np.sort(rng.choice(cols, 5, replace=False)))
    mean = sum(r.size for r in rows) // (1 + others)
    assert (mean <= 1024) == (others > 0)
    crow = np.concatenate([[0], np.cumsum([r.size for r in rows])]).astype(np.int64)
    args = as_types(crow, np.concatenate(rows).astype(np.int64), np.int32, np.float16)
    assert_same(spmm_npu.csr_to_bcsr(*gpu(*args), len(rows), cols, 16), O.csr_to_bcsr(*args, len(rows), cols, 16))
    assert_same(spmm_npu.block_level_split(*gpu(*args), len(rows), cols, 0.6, 16),
                O.block_level_split(*args, len(rows), cols, 0.6, 16))
    assert_same(spmm_npu.preprocess(*gpu(*args), len(rows), cols), O.preprocess(*args, len(rows), cols))


def test_first_position_past_zero(spmm_npu):
    """A row pointer that starts past the first stored nonzero."""
    crow, col = matrix(500)
    crow, col = crow + 11, np.concatenate([np.arange(11), col])
    args = as_types(crow, col, np.int32, np.float32)
    assert_same(spmm_npu.csr_to_bcsr(*gpu(*args), 37, 500, 16), O.csr_to_bcsr(*args, 37, 500, 16))


def test_repeated_and_invalid_columns_take_the_sorting_pipeline(spmm_npu):
    crow, col = matrix(500)
    args = as_types(crow, col, np.int32, np.float32)
    twice = args[1].copy()
    r = int(np.nonzero(np.diff(crow) > 3)[0][5])
    twice[crow[r] + 1] = twice[crow[r]]  # the row's second nonzero repeats its first column
    assert_same(spmm_npu.csr_to_bcsr(*gpu(args[0], twice, args[2]), 37, 500, 16),
                O.csr_to_bcsr(args[0], twice, args[2], 37, 500, 16))
    down = args[1].copy()
    down[crow[r]], down[crow[r] + 1] = args[1][crow[r] + 1], args[1][crow[r]]
    with pytest.raises(ValueError, match="ascending"):
        spmm_npu.csr_to_bcsr(*gpu(args[0], down, args[2]), 37, 500, 16)
    for bad in (500, -1):
        out = args[1].copy()
        out[crow[r + 1] - 1 if bad > 0 else crow[r]] = bad
        with pytest.raises(RuntimeError, match="out of range"):
            spmm_npu.csr_to_bcsr(*gpu(args[0], out, args[2]), 37, 500, 16)
    back = args[0].copy()
    back[r + 1], back[r] = back[r], back[r + 1]
    with pytest.raises(ValueError, match="row pointer"):
        spmm_npu.csr_to_bcsr(*gpu(back, args[1], args[2]), 37, 500, 16)


@pytest.mark.parametrize("cols", [33, 129, 4097, 131073, 1 << 20, (1 << 20) + 1])
@pytest.mark.parametrize("window", [3, 16])
def test_split(spmm_npu, cols, window):
    """Ratios that move nothing, everything, and part of an occupancy; a window
    of more blocks than the LDS holds."""
    crow, col = matrix(cols, seed=1)
    args = as_types(crow, col, np.int32, np.float32)
    for a in (0.0, 0.02, 295.0 / 505.0, 2.5, 40.0, 1e9, float("inf"), float("nan"), -1.0):
        assert_same(spmm_npu.block_level_split(*gpu(*args), 37, cols, a, window),
                    O.block_level_split(*args, 37, cols, a, window))


def square(n, seed=0):
    """Windows of different densities, a long row, occupancies from 1 to 16 and
    a last window of n % 16 rows."""
    rng = np.random.default_rng(n + seed)
    parts = []
    for r in range(n):
        k = int(rng.integers(0, 6)) + (20 if (r // 16) % 5 == 0 else 0)
        near = r // 16 * 16 + rng.integers(0, 48, k)
        far = rng.integers(0, n, 3)
        parts.append(np.unique(np.concatenate([near, far]) % n))
    parts[min(40, n - 1)] = np.unique(rng.integers(0, n, min(n, 6000)))
    crow = np.zeros(n + 1, np.int64)
    crow[1:] = np.cumsum([p.size for p in parts])
    return crow, np.concatenate(parts).astype(np.int64)


@pytest.mark.parametrize("n", [1, 15, 16, 17, 100, 1600, 5003])
@pytest.mark.parametrize("layout", [False, True])
def test_preprocess(spmm_npu, n, layout):
    crow, col = square(n)
    for index, value in ((np.int32, np.float16), (np.int64, np.float32), (np.int32, np.float64)):
        args = as_types(crow, col, index, value)
        assert_same(spmm_npu.preprocess(*gpu(*args), n, n, graph_layout=layout),
                    O.preprocess(*args, n, n, graph_layout=layout))


@pytest.mark.parametrize("rows", [16 * 8192, 16 * 8192 + 5])
def test_preprocess_either_side_of_the_window_sort(spmm_npu, rows):
    """8192 windows are ranked by counting, more by the device sort."""
    rng = np.random.default_rng(rows)
    r = np.sort(rng.integers(0, rows, 40000))
    key = np.unique(r * 3000 + rng.integers(0, 3000, r.size))
    crow = np.zeros(rows + 1, np.int64)
    crow[1:] = np.cumsum(np.bincount(key // 3000, minlength=rows))
    args = as_types(crow, key % 3000, np.int32, np.float16)
    assert_same(spmm_npu.preprocess(*gpu(*args), rows, 3000), O.preprocess(*args, rows, 3000))


@pytest.mark.parametrize("cols", [4097, 300000, 1 << 20])
def test_preprocess_wide_marginal_window(spmm_npu, cols):
    """One window holds nearly all nonzeros, so it is the marginal one: its
    blocks fit the LDS arrays, or not (2^20 columns leave no room)."""
    crow, col = matrix(cols, seed=2)
    args = as_types(crow, col, np.int32, np.float32)
    assert_same(spmm_npu.preprocess(*gpu(*args), 37, cols), O.preprocess(*args, 37, cols))


@pytest.mark.parametrize("n", [32768, 32769])
def test_longest_window(spmm_npu, n):
    """One nonzero more sends the matrix to the sorting pipeline."""
    crow = np.array([0, n - 20000, n, n + 1], np.int64)
    rng = np.random.default_rng(n)
    col = np.concatenate([np.sort(rng.choice(40000, k, replace=False)) for k in (n - 20000, 20000, 1)])
    crow, col = crow - np.array([0, 0, 1, 1]), np.delete(col, n - 1)  # n nonzeros in the one window
    args = as_types(crow, col, np.int32, np.float16)
    assert_same(spmm_npu.csr_to_bcsr(*gpu(*args), 3, 40000, 16), O.csr_to_bcsr(*args, 3, 40000, 16))
    assert_same(spmm_npu.block_level_split(*gpu(*args), 3, 40000, 0.6, 16),
                O.block_level_split(*args, 3, 40000, 0.6, 16))
    assert_same(spmm_npu.preprocess(*gpu(*args), 3, 40000), O.preprocess(*args, 3, 40000))


@pytest.mark.parametrize("first", [0, 11])
def test_handed_over_matrices_keep_their_first_position(spmm_npu, first):
    """The sorting pipeline takes a handed-over matrix's first position and
    nonzeros from the window plan: row pointers that start past zero, and end
    before the last stored nonzero, with a repeated column."""
    crow, col = square(500)
    r = int(np.nonzero(np.diff(crow) > 3)[0][5])
    col = col.copy()
    col[crow[r] + 1] = col[crow[r]]
    crow, col = crow + first, np.concatenate([np.arange(first), col, np.arange(7)])
    args = as_types(crow, col, np.int32, np.float32)
    assert_same(spmm_npu.csr_to_bcsr(*gpu(*args), 500, 500, 16), O.csr_to_bcsr(*args, 500, 500, 16))
    assert_same(spmm_npu.csr_to_ascend_cube(*gpu(*args), 500, 500, 16), O.csr_to_ascend_cube(*args, 500, 500, 16))
    assert_same(spmm_npu.block_level_split(*gpu(*args), 500, 500, 0.6, 16),
                O.block_level_split(*args, 500, 500, 0.6, 16))
    assert_same(spmm_npu.preprocess(*gpu(*args), 500, 500), O.preprocess(*args, 500, 500))
    with pytest.raises(ValueError, match="end at nnz"):
        spmm_npu.preprocess(*gpu(*args), 500, 500, graph_layout=True)


def test_graph_plans_of_several_threads_and_streams(spmm_npu):
    """The counts' error word reaches the host in a word of its own per thread:
    four threads with a stream each, matrices that are handed over and others
    in turn."""
    plans = []
    for n, turned in ((333, False), (334, True), (1601, False), (1602, True)):
        crow, col = square(n)
        if turned:
            col = np.concatenate([col[a:b][::-1] for a, b in zip(crow, crow[1:])])
        args = as_types(crow, col, np.int32, np.float32)
        plans.append((n, gpu(*args), O.preprocess(*args, n, n, graph_layout=True)))
    torch.cuda.synchronize()

    def work(t):
        stream, out = torch.cuda.Stream(), []
        with torch.cuda.stream(stream):
            for i in range(12):
                n, args, _ = plans[(t + i) % 4]
                out.append(spmm_npu.preprocess(*args, n, n, graph_layout=True))
        stream.synchronize()
        return out

    with concurrent.futures.ThreadPoolExecutor(4) as pool:
        for t, out in enumerate(pool.map(work, range(4))):
            for i, got in enumerate(out):
                assert_same(got, plans[(t + i) % 4][2])


@pytest.mark.parametrize("unsorted", [False, True])
def test_row_pointers_that_decrease_are_refused(spmm_npu, unsorted):
    """Also where another window's columns alone hand the matrix over."""
    crow, col = square(700)
    if unsorted:
        col = col[::-1].copy()
    back = crow.copy()
    back[651], back[650] = crow[650], crow[651]
    args = gpu(*as_types(back, col, np.int32, np.float32))
    for call in (lambda: spmm_npu.csr_to_bcsr(*args, 700, 700, 16),
                 lambda: spmm_npu.csr_to_ascend_cube(*args, 700, 700, 16),
                 lambda: spmm_npu.block_level_split(*args, 700, 700, 0.6, 16),
                 lambda: spmm_npu.preprocess(*args, 700, 700),
                 lambda: spmm_npu.preprocess(*args, 700, 700, graph_layout=True)):
        with pytest.raises(ValueError, match="row pointer"):
            call()


def hub_column(n, hub, seed=4):
    """Short rows, the first `hub` of which hold column 7 too."""
    rng = np.random.default_rng(seed)
    key = np.unique(np.concatenate([np.arange(hub) * n + 7, rng.integers(0, n, 2 * n) + np.arange(2 * n) // 2 * n]))
    crow = np.zeros(n + 1, np.int64)
    crow[1:] = np.cumsum(np.bincount(key // n, minlength=n))
    return crow, key % n


@pytest.mark.parametrize("hub", [32000, 40000])
def test_hub_column_of_the_packed_transpose(spmm_npu, hub):
    """No window of A is long, but the transpose's window that holds the hub
    column is: of at most 32768 nonzeros (taken window by window), or more
    (only the transpose's split finds that out, after its other windows have
    begun, and the matrix goes to the sorting pipeline)."""
    n = 40000
    crow, col = hub_column(n, hub)
    assert np.diff(crow[::16]).max() < 64
    args = as_types(crow, col, np.int32, np.float32)
    assert_same(spmm_npu.preprocess(*gpu(*args), n, n, graph_layout=True), O.preprocess(*args, n, n, graph_layout=True))


@pytest.mark.parametrize("layout", [False, True])
def test_unsorted_rows_take_the_sorting_pipeline(spmm_npu, layout):
    crow, col = square(333)
    col = col.copy()
    for r in range(0, 333, 7):
        col[crow[r]:crow[r + 1]] = col[crow[r]:crow[r + 1]][::-1]
    args = as_types(crow, col, np.int32, np.float32)
    assert_same(spmm_npu.preprocess(*gpu(*args), 333, 333, graph_layout=layout),
                O.preprocess(*args, 333, 333, graph_layout=layout))
    assert_same(spmm_npu.block_level_split(*gpu(*args), 333, 333, 0.6, 16),
                O.block_level_split(*args, 333, 333, 0.6, 16))
