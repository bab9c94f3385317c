"""Which conversions go window by window (ascend-spmm_amd/csrc/window_rule.h):
the rule is host arithmetic on the sizes, compiled here by itself."""

import ctypes
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ascend-spmm_amd", "csrc")
BLOCKS, SPLIT, TASK, TASK_LAYOUT = range(4)


@pytest.fixture(scope="module")
def eligible(tmp_path_factory):
    out = tmp_path_factory.mktemp("rule")
    source, library = out / "rule.cpp", out / "rule.so"
    source.write_text('#include "window_rule.h"\n'
                      'extern "C" int rule(int op, long long rows, long long cols, long long nnz, long long w) {\n'
                      "  return spmm::win::eligible(static_cast<spmm::win::Op>(op), rows, cols, nnz, w);\n}\n")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I", CSRC, str(source), "-o", str(library)],
                   check=True)
    rule = ctypes.CDLL(str(library)).rule
    rule.argtypes = [ctypes.c_int] + [ctypes.c_longlong] * 4
    return lambda *a: bool(rule(*a))


@pytest.mark.parametrize("op", [BLOCKS, SPLIT, TASK])
@pytest.mark.parametrize("window", [1, 3, 16])
def test_windows_fit_a_grid_of_1024_threads_each(eligible, op, window):
    """A grid of one work-group per window stays below 2^32 threads."""
    most = 2**32 // 1024 - 1
    nnz = 2**31 - 1
    assert eligible(op, window * most, 64, nnz, window)
    assert not eligible(op, window * most + 1, 64, nnz, window)
    assert not eligible(op, 2**31 - 100, 64, nnz, window)


def test_sizes_the_kernels_do_not_hold(eligible):
    assert eligible(BLOCKS, 4096, 2**20, 10**6, 16) and not eligible(BLOCKS, 4096, 2**20 + 1, 10**6, 16)
    assert not eligible(BLOCKS, 4096, 4096, 2**31, 16)
    for rows, cols, nnz, window in ((0, 5, 5, 16), (5, 0, 5, 16), (5, 5, 0, 16), (5, 5, 5, 0), (5, 5, 5, 17)):
        assert not eligible(SPLIT, rows, cols, nnz, window)
    # the transpose's columns are the packed rows, whole windows of them
    assert eligible(TASK_LAYOUT, 2**20, 2**20, 2**28, 16) and not eligible(TASK_LAYOUT, 2**20 + 1, 2**20, 2**28, 16)


K20 = 2**20
# (op, rows, columns, nonzeros, window), the sorting and the window pipeline's
# times on them (us): more columns, rows, nonzeros or smaller windows decide.
MEASURED = [
    (BLOCKS, K20, K20, 1 << 20, 16, 381, 3065), (BLOCKS, K20, K20, 1 << 20, 1, 365, 48000),
    (BLOCKS, K20, K20, 1 << 24, 16, 2289, 3225), (BLOCKS, 1 << 18, 1 << 18, 1 << 20, 16, 370, 206),
    (BLOCKS, K20, 1 << 12, 1 << 22, 16, 647, 441), (BLOCKS, K20, 1 << 12, 1 << 18, 16, 264, 417),
    (BLOCKS, 1 << 16, 1 << 12, 1 << 19, 1, 288, 412), (BLOCKS, 1 << 12, K20, 1 << 18, 16, 281, 43),
    (SPLIT, K20, K20, 1 << 20, 1, 672, 41668), (SPLIT, K20, 1 << 19, 1 << 22, 16, 1280, 1366),
    (SPLIT, 1 << 15, K20, 1 << 15, 16, 350, 120), (SPLIT, K20, 1 << 12, 1 << 20, 4, 676, 1390),
    (TASK, K20, K20, 1 << 22, 16, 1280, 2011), (TASK, 1 << 19, 1 << 19, 1 << 23, 16, 1816, 588),
    (TASK, K20, 1 << 18, 1 << 18, 16, 685, 716), (TASK, 1 << 18, 1 << 18, 1 << 20, 16, 745, 269),
    (TASK_LAYOUT, K20, K20, 1 << 22, 16, 2984, 5030), (TASK_LAYOUT, 1 << 18, 1 << 18, 1 << 22, 16, 2776, 724),
]


@pytest.mark.parametrize("op,rows,cols,nnz,window,sorting,windows", MEASURED)
def test_the_faster_pipeline_is_tried(eligible, op, rows, cols, nnz, window, sorting, windows):
    assert eligible(op, rows, cols, nnz, window) == (windows < sorting)


@pytest.mark.parametrize("op", [BLOCKS, SPLIT, TASK, TASK_LAYOUT])
def test_more_windows_or_columns_never_turn_a_matrix_eligible(eligible, op):
    """One change from eligible to not along rows (at fixed nonzeros) and columns."""
    def changes(flags):
        assert flags[0] and not flags[-1]
        return sum(a != b for a, b in zip(flags, flags[1:]))

    rows = [1 << k for k in range(4, 21)]
    assert changes([eligible(op, r, 1 << 12, 1 << 16, 1) for r in rows]) == 1
    assert changes([eligible(op, 1 << 18, 1 << k, 1 << 18, 16) for k in range(8, 21)]) == 1
