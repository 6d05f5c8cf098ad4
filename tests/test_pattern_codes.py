"""Host map of a sparse pattern into the BTA blocks (bta_pattern_codes) against
the definition: every entry of a random COO pattern, entries outside the blocks
among them, in both index widths, both triangles and the lower one only."""
import ctypes as C

import numpy as np
import pytest

from pyinla_amd import _lib


def _expected(rows, cols, n, b, a, lower_only):
    idx, codes = [], []
    for e, (r, c) in enumerate(zip(rows.tolist(), cols.tolist())):
        if lower_only and r < c:
            continue
        if r < n * b and c < n * b:
            bi, bj = r // b, c // b
            if bi == bj:
                v = (bi * b + r % b) * b + c % b
            elif bi == bj + 1:
                v = (1 << 60) | ((bj * b + r % b) * b + c % b)
            else:
                continue
        elif n * b <= r < n * b + a and c < n * b:
            v = (2 << 60) | ((c // b * a + r - n * b) * b + c % b)
        elif n * b <= r < n * b + a and n * b <= c < n * b + a:
            v = (3 << 60) | ((r - n * b) * a + c - n * b)
        else:
            continue
        idx.append(e)
        codes.append(v)
    return idx, codes


@pytest.mark.parametrize("n,b,a", [(1, 1, 0), (1, 1, 1), (5, 1, 2), (4, 3, 0), (3, 7, 2), (6, 49, 5), (2, 100, 64)])
@pytest.mark.parametrize("dtype", [np.int32, np.int64])
@pytest.mark.parametrize("lower_only", [0, 1])
def test_against_definition(n, b, a, dtype, lower_only):
    rng = np.random.default_rng(n * 100 + b + a)
    N = n * b + a + 3  # three rows past the matrix
    rows, cols = rng.integers(0, N, 4000).astype(dtype), rng.integers(0, N, 4000).astype(dtype)
    near = rng.integers(-b, b + 1, 4000)
    cols[::2] = np.clip(rows[::2] + near[::2], 0, N - 1)  # entries of and next to the diagonal blocks
    idx, code, count = np.zeros(4000, np.int64), np.zeros(4000, np.uint64), C.c_int64()
    p = lambda x: C.c_void_p(x.ctypes.data)
    lib = _lib.load()
    assert lib.bta_pattern_codes(p(rows), p(cols), rows.itemsize, 4000, n, b, a, lower_only, p(idx), p(code),
                                 C.byref(count)) == 0
    ei, ec = _expected(rows, cols, n, b, a, lower_only)
    assert count.value == len(ei)
    assert idx[:count.value].tolist() == ei and code[:count.value].tolist() == ec


def test_arguments():
    lib, count = _lib.load(), C.c_int64()
    assert lib.bta_pattern_codes(None, None, 4, 0, 1, 1, 0, 0, None, None, C.byref(count)) == 0 and count.value == 0
    assert lib.bta_pattern_codes(None, None, 4, 1, 1, 1, 0, 0, None, None, C.byref(count)) == -1
    assert lib.bta_pattern_codes(None, None, 2, 0, 1, 1, 0, 0, None, None, C.byref(count)) == -1
    # the block of a row by a product with 1 / b, on both sides of every block edge
    for b in (3, 7, 49, 1999):
        n = 2_000_000_000 // b
        edge = np.unique(np.linspace(1, n - 1, 500).astype(np.int64)) * b
        rows = np.concatenate([edge - 1, edge])
        idx, code = np.zeros(len(rows), np.int64), np.zeros(len(rows), np.uint64)
        assert lib.bta_pattern_codes(C.c_void_p(rows.ctypes.data), C.c_void_p(rows.ctypes.data), 8, len(rows), n, b, 0,
                                     0, C.c_void_p(idx.ctypes.data), C.c_void_p(code.ctypes.data), C.byref(count)) == 0
        assert count.value == len(rows)
        assert np.array_equal(code, (rows // b * (b * b) + rows % b * (b + 1)).astype(np.uint64))
