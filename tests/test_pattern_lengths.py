"""The native pattern map reads as many columns as there are rows: index arrays of
different lengths are refused before they reach it."""
from types import SimpleNamespace

import numpy as np
import pytest

from pyinla_amd import _lib
from pyinla_amd.solver import SerinvSolver


def _codes(rows, cols):
    stub = SimpleNamespace(n_diag_blocks=3, diagonal_blocksize=2, arrowhead_blocksize=0, lib=_lib.load(),
                           _index_pair=SerinvSolver._index_pair)
    return SerinvSolver._pattern_codes(stub, rows, cols, "bt", lower_only=False)


@pytest.mark.parametrize("dtype", [np.int32, np.int64])
@pytest.mark.parametrize("nr,nc", [(6, 5), (5, 6), (6, 0), (0, 1)])
def test_lengths_that_differ_are_refused(nr, nc, dtype):
    with pytest.raises(ValueError, match="do not match"):
        _codes(np.arange(nr, dtype=dtype), np.arange(nc, dtype=dtype))


def test_equal_lengths_of_any_integer_type():
    idx, codes = _codes(np.arange(6, dtype=np.int32), list(range(6)))
    assert idx.tolist() == [0, 1, 2, 3, 4, 5] and codes.tolist() == [0, 3, 4, 7, 8, 11]
    assert len(_codes([], [])[0]) == 0
