"""One tile per block (b <= 64), factorization and selected inversion, each as
one workgroup: block sizes around the 16-wide block columns and the tile's
quadrants, arrow heights around the same, against the oracle; and what a
factorization that fails reports.  Bars as in the other solver tests: 1e-9 of
the largest entry, 1e-10 of the log-determinant."""
import numpy as np
import pytest
import torch

from oracle import bta as ob
from pyinla_amd.solver import SerinvSolver
from pyinla_amd.workloads import known_factor_bta

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 0), (3, 1, 1), (2, 3, 2), (4, 15, 1), (4, 16, 16), (5, 17, 17), (3, 31, 5), (3, 32, 32), (3, 33, 33),
          (2, 40, 64), (3, 48, 3), (3, 49, 0), (2, 63, 7), (4, 64, 31), (2, 64, 64), (7, 64, 0)]


def _solver(kf, n, b, a):
    s = SerinvSolver(None, b, n, a, use_graph=False)
    s.load_blocks(kf.Q_D, kf.Q_L, kf.Q_B if a else None, kf.Q_T if a else None)
    return s


def _close(got, ref):
    assert np.abs(got.cpu().numpy() - ref).max() <= 1e-9 * np.abs(ref).max()


@pytest.mark.parametrize("n,b,a", SHAPES)
def test_factor_and_selected_inverse(cuda, n, b, a):
    kf = known_factor_bta(n, b, a, seed=31 * n + b + a)
    s, sp = _solver(kf, n, b, a), "bta" if a else "bt"
    s.factorize(sp)
    info, ld = s.status()
    assert info == 0
    _close(s.A_diagonal_blocks, kf.Lf_D)
    ld_ref = 2 * np.log(np.diagonal(kf.Lf_D, axis1=1, axis2=2)).sum() + (2 * np.log(np.diag(kf.Lf_T)).sum() if a else 0)
    assert abs(ld - ld_ref) <= 1e-10 * max(abs(ld_ref), 1.0)
    if n > 1:
        _close(s.A_lower_diagonal_blocks, kf.Lf_L)
    if a:
        _close(s.A_arrow_bottom_blocks, kf.Lf_B)
        _close(torch.tril(s.A_arrow_tip_block), kf.Lf_T)
    x = np.random.default_rng(b).normal(size=n * b + a)
    xr = x.copy()
    for tr in "NC":
        ob.pobtas(kf.Lf_D, kf.Lf_L, kf.Lf_B, kf.Lf_T, xr, tr) if a else ob.pobts(kf.Lf_D, kf.Lf_L, xr, tr)
    s.solve(x, sp)
    assert np.abs(x - xr).max() <= 1e-9 * np.abs(xr).max()
    s.selected_inversion(sp)
    D, L, B, T = kf.Lf_D.copy(), kf.Lf_L.copy(), kf.Lf_B.copy() if a else None, kf.Lf_T.copy() if a else None
    ob.pobtasi(D, L, B, T) if a else ob.pobtsi(D, L)
    _close(s.A_diagonal_blocks, D)
    if n > 1:
        _close(s.A_lower_diagonal_blocks, L)
    if a:
        _close(s.A_arrow_bottom_blocks, B)
        _close(s.A_arrow_tip_block, T)


@pytest.mark.parametrize("n,b,a,block,row", [(3, 40, 2, 1, 17), (2, 64, 0, 0, 63), (4, 5, 3, 3, 0)])
def test_failing_pivot(cuda, n, b, a, block, row):
    kf = known_factor_bta(n, b, a, seed=5)
    kf.Q_D[block, row, row] = -1.0
    infos = []
    for mode in ("auto", "columns"):
        s = _solver(kf, n, b, a)
        s.set_panel(mode)
        s.factorize("bta" if a else "bt")
        infos.append(s.status()[0])
    assert infos == [block * b + row + 1] * 2
