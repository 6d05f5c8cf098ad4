"""The panel's helpers where their tile paths change: ragged last rows and
columns of every quadrant, arrows of every width up to a full tile, hand-off
tiles updated once, twice and more, and runs of updates shorter and longer than
a group."""
import numpy as np
import pytest

from oracle import bta as ob
from pyinla_amd.workloads import known_factor_bta

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("b,a,helpers", [
    (129, 1, 0), (192, 0, 0), (193, 16, 0), (223, 31, 0), (225, 33, 1), (240, 63, 3), (256, 64, 9),
    (321, 2, 0), (449, 47, 17), (831, 17, 0), (961, 64, 40), (1090, 5, 0)])
def test_factor_helper_edges(cuda, b, a, helpers):
    """Factor blocks rel 1e-9 and log-determinant rel 1e-10 of the known factor."""
    from pyinla_amd.solver import SerinvSolver
    n = 3
    kf = known_factor_bta(n, b, a, seed=b + a, norm_b=92)
    s = SerinvSolver(None, b, n, a, reserve="factor")
    s.set_panel("flow", helpers)
    for _ in range(2):
        s.load_blocks(kf.Q_D, kf.Q_L, kf.Q_B if a else None, kf.Q_T if a else None)
        s.factorize("bta" if a else "bt")
        info, ld = s.status()
        assert info == 0
        ref = ob.logdet(kf.Lf_D, kf.Lf_T) if a else 2 * np.log(np.diagonal(kf.Lf_D, axis1=1, axis2=2)).sum()
        assert abs(ld - ref) <= 1e-10 * abs(ref)
        pairs = [(s.A_diagonal_blocks, kf.Lf_D), (s.A_lower_diagonal_blocks, kf.Lf_L)]
        if a:
            pairs += [(s.A_arrow_bottom_blocks, kf.Lf_B), (s.A_arrow_tip_block, kf.Lf_T)]
        for got, want in pairs:
            got = got.cpu().numpy()
            assert np.abs(got - want).max() <= 1e-9 * np.abs(want).max()
