"""The panel's chain and the 64x64 tile factorization where their forms change:
last tiles of every width around the 16-wide blocks, odd leading dimensions,
chains of one, two and more columns, and the first failing pivot at every
position of a tile."""
import numpy as np
import pytest

from oracle import bta as ob
from pyinla_amd.workloads import known_factor_bta

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("b", [16, 33, 64, 65, 79, 80, 81, 95, 96, 97, 112, 127, 128, 129, 192, 193, 255, 320])
@pytest.mark.parametrize("panel", ["flow", "columns"])
def test_factor_tile_edges(cuda, b, panel):
    """Factor blocks rel 1e-9 and log-determinant rel 1e-10 of the known factor."""
    from pyinla_amd.solver import SerinvSolver
    n, a = 3, 5
    kf = known_factor_bta(n, b, a, seed=b, norm_b=92 if b > 92 else None)
    s = SerinvSolver(None, b, n, a, reserve="factor")
    s.set_panel(panel)
    # only the lower triangle of a diagonal block is read
    D = np.tril(kf.Q_D) + np.triu(np.full((n, b, b), 7.0), 1)
    s.load_blocks(D, kf.Q_L, kf.Q_B, kf.Q_T)
    s.factorize("bta")
    info, ld = s.status()
    assert info == 0
    ref = ob.logdet(kf.Lf_D, kf.Lf_T)
    assert abs(ld - ref) <= 1e-10 * abs(ref)
    for got, want in ((s.A_diagonal_blocks, kf.Lf_D), (s.A_lower_diagonal_blocks, kf.Lf_L),
                      (s.A_arrow_bottom_blocks, kf.Lf_B), (s.A_arrow_tip_block, kf.Lf_T)):
        got = got.cpu().numpy()
        assert np.abs(got - want).max() <= 1e-9 * np.abs(want).max()
    assert not np.triu(s.A_diagonal_blocks.cpu().numpy(), 1).any()


@pytest.mark.parametrize("b,panel", [(150, "flow"), (150, "columns"), (40, "columns")])
def test_first_failing_pivot(cuda, b, panel):
    """info is the 1-based row of the first pivot that is not positive."""
    from pyinla_amd.solver import SerinvSolver
    n = 2
    s = SerinvSolver(None, b, n, 0, reserve="factor")
    s.set_panel(panel)
    Q = np.random.default_rng(3).normal(size=(b, b)) * 0.01
    base = np.eye(b) * 4.0 + Q + Q.T
    for row in [0, 1, 2, 3, 4, 15, 16, 31, 38] + ([63, 64, 66, 127, 128, 149] if b > 64 else []):
        for blk in (0, 1):
            D = np.stack([base, base])
            D[blk, row, row] = -1.0
            s.load_blocks(D, np.zeros((n - 1, b, b)))
            s.factorize("bt")
            assert s.status()[0] == blk * b + row + 1
    s.load_blocks(np.stack([base, base]), np.zeros((n - 1, b, b)))
    s.factorize("bt")
    info, ld = s.status()
    assert info == 0 and abs(ld - 2 * np.linalg.slogdet(base)[1]) <= 1e-10 * abs(ld)
