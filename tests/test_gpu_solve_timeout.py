"""A triangular sweep that gives up waiting says so: SerinvSolver.solve raises, the
error is reported once, and the factor still solves.  The bound of a wait is set to
zero, so that the first look at a vector that is not there yet ends the wait; every
kernel runs to its end."""
import numpy as np
import pytest

from oracle import bta as ob
from pyinla_amd.workloads import known_factor_bta

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

SOLVE_WAIT = 11  # BTA_OPT_SOLVE_WAIT


@pytest.mark.parametrize("b,nrhs", [(130, 1), (1500, 1), (700, 9)])
def test_solve_reports_a_timeout(cuda, b, nrhs):
    from pyinla_amd import _lib
    from pyinla_amd.solver import SerinvSolver
    n, a = 6, 3
    kf = known_factor_bta(n, b, a, seed=b, norm_b=92)
    s = SerinvSolver(None, b, n, a, reserve="solve")
    s.load_blocks(kf.Q_D, kf.Q_L, kf.Q_B, kf.Q_T)
    s.factorize("bta")
    R = np.random.default_rng(b).normal(size=(n * b + a, nrhs))
    ref = R.copy()
    ob.pobtas(kf.Lf_D, kf.Lf_L, kf.Lf_B, kf.Lf_T, ref, "N")
    ob.pobtas(kf.Lf_D, kf.Lf_L, kf.Lf_B, kf.Lf_T, ref, "C")
    for _ in range(2):
        _lib.check(s.lib.bta_ws_set_option(s._ws, SOLVE_WAIT, 0), "set_option")
        host = R.copy()
        with pytest.raises(_lib.BTALibraryError, match="solve failed: in-kernel wait timed out"):
            s.solve(host, "bta")
        assert np.array_equal(host, R)
        assert s.status()[0] == 0  # the factorization itself is fine, the solve's error was reported
        _lib.check(s.lib.bta_ws_set_option(s._ws, SOLVE_WAIT, 20000), "set_option")
        # no new factorization in between
        got = s.solve(torch.from_numpy(R.copy()).to(cuda), "bta").cpu().numpy()
        assert np.abs(got - ref).max() <= 1e-9 * np.abs(ref).max()


def test_status_reports_a_sweep_too(cuda):
    """bta_potrs on its own: bta_ws_status is the place to look, and it reports once."""
    import ctypes as C

    from pyinla_amd import _lib
    from pyinla_amd.solver import SerinvSolver, _ptr, _stream_ptr
    n, b, a = 6, 1500, 0
    kf = known_factor_bta(n, b, a, seed=3, norm_b=92)
    s = SerinvSolver(None, b, n, a, reserve="solve")
    s.load_blocks(kf.Q_D, kf.Q_L)
    s.factorize("bt")
    _lib.check(s.lib.bta_ws_set_option(s._ws, SOLVE_WAIT, 0), "set_option")
    x = torch.ones(n * b, dtype=torch.float64, device=cuda)
    D, L, B, T, _ = s._blocks("bt")
    _lib.check(s.lib.bta_potrs(s._ws, _ptr(D), _ptr(L), _ptr(B), _ptr(T), n, b, a, C.c_void_p(x.data_ptr()), 1, 1, 0,
                               _stream_ptr(s.device)), "bta_potrs")
    with pytest.raises(_lib.BTALibraryError, match="timed out"):
        s.status()
    assert s.status()[0] == 0
    assert s.lib.bta_ws_set_option(s._ws, SOLVE_WAIT, -1) == -1
