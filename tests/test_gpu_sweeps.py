"""Triangular sweeps at the edges of their forms: blocks swept by one workgroup
and by many (b = 64 / 65), the sizes where the loads in flight and the rounds
change (512, 1024, 2048), odd leading dimensions, with and without an arrow, one
right-hand side and groups of 4 and 8 with remainders, a leading dimension larger
than the number of right-hand sides, and non-finite right-hand sides."""
import ctypes as C

import numpy as np
import pytest

from oracle import bta as ob
from pyinla_amd.workloads import known_factor_bta

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

# rel 1e-9 of the solution, the bar of every solve against the oracle
TOL = 1e-9


def _factored(n, b, a, seed):
    from pyinla_amd.solver import SerinvSolver
    kf = known_factor_bta(n, b, a, seed=seed, norm_b=92 if b > 92 else None)
    s = SerinvSolver(None, b, n, a, reserve="solve")
    s.load_blocks(kf.Q_D, kf.Q_L, kf.Q_B if a else None, kf.Q_T if a else None)
    s.factorize("bta" if a else "bt")
    return kf, s


def _oracle(kf, R):
    """Solution by the known factor (no factorization on the host)."""
    a = kf.a
    x = R.copy()
    args = (kf.Lf_D, kf.Lf_L) + ((kf.Lf_B, kf.Lf_T) if a else (None, None))
    ob.pobtas(*args, x, "N")
    ob.pobtas(*args, x, "C")
    return x


@pytest.mark.parametrize("b", [1, 2, 7, 63, 64, 65, 127, 130, 511, 512, 513, 1023, 1024, 1025])
@pytest.mark.parametrize("a,nrhs", [(0, 1), (6, 1), (64, 3), (1, 9)])
def test_solve_forms(cuda, b, a, nrhs):
    n = 3
    kf, s = _factored(n, b, a, seed=b + a)
    R = np.random.default_rng(b).normal(size=(n * b + a, nrhs))
    ref = _oracle(kf, R)
    x = torch.from_numpy(R[:, 0].copy() if nrhs == 1 else R.copy()).to(cuda)
    got = s.solve(x, "bta" if a else "bt").cpu().numpy().reshape(ref.shape)
    assert np.abs(got - ref).max() <= TOL * np.abs(ref).max()


@pytest.mark.parametrize("n,b,nrhs", [(2, 2047, 1), (2, 2048, 5), (2, 2049, 1), (2, 2100, 5), (1, 300, 1), (1, 40, 2)])
def test_solve_large_and_single_blocks(cuda, n, b, nrhs):
    a = 3
    kf, s = _factored(n, b, a, seed=b)
    R = np.random.default_rng(b).normal(size=(n * b + a, nrhs))
    ref = _oracle(kf, R)
    got = s.solve(torch.from_numpy(R.copy()).to(cuda), "bta").cpu().numpy()
    assert np.abs(got - ref).max() <= TOL * np.abs(ref).max()


@pytest.mark.parametrize("b", [40, 200])
def test_solve_leading_dimension(cuda, b):
    """Right-hand sides inside a wider array: the other columns stay untouched."""
    from pyinla_amd import _lib
    from pyinla_amd.solver import _ptr, _stream_ptr
    n, a, nrhs, ld = 4, 2, 3, 7
    kf, s = _factored(n, b, a, seed=5)
    R = np.random.default_rng(1).normal(size=(n * b + a, ld))
    ref = _oracle(kf, R[:, :nrhs].copy())
    x = torch.from_numpy(R.copy()).to(cuda)
    D, L, B, T, _ = s._blocks("bta")
    for trans in (0, 1):
        _lib.check(s.lib.bta_potrs(s._ws, _ptr(D), _ptr(L), _ptr(B), _ptr(T), n, b, a, C.c_void_p(x.data_ptr()),
                                   nrhs, ld, trans, _stream_ptr(s.device)), "bta_potrs")
    got = x.cpu().numpy()
    assert np.abs(got[:, :nrhs] - ref).max() <= TOL * np.abs(ref).max()
    assert np.array_equal(got[:, nrhs:], R[:, nrhs:])


@pytest.mark.parametrize("b", [48, 130])
def test_solve_non_finite(cuda, b):
    """A NaN of any payload, the sweeps' own marker among them, or an infinity
    in the right-hand side comes back as NaN / inf values, and the factor is
    usable afterwards."""
    n, a = 3, 2
    kf, s = _factored(n, b, a, seed=9)
    marker = np.array([0x7FF4C0DEC0DE0001], dtype=np.uint64).view(np.float64)
    for bits in (marker, np.array([np.nan]), np.array([np.inf])):
        for at in (0, n * b - 1, n * b):
            x = torch.zeros(n * b + a, dtype=torch.float64, device=cuda)
            x[at:at + 1] = torch.from_numpy(bits.copy()).to(cuda)
            s.solve(x, "bta")
            assert not torch.isfinite(x).all()
    R = np.random.default_rng(2).normal(size=n * b + a)
    ref = _oracle(kf, R[:, None].copy())[:, 0]
    got = s.solve(torch.from_numpy(R).to(cuda), "bta").cpu().numpy()
    assert np.abs(got - ref).max() <= TOL * np.abs(ref).max()


def test_two_sweeps_share_the_device(cuda):
    """Solves of three factors on three streams at once: each sweep wants more
    workgroups than the others leave room for."""
    n, b, a = 6, 1500, 2
    made = [_factored(n, b, a, seed=20 + q) for q in range(3)]
    streams = [torch.cuda.Stream(device=cuda) for _ in made]
    rng = np.random.default_rng(3)
    Rs = [rng.normal(size=n * b + a) for _ in made]
    xs = [torch.from_numpy(R.copy()).to(cuda) for R in Rs]
    for kf_s in made:
        kf_s[1].prepare_block_inverses("bta")
    torch.cuda.synchronize()
    from pyinla_amd import _lib
    from pyinla_amd.solver import _ptr
    for _ in range(3):
        for (kf, s), st, x, R in zip(made, streams, xs, Rs):
            with torch.cuda.stream(st):
                x.copy_(torch.from_numpy(R))
                D, L, B, T, _a = s._blocks("bta")
                for trans in (0, 1):
                    _lib.check(s.lib.bta_potrs(s._ws, _ptr(D), _ptr(L), _ptr(B), _ptr(T), n, b, a,
                                               C.c_void_p(x.data_ptr()), 1, 1, trans,
                                               C.c_void_p(st.cuda_stream)), "bta_potrs")
        torch.cuda.synchronize()
    for (kf, s), x, R in zip(made, xs, Rs):
        ref = _oracle(kf, R[:, None].copy())[:, 0]
        assert np.abs(x.cpu().numpy() - ref).max() <= TOL * np.abs(ref).max()
        assert s.status()[0] == 0


@pytest.mark.parametrize("n,b,a,nrhs", [(5, 65, 2, 33), (3, 130, 0, 17), (40, 200, 3, 25), (3, 520, 4, 23),
                                        (2, 1030, 5, 16), (200, 70, 1, 32)])
def test_groups_side_by_side(cuda, n, b, a, nrhs):
    """Groups of 8 in one launch: 4 and fewer at a time, the last one ragged,
    and the next launch's right behind."""
    kf, s = _factored(n, b, a, seed=b + nrhs)
    R = np.random.default_rng(b).normal(size=(n * b + a, nrhs))
    ref = _oracle(kf, R)
    for _ in range(2):
        got = s.solve(torch.from_numpy(R.copy()).to(cuda), "bta" if a else "bt").cpu().numpy()
        assert np.abs(got - ref).max() <= TOL * np.abs(ref).max()
