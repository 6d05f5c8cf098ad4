"""The register-staged grouped GEMM: every kernel the size rule chooses, at the
edges of its tiles -- widths and K of 1 and 2, odd leading dimensions, ragged
last tiles, K parts with an uneven or empty share -- against float64 matmul, and
the selected inversion (several products of different operand orders in one
accumulator, triangular operands, mirrored output) against the oracle.
Bars: FP64 accumulation of K terms of O(1), |error| <= 2 K eps max|A| max|B|
(5 for the largest of 1e6 normal draws) and the 1e-9 of the solver's tests."""
import ctypes as C

import numpy as np
import pytest
import torch

from oracle import bta as ob
from pyinla_amd import _lib
from pyinla_amd.solver import SerinvSolver
from pyinla_amd.workloads import known_factor_bta

pytestmark = pytest.mark.gpu


def _ptr(t):
    return C.c_void_p(t.data_ptr())


# (m, n, k): 32 x 32 tiles over four waves; the same over one (45^2 tiles);
# 64 x 64 tiles, K in two parts (22^2); 64 x 64 tiles (32 x 32 and 31 x 32)
SHAPES = [(1, 1, 1), (1, 40, 2), (2, 3, 9), (31, 33, 7), (32, 32, 8), (33, 65, 31), (417, 417, 417), (6, 2001, 333),
          (2001, 6, 64), (1431, 1409, 37), (1440, 1440, 40), (1407, 1345, 129), (2001, 2045, 65), (1984, 2048, 17)]


@pytest.mark.parametrize("m,n,k", SHAPES)
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("alpha,beta,pad", [(1.0, 0.0, 0), (-1.0, 1.0, 1), (-1.5, 0.5, 3)])
def test_against_matmul(cuda, m, n, k, ta, tb, alpha, beta, pad):
    lib = _lib.load()
    g = torch.Generator(device=cuda)
    g.manual_seed(m * 7 + n * 3 + k + 11 * ta + 5 * tb)
    f64 = dict(dtype=torch.float64, device=cuda)
    # operands end with their allocation's last element
    A = torch.randn(((k, m) if ta else (m, k)), generator=g, **f64)
    B = torch.randn(((n, k) if tb else (k, n)), generator=g, **f64)
    Cm = torch.randn((m, n + pad), generator=g, **f64)
    ref = beta * Cm[:, :n] + alpha * ((A.T.contiguous() if ta else A) @ (B.T.contiguous() if tb else B))
    out = Cm.clone()
    st = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    _lib.check(lib.bta_gemm(_ptr(A), A.shape[1], ta, _ptr(B), B.shape[1], tb, _ptr(out), n + pad, m, n, k, alpha, beta,
                            0, st), "bta_gemm")
    torch.cuda.synchronize()
    assert (out[:, :n] - ref).abs().max().item() <= 2 * (k + 2) * 2.3e-16 * 25 * 1.5
    assert torch.equal(out[:, n:], Cm[:, n:])


# a = 1 (products of K = 1), b = 1, odd b on both sides of a tile edge; b = 801
# has 32 x 32 tiles in every launch, b = 1391 64 x 64 ones
@pytest.mark.parametrize("n,b,a", [(2, 1, 1), (3, 1, 2), (3, 31, 1), (3, 33, 1), (4, 65, 2), (3, 417, 1), (2, 801, 3),
                                   (2, 1391, 2)])
def test_selected_inversion(cuda, n, b, a):
    kf = known_factor_bta(n, b, a, seed=n * b + a, norm_b=92 if b > 92 else None)
    s = SerinvSolver(None, b, n, a, use_graph=False)
    s.load_blocks(kf.Q_D, kf.Q_L, kf.Q_B, kf.Q_T)
    s.factorize("bta")
    s.selected_inversion("bta")
    D, L, B, T = kf.Lf_D.copy(), kf.Lf_L.copy(), kf.Lf_B.copy(), kf.Lf_T.copy()
    ob.pobtasi(D, L, B, T)
    for got, ref in ((s.A_diagonal_blocks, D), (s.A_lower_diagonal_blocks, L), (s.A_arrow_bottom_blocks, B),
                     (s.A_arrow_tip_block, T)):
        assert np.abs(got.cpu().numpy() - ref).max() <= 1e-9 * np.abs(ref).max()
