"""Helper shares and wave sizes of a batched factorization: problems whose tile
columns differ by up to 16 : 1 (a few helpers beside most of the chip), one
workgroup per CU and two, waves of 20, of 17 + the rest, each equal to its own
single factorization (the same tasks in the same order per tile) within 1e-12
of the largest entry, and the same log-determinant within 1e-12."""
import numpy as np
import pytest
import torch

from pyinla_amd.batch import BatchedFactorization
from pyinla_amd.solver import SerinvSolver
from pyinla_amd.workloads import known_factor_bta_torch

pytestmark = pytest.mark.gpu

BATCHES = [[(3, 1030, 5), (9, 70, 5)], [(2, 900, 0), (4, 130, 2), (3, 200, 0)],
           [(4, 300, 3), (2, 1200, 3), (6, 400, 3)], [(5, 100, 1)] * 20, [(3, 66 + 13 * q, q % 4) for q in range(23)],
           [(2, 640, 2)] * 5]


@pytest.mark.parametrize("shapes", BATCHES, ids=lambda s: "-".join("x".join(map(str, t)) for t in s[:3]) + f"-{len(s)}")
def test_equals_single(cuda, shapes):
    Q = [known_factor_bta_torch(n, b, a, 7 * q + b, cuda, norm_b=92 if b > 92 else None)[1]
         for q, (n, b, a) in enumerate(shapes)]
    sps = ["bta" if a else "bt" for _, _, a in shapes]
    solvers = [SerinvSolver(None, b, n, a, reserve="factor") for n, b, a in shapes]
    batch = BatchedFactorization(solvers, sps)
    for _ in range(2):  # the second pass reuses the exchange buffers
        for s, q in zip(solvers, Q):
            s.load_blocks(*q)
        batch.factorize()
        status = batch.status()
    for s, q, sp, (n, b, a), (info, ld) in zip(solvers, Q, sps, shapes, status):
        one = SerinvSolver(None, b, n, a, reserve="factor")
        one.load_blocks(*q)
        one.factorize(sp)
        info1, ld1 = one.status()
        assert info == info1 == 0 and abs(ld - ld1) <= 1e-12 * abs(ld1)
        for x, y in ((s.A_diagonal_blocks, one.A_diagonal_blocks), (s.A_lower_diagonal_blocks, one.A_lower_diagonal_blocks),
                     (s.A_arrow_bottom_blocks, one.A_arrow_bottom_blocks)):
            if x is not None and x.numel():
                assert (x - y).abs().max().item() <= 1e-12 * y.abs().max().item()
        if a:
            d = torch.tril(s.A_arrow_tip_block) - torch.tril(one.A_arrow_tip_block)
            assert d.abs().max().item() <= 1e-12 * one.A_arrow_tip_block.abs().max().item()
    assert np.isfinite([ld for _, ld in status]).all()
