"""Batched Poisson solves at the edges of the two tile sizes.

Large tiles need 512 of them and sums of 160: one batch of each kind right at
the line, with remainders of every tile, and a batch of the smallest problems.
Also a right-hand side of zeros beside others, and a tolerance no cycle reaches.
"""
import numpy as np
import pytest

from picmcc import PoissonBatch, poisson_cases
from poisson_oracle import rel_residual

pytestmark = pytest.mark.gpu

# large tiles of the batches: 575 and 529, then 485; 525 with sides of 159; 8
BATCHES = {"large": [(160, 160)] * 17 + [(129, 192)] * 3 + [(161, 175), (177, 97)],
           "large1": [(720, 727)], "few": [(160, 160)] * 17 + [(129, 192)] * 2,
           "short": [(159, 159)] * 21, "tiny": [(1, 1), (1, 5), (17, 1), (2, 2), (15, 16), (16, 17), (33, 31)]}


@pytest.mark.parametrize("name", BATCHES)
def test_residuals(name):
    sizes = BATCHES[name]
    n = len(sizes)
    bcs = [poisson_cases.BC_PATTERNS[k % 4] for k in range(n)]
    rng = np.random.default_rng(n)
    rhs = [rng.standard_normal(a * b) for a, b in sizes]
    if n > 1:
        rhs[1][:] = 0.0
    pb = PoissonBatch(sizes, bcs)
    try:
        for _ in range(2):
            pb.set_rhs(np.concatenate(rhs))
            pb.solve(tol=1e-10, max_cycles=3)
            x, rel, bad = pb.result()
            assert bad == 0 and np.all(rel <= 1e-10)
            for k, (a, b) in enumerate(sizes):
                xk = x[pb.offsets[k]:pb.offsets[k + 1]]
                if n > 1 and k == 1:
                    assert not np.any(xk)
                else:
                    assert rel_residual(a, b, bcs[k], rhs[k], xk) <= 1e-10
        # out of cycles: all but the zero problem, whose start is its solution
        # (1 x 1 and 1 x 5 problems may be solved without any rounding)
        pb.solve(tol=1e-30, max_cycles=2)
        y, rel, bad = pb.result()
        exact = int(np.sum(rel == 0.0))
        assert bad == n - exact and exact <= (4 if name == "tiny" else 1)
        # the second cycle only takes rounding off the first one's solution
        assert np.linalg.norm(y - x) <= 1e-9 * np.linalg.norm(x)
    finally:
        pb.close()
