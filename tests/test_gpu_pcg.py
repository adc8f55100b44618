"""The register-resident PCG at the edges of its launch shapes.

One block holds 512 threads of 1, 2, 4 or 8 rows; above 4096 unknowns blocks of
1024 or 2048 rows exchange their ghosts.  Each operator below sits at such an
edge (unknowns in the id).  The solution's true residual, formed on the host
from the set-up's matrix, must meet the requested tolerance.
"""
import numpy as np
import pytest
import scipy.sparse as sp

from picmcc import Case, FP32_REFINED, FP64_PLAIN, HostSetup, decks

pytestmark = pytest.mark.gpu

TOL = 1e-10


def deck(ncx, ncy, dielectric):
    d = decks.ccp_deck(ncx=ncx, ncy=ncy, ppc=2, volts=100.0)
    if dielectric:
        g = d["Geometry"]
        g["ConductorSpec"][0].update({"Y0": ncy - 2, "Y1": ncy})
        g["ConductorSpec"][1].update({"Y0": 0, "Y1": 1})
        g["DielectricSpec"] = [{"M_ID": 3, "X0": 3 * ncx // 4, "X1": ncx, "Y0": 1, "Y1": ncy - 2, "Epsilon": 4.0}]
    return d


# unknowns (ncx + 1)(ncy - 1) without the dielectric
SHAPES = [(2, 2, False, (1, 512)), (63, 9, False, (1, 512)), (26, 20, False, (1, 512)), (63, 33, False, (1, 512)),
          (40, 51, False, (1, 512)), (63, 65, False, (1, 512)), (16, 242, False, (5, 512)), (90, 90, True, None),
          (300, 220, False, (33, 512))]


@pytest.mark.parametrize("prec", [FP32_REFINED, FP64_PLAIN], ids=["f32", "f64"])
@pytest.mark.parametrize("ncx,ncy,dielectric,shape", SHAPES,
                         ids=[f"{(a + 1) * (b - 1)}{'d' if d else ''}" for a, b, d, _ in SHAPES])
def test_residual_meets_the_tolerance(ncx, ncy, dielectric, shape, prec):
    d = deck(ncx, ncy, dielectric)
    h = HostSetup(d, prec, load=False)
    A = sp.csr_matrix((h.array("Aval").astype(np.float64), h.array("Aj"), h.array("Ai")))
    h.close()
    c = Case(d, prec, field_solver=1)
    try:
        if shape:
            assert c.field_solver_shape() == shape
        n = c.info().A_size
        rng = np.random.default_rng(n)
        for k in range(3):   # from zero, from the last solution, and a zero right-hand side
            b = rng.standard_normal(n) if k < 2 else np.zeros(n)
            c.set_array("b", b)
            c.field_solve()
            c.sync()
            b = c.array("b").astype(np.float64)
            x = c.array("xsol")
            if k == 2:
                assert not np.any(x)
                continue
            it, _, rel = c.last_field_solve()
            assert it > 0 and rel <= TOL
            # the recurrence's residual and the true one part by rounding:
            # at most a few eps |A| |x| over the iterations
            drift = 64 * np.finfo(np.float64).eps * np.linalg.norm(abs(A) @ abs(x))
            assert np.linalg.norm(b - A @ x) <= TOL * np.linalg.norm(b) + drift
    finally:
        c.close()
