"""The separable solve for permittivities e(x) f(y), against the PCG's rule.

Dielectric side walls and layers over a whole electrode take it; a block that
ends inside the gap does not.  Each solution's true residual, formed on the
host from the set-up's matrix, must meet the requested tolerance, and whole
captured steps must equal the steps launched one by one.
"""
import numpy as np
import pytest
import scipy.sparse as sp

from picmcc import Case, FP32_REFINED, FP64_PLAIN, HostSetup, decks

pytestmark = pytest.mark.gpu
TOL = 1e-10


def deck(ncx, ncy, walls, eps, ppc=2):
    d = decks.ccp_deck(ncx=ncx, ncy=ncy, ppc=ppc, volts=100.0)
    g = d["Geometry"]
    g["ConductorSpec"][0].update({"Y0": ncy - 2, "Y1": ncy})
    g["ConductorSpec"][1].update({"Y0": 0, "Y1": 1})
    side = {"X0": 3 * ncx // 4, "X1": ncx, "Y0": 1, "Y1": ncy - 2}
    spans = {"side": [side], "sides": [{**side, "X0": 0, "X1": 1}, side],
             "layer": [{"X0": 0, "X1": ncx, "Y0": 1, "Y1": 1 + max(1, ncy // 8)}],
             "block": [{**side, "Y1": ncy // 2}]}[walls]
    g["DielectricSpec"] = [{"M_ID": 3 + k, "Epsilon": eps, **s} for k, s in enumerate(spans)]
    return d


# the smallest, odd sizes, one above the tiles of 64 and 128, a long one
DECKS = [(4, 6, "side", 4.0, 2), (33, 21, "sides", 4.0, 2), (33, 21, "layer", 9.3, 2), (65, 68, "side", 80.0, 2),
         (128, 131, "layer", 3.9, 2), (300, 220, "sides", 2.1, 2), (1000, 12, "side", 4.0, 2),
         (33, 21, "block", 4.0, 0), (1030, 8, "side", 4.0, 0)]
IDS = [f"{a}x{b}-{w}-{e:g}" for a, b, w, e, _ in DECKS]


@pytest.mark.parametrize("prec", [FP32_REFINED, FP64_PLAIN], ids=["f32", "f64"])
@pytest.mark.parametrize("ncx,ncy,walls,eps,kind", DECKS, ids=IDS)
def test_residual_meets_the_tolerance(ncx, ncy, walls, eps, kind, prec):
    d = deck(ncx, ncy, walls, eps)
    h = HostSetup(d, prec, load=False)
    A = sp.csr_matrix((h.array("Aval").astype(np.float64), h.array("Aj"), h.array("Ai")))
    h.close()
    c = Case(d, prec, field_solver=2)
    try:
        assert c.field_solver_kind() == kind
        n = c.info().A_size
        rng = np.random.default_rng(n)
        for k in range(3):   # from zero, from the last solution, and a zero right-hand side
            c.set_array("b", rng.standard_normal(n) if k < 2 else np.zeros(n))
            c.field_solve()
            c.sync()
            b = c.array("b").astype(np.float64)
            x = c.array("xsol")
            if k == 2:
                # rounding of the last solution: none is left over
                assert np.linalg.norm(A @ x) <= 1e-9 * np.linalg.norm(last)
                continue
            it, _, rel = c.last_field_solve()
            assert it > 0 and rel <= TOL
            # the path's own norm of its FP64 residual, re-formed with other rounding
            assert np.linalg.norm(b - A @ x) <= 1.05 * TOL * np.linalg.norm(b)
            last = b
    finally:
        c.close()


@pytest.mark.parametrize("prec", [FP32_REFINED, FP64_PLAIN], ids=["f32", "f64"])
@pytest.mark.parametrize("walls", ["side", "layer"])
def test_captured_steps_equal_plain_ones(walls, prec, monkeypatch):
    d = deck(33, 29, walls, 4.0, ppc=20)
    g = Case(d, prec, field_solver=2)
    monkeypatch.setenv("PIC_NO_GRAPH", "1")
    e = Case(d, prec, field_solver=2)
    try:
        for _ in range(3):
            g.step(5)
            g.sync()
            e.step(5)
            e.sync()
            assert np.array_equal(g.array("phi"), e.array("phi"))
            for sp_ in range(2):
                assert g.info().np[sp_] == e.info().np[sp_]
    finally:
        g.close()
        e.close()
