"""Whole argon steps where the launch shapes change.

The count pass gives a wave one, two or four cells, by the number of cells
(8192 and 16384), in a batch by all its cases' together.  A step must equal
the stages one by one bit for bit on both sides of each line, and a batch of
small and large cases the cases stepped alone.
"""
import numpy as np
import pytest
import scipy.sparse as sp

from picmcc import Batch, Case, FP32_REFINED, FP64_PLAIN, HostSetup, PicError, decks

pytestmark = pytest.mark.gpu
SIZES = [(90, 91), (64, 128), (103, 159), (128, 128), (131, 129)]


def deck(ncx, ncy, dx=2e-4, ppc=6):
    return decks.ccp_deck(ncx=ncx, ncy=ncy, dx=dx, ppc=ppc, volts=200.0)


def equal(a, b):
    for s in range(2):
        pa, pb = a.particles(s), b.particles(s)
        for k in ("cell_start", "id", "x", "y", "vx", "vy", "vz"):
            assert np.array_equal(pa[k], pb[k]), f"species {s} field {k}"
    for nm in ("mccr", "next_id", "CondCharge", "den", "phi", "Ex", "Ey", "sum_den", "sum_phi"):
        assert np.array_equal(a.array(nm), b.array(nm)), nm


@pytest.mark.parametrize("prec", [FP32_REFINED, FP64_PLAIN], ids=["f32", "f64"])
@pytest.mark.parametrize("ncx,ncy", SIZES)
def test_step_equals_stages(ncx, ncy, prec):
    a = Case(deck(ncx, ncy), prec, field_solver=2)
    b = Case(deck(ncx, ncy), prec, field_solver=2)
    try:
        a.step(4)
        b.run_staged(4)
        a.sync()
        b.sync()
        equal(a, b)
        assert a.array("mccr").sum() > 0
    finally:
        a.close()
        b.close()


@pytest.mark.parametrize("sizes", [[(24, 17), (92, 96)], [(40, 40), (92, 96), (64, 128)]],
                         ids=["over8192", "over16384"])
def test_batch_of_mixed_sizes_equals_cases_alone(sizes):
    alone = [Case(deck(*s), FP32_REFINED) for s in sizes]
    cs = [Case(deck(*s), FP32_REFINED) for s in sizes]
    bt = Batch(cs)
    try:
        bt.step(5)
        bt.sync()
        for a, c in zip(alone, cs):
            a.step(5)
            a.sync()
            equal(a, c)
    finally:
        bt.close()
        for c in alone + cs:
            c.close()


# interior rows of these add up to one FP32 ulp instead of 0
@pytest.mark.parametrize("ncx,ncy", [(75, 181), (32, 24)])
def test_separable_solve_takes_one_cycle(ncx, ncy):
    """An operator off the 5-point model by one ulp on its diagonal is still
    solved by one cycle; the true residual meets the tolerance."""
    d = deck(ncx, ncy)
    h = HostSetup(d, FP32_REFINED, load=False)
    A = sp.csr_matrix((h.array("Aval").astype(np.float64), h.array("Aj"), h.array("Ai")))
    h.close()
    c = Case(d, FP32_REFINED)
    try:
        assert c.field_solver_kind() == 1
        n = c.info().A_size
        c.set_array("b", np.random.default_rng(n).standard_normal(n))
        c.field_solve()
        c.sync()
        b = c.array("b").astype(np.float64)
        it, outer, rel = c.last_field_solve()
        assert (it, outer) == (1, 1) and rel <= 1e-10
        assert np.linalg.norm(b - A @ c.array("xsol")) <= 1.05e-10 * np.linalg.norm(b)
    finally:
        c.close()


def test_batch_keeps_its_refusal_of_mixed_solves():
    """Operators on and off the model by the diagonal's rounding do not share a batch."""
    cs = [Case(deck(75, 181), FP32_REFINED), Case(deck(64, 64), FP32_REFINED)]
    try:
        with pytest.raises(PicError):
            Batch(cs)
    finally:
        for c in cs:
            c.close()
