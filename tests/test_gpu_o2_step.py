"""Whole oxygen steps (two passes over the particles) equal the stages one by
one, bit for bit: particles, ids, buckets, reaction counts, detachment
removals, wall counts and fields.

The decks sit where the passes can go wrong: one cell per wave; more particles
per cell than a wave loads at once, and more O- around a cell than the victim
pass keeps keys of; four cells per wave with a ragged last wave; walls that
absorb and charge.
"""
import numpy as np
import pytest

from picmcc import Case, FP32_REFINED, FP64_PLAIN, decks

pytestmark = pytest.mark.gpu

NEUTRALS = {"O2A": 2e21, "O2B": 2e21, "OP": 2e21, "OD": 2e21}
SHAPES = {"small": dict(ncx=9, ncy=14, ppc=40), "dense": dict(ncx=3, ncy=4, ppc=700),
          "wide": dict(ncx=133, ncy=125, ppc=5), "dielectric": dict(ncx=16, ncy=12, ppc=30)}


def deck(gas, shape, ions=True):
    d = decks.oxygen_deck(gas=gas, pres_torr=0.3, volts=200.0, ion_collisions=ions, capacity_factor=4.0,
                          ion_densities={"O-": 8e14}, neutral_densities=NEUTRALS, **SHAPES[shape])
    if shape == "dielectric":
        g = d["Geometry"]
        g["ConductorSpec"][0].update({"Y0": 10, "Y1": 12})
        g["ConductorSpec"][1].update({"Y0": 0, "Y1": 1})
        g["DielectricSpec"] = [{"M_ID": 3, "X0": 12, "X1": 16, "Y0": 1, "Y1": 10, "Epsilon": 4.0}]
    return d


@pytest.mark.parametrize("shape", list(SHAPES))
@pytest.mark.parametrize("gas,ions", [(1, True), (1, False), (2, True)], ids=["O2", "O2-electrons", "ArO2"])
@pytest.mark.parametrize("prec", [FP32_REFINED, FP64_PLAIN], ids=["f32", "f64"])
def test_step_equals_stages(prec, gas, ions, shape):
    # the separable solve where the operator allows it, so that replays of the
    # captured step are covered too
    a = Case(deck(gas, shape, ions), prec, field_solver=2)
    b = Case(deck(gas, shape, ions), prec, field_solver=2)
    try:
        nsp = a.info().nsp
        for step in range(6):
            if shape == "dense":
                # O- as dense as the gas (the targets of detachment), 20 eV electrons
                for c in (a, b):
                    den = c.array("den").reshape(nsp, -1)
                    den[-1] *= 1e6
                    c.set_array("den", den.ravel())
                    if step == 0:
                        e = c.particles(0)
                        for k in ("vx", "vy", "vz"):
                            e[k] = e[k] * 2.8
                        c.set_particles(0, e, int(c.array("next_id")[0]))
            a.step(1)
            b.run_staged(1)
            if step % 2 == 0 and step < 5:
                continue
            a.sync()
            b.sync()
            for s in range(nsp):
                pa, pb = a.particles(s), b.particles(s)
                for k in ("cell_start", "id", "x", "y", "vx", "vy", "vz"):
                    assert np.array_equal(pa[k], pb[k]), f"step {step} species {s} field {k}"
            for nm in ("mccr", "detach_removed", "next_id", "CondCharge", "Lost", "den", "phi", "Ex", "Ey", "Sigma",
                       "sigma_sp", "sum_den", "sum_phi"):
                assert np.array_equal(a.array(nm), b.array(nm)), f"step {step}: {nm}"
        assert a.info().tstep == b.info().tstep == 6
        assert a.array("mccr").sum() > 0
        if shape == "dense":
            assert a.array("detach_removed").sum() > 0, "no detachment happened"
    finally:
        a.close()
        b.close()
