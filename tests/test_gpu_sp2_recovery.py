"""One-launch purifications that do not deliver: a launch whose blocks stop
waiting for one another (a limit of 0 us on a barrier's own bounded wait, which
every block then leaves by itself), and a degenerate Gershgorin interval."""

from __future__ import annotations

import numpy as np
import pytest

from vibeqc_amd import AOBasis, Atom, FockBuildSpec, FockPlan, shells_for
from vibeqc_amd.geometry import water_cluster

pytestmark = pytest.mark.gpu

TIGHT = {"energy_tolerance": 1e-12, "density_tolerance": 1e-10}


def _solve(atoms, multiplicity):
    orbital = AOBasis(atoms, shells_for("cc-pvdz", atoms), multiplicity=multiplicity)
    auxiliary = AOBasis(atoms, shells_for("cc-pvdz-jkfit", atoms), multiplicity=multiplicity)
    spec = FockBuildSpec.hf("restricted" if multiplicity == 1 else "unrestricted")
    with FockPlan(orbital, spec, auxiliary=auxiliary) as plan:
        result = plan.solve(compute_forces=True, **TIGHT)
        return result, plan.last_solve_stats()


@pytest.mark.parametrize("spin", ["restricted", "unrestricted"])
def test_a_wait_that_runs_out_costs_one_purification(spin, monkeypatch):
    """n = 96 takes several workgroups.  The solve goes on stepwise, so
    every counted density is still a purification (RHF: the guess' launch gave
    up; UHF: both spins' of the first iteration).  Both runs converge the
    density to 1e-10 RMS; energies are second order in that, and forces linear
    with coefficients of order one per function: 1e-7 covers n^2 of them."""
    atoms = tuple(water_cluster(4, 3.4 * 4 ** (1.0 / 3.0), seed=5))
    multiplicity = 1
    if spin == "unrestricted":
        # An amino radical in the place of one water: n = 72 + 24.
        x = max(a.position[0] for a in atoms[:9]) + 5.0
        atoms = atoms[:9] + (Atom(7, (x, 0.0, 0.0)), Atom(1, (x + 1.2, 1.51, 0.0)), Atom(1, (x + 1.2, -1.51, 0.02)))
        multiplicity = 2
    usual, _ = _solve(atoms, multiplicity)
    monkeypatch.setenv("VIBEQC_SP2_WAIT_US", "0")
    short, stats = _solve(atoms, multiplicity)
    spins = 1 if multiplicity == 1 else 2
    assert stats["purified_densities"] >= spins * (stats["iterations"] - 1)
    assert abs(short.energy - usual.energy) < 1e-9
    assert np.abs(np.asarray(short.forces) - np.asarray(usual.forces)).max() < 1e-7


def test_degenerate_interval_goes_to_the_eigensolver():
    """Two H atoms 60 bohr apart: F in the orthonormal basis is a multiple of the
    unit matrix in the core guess, whose interval has no width.  That density
    comes from the eigensolver, which may pick any orbital of the pair: one
    electron pair, idempotent."""
    atoms = (Atom(1, (0.0, 0.0, 0.0)), Atom(1, (0.0, 0.0, 60.0)))
    orbital = AOBasis(atoms, shells_for("sto-3g", atoms))
    auxiliary = AOBasis(atoms, shells_for("cc-pvdz-jkfit", atoms))
    with FockPlan(orbital, auxiliary=auxiliary) as plan:
        result = plan.solve(energy_tolerance=1e-8, density_tolerance=1e-6)
        overlap, _ = plan.one_electron()
    d = np.asarray(result.density)
    assert abs(np.sum(d * overlap) - 2.0) < 1e-10
    assert np.abs(d @ overlap @ d - 2.0 * d).max() < 1e-10
