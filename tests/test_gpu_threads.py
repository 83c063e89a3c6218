"""Plans that overlap: solved, opened and closed by several threads at once,
each on its own stream.  Every result is that of the same call alone, bit for
bit (all sums of a solve have a fixed order), and every density comes from a
purification (a wait that ran out would leave it to the eigensolver)."""

from __future__ import annotations

from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

from vibeqc_amd import AOBasis, Atom, Calculator, FockPlan, shells_for
from vibeqc_amd.geometry import water_cluster

pytestmark = pytest.mark.gpu


def _atoms(waters, hydrogens=0):
    atoms = tuple(water_cluster(waters, 3.2 * waters ** (1.0 / 3.0), seed=40 + waters))
    x = max(a.position[0] for a in atoms) + 6.0
    for k in range(hydrogens):
        atoms += (Atom(1, (x, 5.0 * k, 0.0)), Atom(1, (x, 5.0 * k, 1.4)))
    return atoms


def test_plans_solved_at_once():
    molecules = [_atoms(3, 1), _atoms(6), _atoms(8), _atoms(16)]  # 82 to 384 functions: several workgroups each
    plans = [FockPlan(AOBasis(m, shells_for("cc-pvdz", m)), auxiliary=AOBasis(m, shells_for("cc-pvdz-jkfit", m)))
             for m in molecules]

    def solve(plan):
        result = plan.solve(energy_tolerance=1e-12, density_tolerance=1e-10)
        stats = plan.last_solve_stats()
        assert stats["purified_densities"] == stats["iterations"]
        return result.energy, np.asarray(result.density)

    alone = [solve(p) for p in plans]
    with ThreadPoolExecutor(len(plans)) as pool:
        together = [list(pool.map(solve, plans)) for _ in range(4)]
    for results in together:
        for (energy, density), (energy0, density0) in zip(results, alone):
            assert energy == energy0
            assert np.array_equal(density, density0)
    for p in plans:
        p.close()


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_plans_opened_and_closed_at_once(precision):
    molecules = [_atoms(2), _atoms(5), _atoms(7), _atoms(10)]

    def point(atoms):
        result = Calculator(precision=precision).singlepoint(atoms)
        return result.energy, np.asarray(result.forces)

    alone = [point(m) for m in molecules]
    with ThreadPoolExecutor(len(molecules)) as pool:
        together = list(pool.map(point, molecules * 6))
    for k, (energy, forces) in enumerate(together):
        assert energy == alone[k % len(alone)][0]
        assert np.array_equal(forces, alone[k % len(alone)][1])


def test_a_batch_beside_single_plans():
    """A batch in one thread, calculators in three others.  The calculators'
    results are exact; the batch's metric factors then come from another
    Cholesky than alone, so its energies agree to the rounding of a metric of
    condition 1e7 (1e-9 of the two-electron energy's 1e2 Eh a molecule, of which
    J and K see a small part): 1e-8 Eh."""
    from threading import Event

    systems = [_atoms(n) for n in (10, 9, 8, 7, 6, 5, 4, 3)]
    calculator = Calculator(energy_tolerance=1e-12, density_tolerance=1e-10)
    alone = np.asarray(calculator.batch_singlepoint(systems, properties=("energy",)).energies)
    molecules = [_atoms(2), _atoms(5), _atoms(7)]
    energies = [Calculator().singlepoint(m).energy for m in molecules]
    stop = Event()

    def keep_busy(k):
        seen = []
        while not stop.is_set():
            seen.append(Calculator().singlepoint(molecules[k]).energy)
        return seen

    with ThreadPoolExecutor(3) as pool:
        others = [pool.submit(keep_busy, k) for k in range(3)]
        try:
            beside = [calculator.batch_singlepoint(systems, properties=("energy",), strict=True) for _ in range(6)]
        finally:
            stop.set()
        for k, other in enumerate(others):
            assert set(other.result()) == {energies[k]}
    for result in beside:
        assert np.abs(np.asarray(result.energies) - alone).max() < 1e-8
