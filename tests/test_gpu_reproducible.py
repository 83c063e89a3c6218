"""Results that must not depend on what else the device is doing.

Members of a batch share the device during their SCFs.  From 65 occupied
orbitals on, their projector factors once came from a library Cholesky that is
not repeatable beside other queues' work; (H2O)16 has 80.
"""

from __future__ import annotations

import numpy as np
import pytest

from vibeqc_amd import AOBasis, Atom, Calculator, FockPlan, shells_for
from vibeqc_amd.geometry import water_cluster

pytestmark = pytest.mark.gpu


def _results(batch):
    result = batch.execute()
    return [(it.energy, it.iterations, it.density_rms, np.asarray(it.forces).tobytes()) for it in result.items]


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_large_members_repeat_bit_for_bit(precision, monkeypatch):
    systems = [water_cluster(n, 3.1 * n ** (1.0 / 3.0), seed=900 + k) for k, n in enumerate([16] * 10 + [15, 14, 13, 8])]
    calculator = Calculator(precision=precision, energy_tolerance=1e-12, density_tolerance=1e-10)
    with calculator.prepare_batch(systems, warm_start=False) as batch:
        concurrent = [_results(batch) for _ in range(3)]
        monkeypatch.setenv("VIBEQC_BATCH_WORKERS", "1")
        alone = _results(batch)
    for again in concurrent:
        assert [k for k, (a, b) in enumerate(zip(again, alone)) if a != b] == []


@pytest.mark.parametrize("hydrogens", [2, 3, 4])
def test_projected_factor_at_the_edge_of_a_cholesky_block(hydrogens):
    """127, 128 and 129 occupied orbitals: one block, and a block with a panel.
    Incremental builds run only on a factor that is the accepted projection of
    the one before, and the density of such orbitals is the occupied projector:
    the converged iterate is within 1e-8 RMS of self-consistency, and 1e-6 of
    the norm leaves that two orders over n elements a row."""
    waters = 25
    atoms = tuple(water_cluster(waters, 3.4 * waters ** (1.0 / 3.0), seed=5))
    x = max(a.position[0] for a in atoms) + 6.0
    for k in range(hydrogens):
        atoms += (Atom(1, (x, 5.0 * k, 0.0)), Atom(1, (x, 5.0 * k, 1.4)))
    nocc = 5 * waters + hydrogens
    orbital, auxiliary = AOBasis(atoms, shells_for("cc-pvdz", atoms)), AOBasis(atoms, shells_for("cc-pvdz-jkfit", atoms))
    with FockPlan(orbital, auxiliary=auxiliary, precision="bf16x3") as plan:
        result = plan.solve(energy_tolerance=1e-10, density_tolerance=1e-8)
        statistics = plan.last_solve_stats()
        overlap, _ = plan.one_electron()
    assert statistics["incremental_builds"] > 0
    d = np.asarray(result.density)
    assert abs(np.sum(d * overlap) - 2 * nocc) < 1e-8
    assert np.linalg.norm(d @ overlap @ d - 2.0 * d) < 1e-6 * np.linalg.norm(d)
