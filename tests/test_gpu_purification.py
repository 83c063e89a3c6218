"""SP2 purification at the edges of its kernels' size ranges: one workgroup
(n <= 80), several workgroups (n <= 400, tiles of 16) and the stepwise path.

Every iteration's density has to come from a purification (a kernel that did
not converge would fall back to the eigensolver), and the converged density has
to be the occupied projector of its own Fock matrix, diagonalised by numpy.
The SCF stops at an RMS density change of 1e-10 over n^2 elements, so with DIIS
contracting the error the density is converged to a few times n 1e-10 in norm;
1e-6 of the density's norm leaves room for a slow last step at every n here.
"""

from __future__ import annotations

import numpy as np
import pytest

from vibeqc_amd import AOBasis, Atom, FockPlan, shells_for
from vibeqc_amd.geometry import water_cluster

pytestmark = pytest.mark.gpu


def _molecule(waters, hydrogens):
    atoms = tuple(water_cluster(waters, 3.4 * max(waters, 1) ** (1.0 / 3.0), seed=5)) if waters else ()
    x = max((a.position[0] for a in atoms), default=0.0) + 6.0
    for k in range(hydrogens):
        atoms += (Atom(1, (x, 5.0 * k, 0.0)), Atom(1, (x, 5.0 * k, 1.4)))
    return atoms


@pytest.mark.parametrize(
    "waters,hydrogens,basis,nbf",
    [(0, 1, "sto-3g", 2), (1, 0, "sto-3g", 7), (1, 0, "cc-pvdz", 24), (2, 0, "cc-pvdz", 48), (3, 0, "cc-pvdz", 72),
     (3, 1, "cc-pvdz", 82), (4, 0, "cc-pvdz", 96),
     (4, 1, "cc-pvdz", 106), (6, 0, "cc-pvdz", 144), (8, 1, "cc-pvdz", 202), (16, 1, "cc-pvdz", 394),
     (17, 0, "cc-pvdz", 408)],
)
def test_purified_density_is_the_occupied_projector(waters, hydrogens, basis, nbf):
    atoms = _molecule(waters, hydrogens)
    orbital = AOBasis(atoms, shells_for(basis, atoms))
    auxiliary = AOBasis(atoms, shells_for("cc-pvdz-jkfit", atoms))
    assert orbital.nao == nbf
    with FockPlan(orbital, auxiliary=auxiliary) as plan:
        result = plan.solve(energy_tolerance=1e-12, density_tolerance=1e-10)
        stats = plan.last_solve_stats()
        assert stats["purified_densities"] == stats["iterations"]
        overlap, _ = plan.one_electron()
        fock = plan.evaluate(result.density).fock
    w, v = np.linalg.eigh(overlap)
    x = (v / np.sqrt(w)) @ v.T
    occupied = x @ np.linalg.eigh(x @ fock @ x)[1][:, : orbital.electrons // 2]
    projector = 2.0 * occupied @ occupied.T
    assert np.linalg.norm(result.density - projector) <= 1e-6 * np.linalg.norm(projector)


@pytest.mark.parametrize("distance,singular", [(1e-6, True), (0.05, False), (1.4, False)])
def test_orthogonaliser_of_close_functions(oracle, distance, singular):
    """The overlap's inverse square root of two H atoms whose functions are
    dependent (smallest eigenvalue about distance^2 / 2: refused below 1e-10),
    nearly so, and apart; energies against the oracle (both converge to 1e-12
    Eh; the metric's cutoff and X at a condition of 1e3 cost four digits)."""
    from _cases import molecule_case
    from vibeqc_amd._native import NativeError

    case = molecule_case("h2", (Atom(1, (0.0, 0.0, 0.0)), Atom(1, (0.0, 0.0, distance))), basis="sto-3g")
    with FockPlan(case.orbital(), auxiliary=case.auxiliary()) as plan:
        if singular:
            with pytest.raises(NativeError, match="linearly dependent"):
                plan.solve()
            return
        energy = plan.solve(energy_tolerance=1e-12, density_tolerance=1e-10).energy
    assert abs(energy - oracle.df_rhf(case.oracle_problem(oracle)).energy) < 1e-8
