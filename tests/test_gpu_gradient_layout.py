"""Forces at the edges of the gradient's partial-sum layout: one and many
blocks of auxiliary functions, every orbital class up to f, and from one to all
64 lanes of a wave per shell pair in the one-electron kernel.

Tolerance: both sides converge to 1e-10 RMS in the density; a force is linear
in that error with coefficients of order one per basis function, so 1e-7
Eh/bohr covers n = 72 with two orders to spare.
"""

from __future__ import annotations

import numpy as np
import pytest

from _cases import molecule_case, posthf_case
from vibeqc_amd.geometry import water_cluster

pytestmark = pytest.mark.gpu


def _case(name):
    if name.startswith("water"):
        n = int(name[5:])
        return molecule_case(name, water_cluster(n, 3.4 * n ** (1.0 / 3.0), seed=11))
    return posthf_case(name)[0]


@pytest.mark.parametrize("name", ["h2", "lih", "f_heh", "water1", "water3"])
def test_forces_match_the_oracle(oracle, name):
    from vibeqc_amd import FockBuildSpec, FockPlan

    case = _case(name)
    shells, aux = case.oracle_shells(oracle), case.oracle_shells(oracle, True)
    problem = case.oracle_problem(oracle)
    scf = oracle.df_rhf(problem, energy_tolerance=1e-12, density_tolerance=1e-10)
    reference = -oracle.df_rhf_gradient(case.z, case.xyz, shells, case.spherical, aux, case.spherical, problem, scf)
    with FockPlan(case.orbital(), FockBuildSpec.hf(), auxiliary=case.auxiliary()) as plan:
        forces = plan.solve(compute_forces=True, energy_tolerance=1e-12, density_tolerance=1e-10).forces
    assert np.abs(forces - reference).max() < 1e-7
    assert np.abs(forces.sum(axis=0)).max() < 1e-9
