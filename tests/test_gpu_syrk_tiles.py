"""J and K at the edges of the SYRK tiles: 16, 64, 128 and 256 rows and one
more or less, in every precision, against the fitted tensor in numpy.

The reference K is W W^T from B (the oracle's exact factor of the metric) in
FP64.  Tolerances, relative to the largest element: FP64 1e-11 (a metric of
condition 1e7 in FP64); FP32 1e-5 (sums of up to 1e5 products, rounding 6e-8
each, adding like their square root); BF16X3 1e-4 (products to 2^-16).
"""

from __future__ import annotations

import numpy as np
import pytest

from _cases import molecule_case
from vibeqc_amd import Atom
from vibeqc_amd.geometry import lowdin_occupied, water_cluster

pytestmark = pytest.mark.gpu

TOLERANCE = {"fp64": 1e-11, "fp32": 1e-5, "bf16x3": 1e-4}


def _case(waters, hydrogens):
    atoms = tuple(water_cluster(waters, 3.4 * waters ** (1.0 / 3.0), seed=3)) if waters else ()
    x = max((a.position[0] for a in atoms), default=0.0) + 4.0
    atoms += tuple(Atom(1, (x, 2.5 * k, 0.3 * (k % 3))) for k in range(hydrogens))
    return molecule_case("syrk", atoms)


@pytest.mark.parametrize("waters,hydrogens,nocc", [(0, 3, 1), (0, 13, 5), (1, 8, 3), (5, 2, 33), (5, 1, 20), (10, 3, 7)])
def test_jk_at_tile_edges(oracle, waters, hydrogens, nocc):
    from vibeqc_amd import FockPlan

    case = _case(waters, hydrogens)
    problem = case.oracle_problem(oracle)
    C = lowdin_occupied(problem.S, nocc, seed=nocc)
    D = 2.0 * C @ C.T
    J, K = oracle.jk(problem.B, D)
    with FockPlan(case.orbital(), auxiliary=case.auxiliary()) as plan:
        for precision, tolerance in TOLERANCE.items():
            plan.set_precision(precision)
            j, k = plan.evaluate_occupied(C)
            assert np.abs(j - J).max() <= tolerance * np.abs(J).max()
            assert np.abs(k - K).max() <= tolerance * np.abs(K).max()
            assert np.array_equal(k, k.T)


def test_wide_tiles_match_fp64():
    """n = 408 takes the 256-wide BF16X3 tiles, whose second row block is
    partly empty; FP64 (64-wide tiles, checked against 64-bit torch below) is the
    reference."""
    from vibeqc_amd import AOBasis, FockPlan, shells_for

    atoms = water_cluster(17, 3.4 * 17 ** (1.0 / 3.0), seed=3)
    with FockPlan(AOBasis(atoms, shells_for("cc-pvdz", atoms)), auxiliary=AOBasis(atoms, shells_for("cc-pvdz-jkfit", atoms))) as plan:
        S, _ = plan.one_electron()
        C = lowdin_occupied(S, 85, seed=2)
        _, K = plan.evaluate_occupied(C)
        plan.set_precision("bf16x3")
        _, k = plan.evaluate_occupied(C)
    assert np.abs(k - K).max() <= TOLERANCE["bf16x3"] * np.abs(K).max()
    assert np.array_equal(k, k.T)


# The 64-bit torch restatement of the performance cases, which shares no code
# with the engine; in a process of its own, since torch and the engine bring
# their own HIP runtimes.
RESTATED = """
import importlib.util, sys
import numpy as np, torch
from vibeqc_amd.geometry import lowdin_occupied, water_cluster
path, waters, nocc, out = sys.argv[1], int(sys.argv[2]), int(sys.argv[3]), sys.argv[4]
spec = importlib.util.spec_from_file_location("performance_cases", path)
cases = importlib.util.module_from_spec(spec)
spec.loader.exec_module(cases)
atoms = water_cluster(waters, 3.4 * waters ** (1.0 / 3.0), seed=3)
integrals = cases._Integrals(atoms, *cases._bases({"molecule": "water"}, atoms), "cuda")
C = lowdin_occupied(integrals.one_electron()[0].cpu().numpy(), nocc, seed=nocc)
J, K = cases._Fitted(integrals).jk(np.sqrt(2.0) * torch.from_numpy(C).cuda())
np.savez(out, C=C, J=J.cpu().numpy(), K=K.cpu().numpy())
"""


@pytest.mark.parametrize("waters,nocc", [(17, 9), (30, 5)])
def test_jk_beyond_400_functions(waters, nocc, tmp_path):
    """n = 408 (narrow FP64 and FP32 tiles, split rule of large n) and 720 (wide
    ones, remainders of 208 rows and 80 columns).  FP64 1e-9: the engine leaves
    out primitive pairs below 1e-10 of the screening threshold, and the metric's
    condition of 1e7 multiplies 1e-16."""
    import subprocess
    import sys
    from pathlib import Path

    from vibeqc_amd import AOBasis, FockPlan, shells_for

    root = Path(__file__).resolve().parent.parent
    subprocess.run([sys.executable, "-c", RESTATED, str(root / "perf" / "cases.py"), str(waters), str(nocc),
                    str(tmp_path / "jk.npz")], cwd=root, check=True, timeout=600)
    reference = np.load(tmp_path / "jk.npz")
    C, J, K = reference["C"], reference["J"], reference["K"]
    atoms = water_cluster(waters, 3.4 * waters ** (1.0 / 3.0), seed=3)
    orbital, auxiliary = AOBasis(atoms, shells_for("cc-pvdz", atoms)), AOBasis(atoms, shells_for("cc-pvdz-jkfit", atoms))
    with FockPlan(orbital, auxiliary=auxiliary) as plan:
        for precision, tolerance in {**TOLERANCE, "fp64": 1e-9}.items():
            plan.set_precision(precision)
            j, k = plan.evaluate_occupied(C)
            assert np.abs(j - J).max() <= tolerance * np.abs(J).max()
            assert np.abs(k - K).max() <= tolerance * np.abs(K).max()
            assert np.array_equal(k, k.T)
