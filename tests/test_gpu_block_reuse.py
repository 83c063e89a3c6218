"""Plans that take device blocks left by other plans, and results downloaded in
several pieces.

A block that another plan still used, a read of what an earlier plan left in a
block, or a piece of a download lost or out of place would change results that
are otherwise fixed-order sums, so every comparison is exact.
"""

from __future__ import annotations

from concurrent.futures import ThreadPoolExecutor
from threading import Lock

import numpy as np
import pytest

from vibeqc_amd import AOBasis, Calculator, FockPlan, shells_for
from vibeqc_amd.geometry import lowdin_occupied, water_cluster

pytestmark = pytest.mark.gpu


def _plan(atoms):
    return FockPlan(
        AOBasis(atoms, shells_for("cc-pvdz", atoms)), auxiliary=AOBasis(atoms, shells_for("cc-pvdz-jkfit", atoms))
    )


def _singlepoint(waters):
    atoms = water_cluster(waters, 3.4 * waters ** (1.0 / 3.0), seed=waters)
    result = Calculator(method="rhf", basis="cc-pvdz", auxiliary_basis="cc-pvdz-jkfit").singlepoint(atoms)
    return result.energy, np.array(result.forces)


def test_plans_one_after_another():
    """Blocks pass between sizes and between host threads (one plan at a time)."""
    sizes = [2, 5, 1, 3, 2, 5, 1]
    first = {n: _singlepoint(n) for n in dict.fromkeys(sizes)}
    lock = Lock()

    def locked(n):
        with lock:
            return _singlepoint(n)

    with ThreadPoolExecutor(3) as threads:
        later = [_singlepoint(n) for n in sizes] + list(threads.map(locked, sizes))
    for n, (energy, forces) in zip(sizes + sizes, later):
        assert energy == first[n][0]
        assert np.array_equal(forces, first[n][1])


def test_plans_side_by_side():
    """A plan kept open while others come, change precision and go."""
    atoms = water_cluster(3, 5.0, seed=3)
    with _plan(atoms) as kept:
        S, _ = kept.one_electron()
        C = lowdin_occupied(S, 15, seed=1)
        kept.set_precision("bf16x3")
        expected = kept.evaluate_occupied(C)
        for waters in (1, 3, 4):
            with _plan(water_cluster(waters, 6.0, seed=waters)) as other:
                S, _ = other.one_electron()
                for precision in ("fp32", "bf16x3", "fp64"):
                    other.set_precision(precision)
                    other.evaluate_occupied(lowdin_occupied(S, 5 * waters, seed=2))
                    J, K = kept.evaluate_occupied(C)
                    assert np.array_equal(J, expected[0]) and np.array_equal(K, expected[1])


@pytest.mark.parametrize("waters", [1, 5, 6, 30, 31, 43])
def test_downloads_in_pieces(waters):
    """n = 24 to 120 in one wait; 144 up with n^2 doubles just below and above
    one 4 MiB piece, and above two.

    J and K are written as mirror images of their lower triangles.
    """
    atoms = water_cluster(waters, 3.4 * waters ** (1.0 / 3.0), seed=waters)
    with _plan(atoms) as plan:
        S, _ = plan.one_electron()
        C = lowdin_occupied(S, 3, seed=waters)
        J, K = plan.evaluate_occupied(C)
        assert np.array_equal(J, J.T) and np.array_equal(K, K.T)
        assert np.abs(np.diag(J)).min() > 0.0 and np.abs(np.diag(K)).min() > 0.0
        again = plan.evaluate_occupied(C)
        assert np.array_equal(J, again[0]) and np.array_equal(K, again[1])


def test_idle_blocks_are_given_back():
    import ctypes as ct

    from vibeqc_amd import _native, release_cached_memory

    hip = _native.load()  # found among its dependencies: the runtime that the engine uses

    def free_bytes():
        free, total = ct.c_size_t(), ct.c_size_t()
        assert hip.hipMemGetInfo(ct.byref(free), ct.byref(total)) == 0
        return free.value

    energy, _ = _singlepoint(6)
    idle = free_bytes()
    release_cached_memory()
    released = free_bytes()
    # (H2O)6's fitted tensor alone is 66 MB, in one block of at most 256 MiB.
    assert released - idle > 60e6
    assert _singlepoint(6)[0] == energy
