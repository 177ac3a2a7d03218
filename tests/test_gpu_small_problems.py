"""The short pipeline of small problems on every mesh that has it: the sort-free
deposit against the sorted one (which runs when the plan asks for the sorted
gather), density, moments and forces bit for bit, with particle counts at the
edges of a workgroup and of the rule, clumps, particles on the box's faces and
masses of both signs and zero.  (The plane-wise transforms run in every other
test of these meshes, against the oracle.)"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

COUNTS = {4: (1, 2048, 2049), 8: (255, 2048), 12: (257,), 16: (1, 16384, 16385), 24: (4099,), 32: (2, 16384, 16385),
          48: (256, 16384), 64: (1, 16384, 16385), 96: (16384, 16385), 128: (7, 8192, 16385)}


def particles(n, box, seed):
    rng = np.random.default_rng(seed)
    pos = rng.uniform(0.0, box, (n, 3))
    pos[n // 2:] = (0.02 * box * rng.normal(0.0, 1.0, (n - n // 2, 3))) % box  # a clump over the corner
    pos[0] = 0.0
    pos[-1] = np.nextafter(box, 0.0)
    mass = rng.uniform(-0.25, 1.5, n)
    mass[::5] = 0.0
    mass[0] = 1.0
    return pos, mass.astype(np.float32).astype(np.float64)


@pytest.mark.parametrize("nm", sorted(COUNTS))
def test_small_problems(pm, nm):
    box = 3.0
    for n in COUNTS[nm]:
        print(f"case small nm={nm} n={n}", flush=True)
        pos, mass = particles(n, box, 100 * nm + n)
        got = []
        for general in (False, True):
            plan = pm.Plan(nm, box, r_split=0.1, keep_density=True, keep_potential=True)
            plan.set_tuning(interp_sorted=general)
            a = plan.accelerations_f64(pos, mass, 1.5)
            idx = np.arange(0, n, 3)
            f = plan.accelerations_f32(*(np.ascontiguousarray(pos[:, k]) for k in range(3)), mass, 1.5, idx=idx)
            got.append((a, np.asarray(f), plan.density(), plan.potential(), plan.cell_moments(),
                        plan.cell_moments()))
        for x, y in zip(*got):
            assert np.array_equal(x, y)


def test_counts_that_alternate(pm):
    """One plan goes from the short pipeline to the sorted one and back."""
    plan = pm.Plan(32, 1.0, keep_density=True)
    for n in (1000, 40000, 300, 16384, 16385, 1):
        print(f"case alternate n={n}", flush=True)
        pos, mass = particles(n, 1.0, n)
        ref = pm.Plan(32, 1.0, keep_density=True)
        ref.set_tuning(interp_sorted=True)
        assert np.array_equal(plan.accelerations_f64(pos, mass, 1.0), ref.accelerations_f64(pos, mass, 1.0))
        assert np.array_equal(plan.density(), ref.density())
        assert np.array_equal(plan.cell_moments(), ref.cell_moments())
