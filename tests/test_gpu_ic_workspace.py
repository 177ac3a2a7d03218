"""Second-order initial conditions on a plan whose meshes and kept workspace
hold an earlier call's fields: other seeds, sub-ranges and force solves in
between give a fresh plan's particles bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [4, 12, 64])
def test_2lpt_on_a_used_plan(pm, n):
    from gadget_ng_pm_hip import ic
    print(f"case 2lpt workspace n={n}", flush=True)
    cells = n ** 3

    def spectrum(k):
        return 0.05 * cells / max(k, 1.0)

    plan = pm.Plan(n, 10.0)
    ic.zeldovich_2lpt_ics(plan, 3, spectrum)
    rng = np.random.default_rng(n)
    pos = rng.uniform(0.0, 10.0, (500, 3))
    plan.accelerations_f64(pos, np.ones(500), 1.0)
    lo, hi = cells // 3, cells // 3 + min(cells // 2, 999)
    got = ic.zeldovich_2lpt_ics(plan, 8, spectrum, lo=lo, hi=hi)
    first = ic.zeldovich_ics(plan, 8, spectrum)
    fresh = pm.Plan(n, 10.0)
    ref = ic.zeldovich_2lpt_ics(fresh, 8, spectrum)
    assert np.array_equal(got[0], ref[0][lo:hi]) and np.array_equal(got[1], ref[1][lo:hi])
    assert np.array_equal(first[0], ic.zeldovich_ics(pm.Plan(n, 10.0), 8, spectrum)[0])
    assert np.array_equal(plan.accelerations_f64(pos, np.ones(500), 1.0), fresh.accelerations_f64(pos, np.ones(500), 1.0))
