"""The short range in units other than ones of order one.  Positions scaled by
a, masses by b and G by c scale the accelerations by c b / a^2; the oracle
works in FP64, where none of these ranges matters.  Pair terms are FP32 of
relative error below 1e-6 on FP32 displacements: 1e-5 rms as in the other
short-range tests."""
import numpy as np
import pytest

import learned_oracle as lo
from helpers import rms_rel

pytestmark = pytest.mark.gpu

# (length of one base unit, mass of one base unit, G)
UNITS = {"natural": (1.0, 1.0, 1.0), "galactic": (1.0, 1e-2, 43007.1), "si": (1e12, 2e30, 6.674e-11),
         "cgs": (1e14, 2e33, 6.674e-8), "cgs_kpc": (3.1e21, 2e37, 6.674e-8), "si_kg": (1e12, 1.0, 6.674e-11),
         "nano": (1e-9, 1e-27, 6.674e-11), "light": (1.0, 1e-37, 1.0)}


@pytest.fixture(scope="module")
def sr(pm):
    from gadget_ng_pm_hip import learned as L
    return L.ShortRange(device=0)


def particles(n, box):
    g = np.random.default_rng(17)
    pos = g.uniform(0.0, box, (n, 3))
    pos[: n // 3] = 0.5 * box + 0.03 * box * g.normal(size=(n // 3, 3))  # small separations too
    return np.mod(pos, box), g.uniform(0.5, 1.5, n)


@pytest.mark.parametrize("unit", sorted(UNITS))
@pytest.mark.parametrize("kernel", ["exact", "reference"])
@pytest.mark.parametrize("ratio", [5.0, 9.0])
@pytest.mark.parametrize("eps", [0.0, 1e-3, 0.05])
def test_units(sr, unit, kernel, ratio, eps):
    print(f"case units unit={unit} kernel={kernel} ratio={ratio} eps={eps}", flush=True)
    a, b, c = UNITS[unit]
    pos, m = particles(600, 12.0)
    pos = (pos * a).astype(np.float32).astype(np.float64)
    m = (m * b).astype(np.float32).astype(np.float64)
    args = (12.0 * a, 3.0 * a / ratio, 3.0 * a)
    got = sr.accelerations(pos, m, *args, eps2=(eps * a) ** 2, g=c, kernel=kernel)
    ref = lo.short_range_direct(pos, m, *args, eps2=(eps * a) ** 2, g=c, kernel=kernel)
    assert np.isfinite(got).all()
    s = a * a / (b * c)  # back to order one, where the squares neither over- nor underflow
    assert rms_rel(got * s, ref * s) < 1e-5


@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
@pytest.mark.parametrize("eps", [0.0, 0.05])
def test_a_mass_that_is_not_finite_stays_within_its_reach(sr, bad, eps):
    """Neither the particle's own acceleration nor those of particles out of
    its reach depend on it."""
    print(f"case mass={bad} eps={eps}", flush=True)
    pos, m = particles(600, 12.0)
    pos = pos.astype(np.float32).astype(np.float64)
    m = m.astype(np.float32).astype(np.float64)
    pos[0] = pos[1]  # a coincident pair exerts nothing, either way
    m[0] = bad
    got = sr.accelerations(pos, m, 12.0, 0.6, 3.0, eps2=eps * eps)
    r = np.sqrt((lo.minimum_image(pos - pos[0], 12.0) ** 2).sum(axis=1))
    keep = np.concatenate([[0, 1], np.nonzero(r > 3.0 * 1.001)[0]])
    others = np.delete(np.arange(600), [0, 1])
    ref = np.empty((len(keep), 3))
    for k, i in enumerate(keep):
        src = np.concatenate([[i], others[others != i]])
        if r[i] > 3.0:  # the coincident partner counts as usual, the bad mass is out of reach
            src = np.concatenate([src, [1]])
        ref[k] = lo.short_range_direct(pos[src], m[src], 12.0, 0.6, 3.0, eps2=eps * eps, idx=[0])[0]
    assert np.isfinite(got[keep]).all()
    assert rms_rel(got[keep], ref) < 1e-5
