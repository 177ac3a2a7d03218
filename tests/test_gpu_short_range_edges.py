"""Limits of the short-range kernels against the oracle's brute force: the
table of the pair law and the formula on either side of the cut where one
takes over from the other, no and little and much softening, coincident
particles, clumps that make a chunk heavy (more particles in reach than one
wavefront takes) with ragged last chunks, and the smallest sets.  Forces are
FP32 sums of FP32 pair terms of relative error below 1e-6, on FP32
displacements: 1e-5 rms as in the other short-range tests."""
import numpy as np
import pytest

import learned_oracle as lo
from helpers import rms_rel

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def sr(pm):
    from gadget_ng_pm_hip import learned as L
    return L.ShortRange(device=0)


@pytest.mark.parametrize("kernel", ["exact", "reference"])
@pytest.mark.parametrize("ratio", [1.0, 5.0, 5.6, 5.7, 9.0])  # r_cut / r_s; the table ends at sqrt(32) = 5.657
@pytest.mark.parametrize("eps", [0.0, 1e-7, 0.05, 1.0])
def test_pair_law_over_its_range(sr, kernel, ratio, eps):
    print(f"case pair law kernel={kernel} ratio={ratio} eps={eps}", flush=True)
    g = np.random.default_rng(int(ratio * 10))
    box, rc = 12.0, 3.0
    pos = g.uniform(0.0, box, (700, 3))
    pos[:200] = 6.0 + 0.3 * g.normal(size=(200, 3))  # small separations too
    pos = pos.astype(np.float32).astype(np.float64)
    m = g.uniform(0.5, 1.5, 700).astype(np.float32).astype(np.float64)
    got = sr.accelerations(pos, m, box, rc / ratio, rc, eps2=eps * eps, kernel=kernel)
    ref = lo.short_range_direct(pos, m, box, rc / ratio, rc, eps2=eps * eps, kernel=kernel)
    assert rms_rel(got, ref) < 1e-5


@pytest.mark.parametrize("clump,rest", [(8192 - 60, 60), (8193, 3), (9001, 700), (20011, 500)])
@pytest.mark.parametrize("eps", [0.0, 0.05])
def test_heavy_chunks(sr, clump, rest, eps):
    print(f"case heavy chunks clump={clump} rest={rest} eps={eps}", flush=True)
    g = np.random.default_rng(clump)
    box, rs, rc = 32.0, 1.25, 6.25
    pos = np.concatenate([16.0 + 0.5 * g.normal(size=(clump, 3)), g.uniform(0.0, box, (rest, 3))]).astype(np.float32)
    pos[pos >= box] = 0.0
    n = len(pos)
    m = g.uniform(0.5, 1.5, n).astype(np.float32)
    got = sr.accelerations(pos, m, box, rs, rc, eps2=eps * eps)
    idx = np.concatenate([g.choice(clump, 60, replace=False), np.arange(clump, n)[:60]])
    ref = lo.short_range_direct(pos.astype(np.float64), m.astype(np.float64), box, rs, rc, eps2=eps * eps, idx=idx)
    assert rms_rel(got[idx], ref) < 1e-5
    assert np.array_equal(got, sr.accelerations(pos, m, box, rs, rc, eps2=eps * eps))


@pytest.mark.parametrize("eps", [0.0, 1e-3])
def test_coincident_particles_exert_nothing_on_each_other(sr, eps):
    print(f"case coincident eps={eps}", flush=True)
    pos = np.array([[1.0, 2.0, 3.0]] * 5 + [[2.0, 2.0, 3.0], [1.0 + 12.0, 2.0, 3.0]])
    m = np.ones(7)
    got = sr.accelerations(pos, m, 12.0, 0.6, 3.0, eps2=eps * eps)
    ref = lo.short_range_direct(pos[4:6], np.array([6.0, 1.0]), 12.0, 0.6, 3.0, eps2=eps * eps)
    assert np.isfinite(got).all()
    for i in (0, 1, 2, 3, 4, 6):
        assert got[i] == pytest.approx(ref[0] / 1.0, rel=1e-5, abs=1e-6)
    assert got[5] == pytest.approx(ref[1], rel=1e-5, abs=1e-6)


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65])
def test_smallest_sets(sr, n):
    print(f"case smallest n={n}", flush=True)
    g = np.random.default_rng(n)
    pos = g.uniform(0.0, 9.0, (n, 3)).astype(np.float32).astype(np.float64)
    got = sr.accelerations(pos, np.ones(n), 9.0, 0.6, 3.0, eps2=0.01)
    ref = lo.short_range_direct(pos, np.ones(n), 9.0, 0.6, 3.0, eps2=0.01)
    assert np.abs(got - ref).max() <= 1e-5 * max(np.abs(ref).max(), 1e-30)


@pytest.mark.parametrize("kernel", ["exact", "reference"])
@pytest.mark.parametrize("ratio", [5.66, 8.0, 13.0, 13.3, 30.0, 1e12])
@pytest.mark.parametrize("eps", [0.0, 0.05])
def test_pair_law_far_beyond_the_split(sr, kernel, ratio, eps):
    """r_cut of many r_s, to past the end of the table (x = 9.3, r_cut = 13.2
    r_s): a set with separations down to 0.1 r_s, and one whose pairs all lie
    in the tail.  There a relative error e of r counts 2 x^2 times: below
    2 * 30 * 2^-23, half of it for r^2 itself, at x^2 < 30."""
    print(f"case far pair law kernel={kernel} ratio={ratio} eps={eps}", flush=True)
    g = np.random.default_rng(int(min(ratio, 1e3) * 10))
    box, rc = 12.0, 3.0
    rs = rc / ratio
    pos = g.uniform(0.0, box, (500, 3))
    pos[:200] = 6.0 + 0.5 * min(rs, 0.5) * g.normal(size=(200, 3))
    pos = pos.astype(np.float32).astype(np.float64)
    m = g.uniform(0.5, 1.5, 500).astype(np.float32).astype(np.float64)
    got = sr.accelerations(pos, m, box, rs, rc, eps2=(eps * rs) ** 2, kernel=kernel)
    assert np.isfinite(got).all()
    if ratio < 100.0:  # (beyond, FP32 positions do not resolve r_s)
        ref = lo.short_range_direct(pos, m, box, rs, rc, eps2=(eps * rs) ** 2, kernel=kernel)
        assert rms_rel(got, ref) < 1e-5
    d = 2.0 ** 0.5 * 5.4 * rs  # x = 5.4
    pairs = np.array([[1.0, 1.0, 1.0], [7.0, 7.0, 7.0]])
    pairs = np.concatenate([pairs, pairs + [d, 0.0, 0.0]]).astype(np.float32).astype(np.float64)
    if 5.66 < ratio < 100.0:
        got = sr.accelerations(pairs, np.ones(4), box, rs, rc, eps2=(eps * rs) ** 2, kernel=kernel)
        ref = lo.short_range_direct(pairs, np.ones(4), box, rs, rc, eps2=(eps * rs) ** 2, kernel=kernel)
        assert rms_rel(got / np.abs(ref).max(), ref / np.abs(ref).max()) < 2.0 * 30.0 * 2.0 ** -23 * 1.5
