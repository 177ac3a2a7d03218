"""Short-range sums whose work items fill more than one row of the launch, and
more of them than one grid dimension takes (2^32 work items of a launch)."""
import numpy as np
import pytest

import learned_oracle as lo
from helpers import rms_rel

pytestmark = pytest.mark.gpu


def test_several_rows_of_workgroups(pm):
    """1.6 particles a cell: some 10^6 light chunks.  1e-5 rms as in the other
    short-range tests (FP32 pair terms of relative error below 1e-6)."""
    from gadget_ng_pm_hip import learned as L
    n, box = 3_300_001, 128.0
    print(f"case rows n={n}", flush=True)
    g = np.random.default_rng(6)
    pos = g.uniform(0.0, box, (n, 3)).astype(np.float32)
    pos[pos >= box] = 0.0
    m = g.uniform(0.5, 1.5, n).astype(np.float32)
    sr = L.ShortRange(device=0)
    got = sr.accelerations(pos, m, box, 0.2, 1.0, eps2=1e-4)
    idx = g.choice(n, 25, replace=False)
    ref = lo.short_range_direct(pos.astype(np.float64), m.astype(np.float64), box, 0.2, 1.0, eps2=1e-4, idx=idx)
    assert np.isfinite(got).all()
    assert rms_rel(got[idx], ref) < 1e-5
    c = (pos.astype(np.float64)).astype(np.int64) % 128
    cell = np.bincount((c[:, 2] * 128 + c[:, 1]) * 128 + c[:, 0], minlength=128 ** 3).reshape((128,) * 3)
    reach = cell.copy()
    for axis in range(3):
        reach = reach + np.roll(reach, 1, axis) + np.roll(reach, -1, axis)
    assert sr.last_pair_count() == int((cell * reach).sum())


def test_more_particles_than_one_grid_dimension_takes(pm):
    """730e6 particles in 200^3 cells may make 18.7e6 workgroups of 256 threads;
    every particle's acceleration is written."""
    from gadget_ng_pm_hip import learned as L
    n, box, period = 730_000_000, 200.0, 1 << 22
    print(f"case large short range n={n}", flush=True)
    g = np.random.default_rng(8)
    lib, f4 = pm.lib(), 4
    coord = [pm.DeviceArray((n,), np.float32) for _ in range(3)]
    for k, a in enumerate(coord):
        # copies of one random sequence, rotated against the other axes'
        base = g.uniform(0.0, box, period).astype(np.float32)
        base[base >= box] = 0.0
        src = pm.DeviceArray.from_host(np.concatenate([base, base]))
        for t, lo_ in enumerate(range(0, n, period)):
            rot = (t * k * 7919) % period
            assert lib.gng_dev_copy(a.ptr + f4 * lo_, src.ptr + f4 * rot, f4 * min(period, n - lo_), 2) == 0
        pm.device_synchronize()
    out = [pm.DeviceArray((n,), np.float32) for _ in range(3)]
    mass = pm.DeviceArray((n,), np.float32)
    fill = pm.DeviceArray.from_host(np.concatenate([np.ones(period), np.full(period, np.nan)]).astype(np.float32))
    for lo_ in range(0, n, period):
        size = f4 * min(period, n - lo_)
        assert lib.gng_dev_copy(mass.ptr + f4 * lo_, fill.ptr, size, 2) == 0
        for o in out:
            assert lib.gng_dev_copy(o.ptr + f4 * lo_, fill.ptr + f4 * period, size, 2) == 0
    pm.device_synchronize()
    sr = L.ShortRange(device=0)
    sr.accelerations_device(*(a.ptr for a in coord), mass.ptr, n, box, 0.2, 1.0, 1e-4, 1.0, L.SR_EXACT,
                            *(o.ptr for o in out))
    pm.device_synchronize()
    for o in out:
        assert np.isfinite(o.numpy()).all()
