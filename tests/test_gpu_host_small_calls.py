"""Host calls whose arrays go through the small mapped buffer, and those just
past its size, give the device entry points' values: without and with an index
list (empty, partial, whole, repeated), for sizes that are no multiple of a
line, repeated so that the buffer is used again."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# 28 bytes a particle in FP64 calls and 16 in FP32 ones fill 2^20 at 37449 and 65536
SIZES = (1, 2, 33, 4097, 37449, 37450, 65536, 65537)


def device_f64(pm, plan, pos, mass, g):
    d_pos, d_m = pm.DeviceArray.from_host(pos), pm.DeviceArray.from_host(mass)
    out = pm.DeviceArray(pos.shape, np.float64)
    plan.solve_device_f64(d_pos.ptr, d_m.ptr, pos.shape[0], out.ptr, g)
    pm.device_synchronize()
    return out.numpy()


@pytest.mark.parametrize("n", SIZES)
def test_small_host_calls(pm, n):
    print(f"case host call n={n}", flush=True)
    rng = np.random.default_rng(n)
    pos = rng.uniform(0.0, 2.0, (n, 3)).astype(np.float32).astype(np.float64)
    mass = rng.uniform(0.5, 1.5, n).astype(np.float32).astype(np.float64)
    plan = pm.Plan(32, 2.0)
    for turn in range(2):
        ref = device_f64(pm, plan, pos, mass, 1.0 + turn)
        assert np.array_equal(plan.accelerations_f64(pos, mass, 1.0 + turn), ref)
        soa = plan.accelerations_f32(*(np.ascontiguousarray(pos[:, k], dtype=np.float32) for k in range(3)),
                                     mass.astype(np.float32), 1.0 + turn)
        assert np.array_equal(np.asarray(soa).T.astype(np.float64), ref)
        for idx in (np.zeros(0, np.int64), np.arange(n)[::-1].copy(), np.arange(0, n, 3), np.zeros(5, np.int64)):
            assert np.array_equal(plan.accelerations_f64(pos, mass, 1.0 + turn, idx=idx), ref[idx])
    for bad in (-1, n):
        with pytest.raises(Exception):
            plan.accelerations_f64(pos, mass, 1.0, idx=np.array([0, bad], np.int64))
