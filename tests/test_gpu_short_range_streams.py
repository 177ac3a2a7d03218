"""One short-range context called on several streams in turn, without waiting
in between: each call's particles, cells, work list and pair-law table live in
the context's buffers, so a call on another stream starts after the one before
it.  The results are those of the calls by themselves, bit for bit."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture
def streams(pm):
    """Two non-blocking streams of the runtime that the library uses."""
    with open("/proc/self/maps") as f:
        hip = ctypes.CDLL(next(line.split()[-1] for line in f if "libamdhip64" in line))
    out = []
    for _ in range(2):
        s = ctypes.c_void_p()
        assert hip.hipStreamCreateWithFlags(ctypes.byref(s), 1) == 0
        out.append(s.value)
    yield out
    pm.device_synchronize()
    for s in out:
        hip.hipStreamDestroy(ctypes.c_void_p(s))


class Call:
    """One particle set with its own geometry, split and output arrays."""

    def __init__(self, pm, seed, n, box, rs, rc, eps, kernel):
        g = np.random.default_rng(seed)
        pos = g.uniform(0.0, box, (n, 3))
        pos[: n // 2] = np.mod(0.5 * box + 0.02 * box * g.normal(size=(n // 2, 3)), box)
        pos[pos >= np.float32(box)] = 0.0
        self.n, self.args = n, (box, rs, rc, eps * eps, 1.0, kernel)
        self.d = [pm.DeviceArray.from_host(np.ascontiguousarray(pos[:, a], dtype=np.float32)) for a in range(3)]
        self.d.append(pm.DeviceArray.from_host(g.uniform(0.5, 1.5, n).astype(np.float32)))
        self.out = [pm.DeviceArray((n,), np.float32) for _ in range(3)]

    def enqueue(self, sr, stream):
        sr.accelerations_device(*(a.ptr for a in self.d), self.n, *self.args, *(a.ptr for a in self.out),
                                stream=stream)

    def result(self):
        return np.stack([a.numpy() for a in self.out])


def test_calls_on_two_streams(pm, streams):
    print("case short range on two streams", flush=True)
    from gadget_ng_pm_hip import learned as L
    calls = [Call(pm, 1, 60000, 32.0, 1.25, 6.25, 0.05, L.SR_EXACT), Call(pm, 2, 3000, 64.0, 0.4, 2.0, 0.0, L.SR_EXACT),
             Call(pm, 3, 40000, 10.0, 0.5, 3.0, 0.1, L.SR_REFERENCE), Call(pm, 4, 65, 9.0, 0.6, 3.0, 0.01, L.SR_EXACT)]
    ref = []
    for c in calls:
        c.enqueue(L.ShortRange(device=0), 0)
        pm.device_synchronize()
        ref.append(c.result())
    # contexts whose buffers already hold the largest set, and a new one whose buffers grow
    used = L.ShortRange(device=0)
    calls[0].enqueue(used, 0)
    for sr in (used, L.ShortRange(device=0)):
        for turn in range(3):
            for k, c in enumerate(calls):
                c.enqueue(sr, streams[(k + turn) % 2])
            pm.device_synchronize()
            for c, r in zip(calls, ref):
                assert np.array_equal(c.result(), r)


def test_cell_order_beside_a_sum(pm, streams):
    print("case cell order beside a sum", flush=True)
    from gadget_ng_pm_hip import learned as L
    big, small = Call(pm, 1, 60000, 32.0, 1.25, 6.25, 0.05, L.SR_EXACT), Call(pm, 5, 5000, 64.0, 0.4, 2.0, 0.0, L.SR_EXACT)
    sr = L.ShortRange(device=0)
    big.enqueue(sr, 0)
    pm.device_synchronize()
    ref = big.result()
    order = pm.DeviceArray((small.n,), np.uint32)
    for _ in range(3):
        big.enqueue(sr, streams[0])
        rc = pm.lib().gng_sr_cell_order(sr._h, *(a.ptr for a in small.d[:3]), small.n, small.args[0], small.args[2],
                                        order.ptr, streams[1])
        assert rc == 0
        pm.device_synchronize()
        assert np.array_equal(big.result(), ref)
        c = np.floor(np.stack([a.numpy() for a in small.d[:3]]).astype(np.float64) * (32.0 / 64.0)).astype(int) % 32
        assert np.array_equal(order.numpy(), np.argsort((c[2] * 32 + c[1]) * 32 + c[0], kind="stable"))
