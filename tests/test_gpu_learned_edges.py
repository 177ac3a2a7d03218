"""Edges of the training kernels: one tile per axis (every halo wraps), more
weight-gradient tiles than workgroups, one and several boxes; loss records in
cell order and in none (more nodes than the workgroup's table holds), zero
weights, a ragged last workgroup."""
import numpy as np
import pytest

import learned_oracle as lo

pytestmark = pytest.mark.gpu


def rel_max(a, b):
    return float(np.abs(np.asarray(a, np.float64) - b).max() / max(np.abs(b).max(), 1e-30))


@pytest.mark.parametrize("nm,boxes,n,ordered", [(16, 1, 257, True), (16, 1, 255, False), (32, 3, 5000, False),
                                                (48, 3, 9001, True)])
def test_loss_and_gradients_at_the_edges(pm, nm, boxes, n, ordered):
    from gadget_ng_pm_hip import learned as L
    print(f"case training edges nm={nm} boxes={boxes} n={n} ordered={ordered}", flush=True)
    g = np.random.default_rng(nm + n)
    box, osc = float(nm), 1.3
    p = {k: v.astype(np.float32) for k, v in lo.init_params(5).items()}
    p["w3"] *= 10.0
    x0 = lo.bf16_round(g.normal(size=(boxes, nm, nm, nm, 8))).astype(np.float32)
    net = L.Net(nm, boxes, device=0)
    net.set_params(p)
    net.write("x0", x0)
    net.forward(boxes)
    pos = g.uniform(0, box, (n, 3)).astype(np.float32)
    pos[: n // 4] = pos[0] + 0.01 * g.normal(size=(n // 4, 3)).astype(np.float32)  # a clump
    pos = np.mod(pos, np.float32(box))
    pos[pos >= box] = 0.0
    bidx = g.integers(0, boxes, n)
    if ordered:
        c = np.floor(pos).astype(np.int64) % nm
        order = np.argsort(((bidx * nm + c[:, 2]) * nm + c[:, 1]) * nm + c[:, 0], kind="stable")
        pos, bidx = pos[order], bidx[order]
    pos4 = np.concatenate([pos, bidx[:, None]], axis=1).astype(np.float32)
    w = np.where(g.random(n) < 0.3, 0.0, g.uniform(0.1, 2.0, n))
    tgt4 = np.concatenate([g.normal(size=(n, 3)), w[:, None]], axis=1).astype(np.float32)
    dp, dt = pm.DeviceArray.from_host(pos4), pm.DeviceArray.from_host(tgt4)
    net.loss_grad(dp.ptr, dt.ptr, n, box, osc)
    y, gy = net.read("y").astype(np.float64), net.read("gy")
    loss = 0.0
    for b in range(boxes):
        sel = pos4[:, 3] == b
        lb, gb = lo.weighted_loss(y[b][..., :3], pos4[sel, :3].astype(np.float64), box, tgt4[sel, :3], tgt4[sel, 3],
                                  osc, n)
        loss += lb
        assert rel_max(gy[b][..., :3], gb) < 1e-5
    assert net.loss() == pytest.approx(loss, rel=1e-5)
    net.backward(boxes)
    gr = L.unpack_params(net.read("grad"))
    x1, x2 = (net.read(k).astype(np.float64) for k in ("x1", "x2"))
    dz3, dz2, dz1 = (net.read(k).astype(np.float64) for k in ("dz3", "dz2", "dz1"))
    for k, xin, dz in (("3", x2, dz3[..., :3]), ("2", x1, dz2), ("1", x0.astype(np.float64), dz1)):
        ref = [lo.conv3d_backward_weights(xin[b], dz[b]) for b in range(boxes)]
        assert rel_max(gr["w" + k], sum(r[0] for r in ref)) < 2e-5, k
        assert rel_max(gr["b" + k], sum(r[1] for r in ref)) < 2e-5, k
