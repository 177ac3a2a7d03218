"""Tiles at the limits of the deposit's slicing: counts at and one past the
slice length, clumps across a tile corner (every slice reads several source
tiles), empty tiles beside heavy ones and an odd number of tiles (a lone tile
in the last two-tile workgroup).  The split deposit's density equals the
unsplit one's bit for bit and the oracle's within its fixed-point rounding."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ITEMS = 8192  # the slice length of solves below 2^23 particles


@pytest.mark.parametrize("nm,count,corner", [(16, ITEMS, False), (16, ITEMS + 1, False), (48, ITEMS + 1, True),
                                             (48, 5 * ITEMS + 3, True), (64, 3 * ITEMS, False), (24, 70001, True)])
@pytest.mark.parametrize("threads,pair", [(256, False), (512, False), (256, True), (512, True)])
def test_slices_at_their_limits(pm, oracle_mod, nm, count, corner, threads, pair):
    print(f"case slices nm={nm} count={count} corner={corner} threads={threads} pair={pair}", flush=True)
    rng = np.random.default_rng(count + nm)
    box = float(nm)
    centre = 16.0 if corner and nm > 16 else 8.0
    pos = (centre + rng.normal(0.0, 0.7, (count, 3)).clip(-6.0, 6.0)) % box
    pos = np.concatenate([pos, rng.uniform(0.0, 2.0, (37, 3))])  # a few particles far from the clump
    mass = rng.uniform(0.5, 1.5, pos.shape[0]).astype(np.float32).astype(np.float64)
    plan = pm.Plan(nm, box, keep_density=True)
    plan.set_tuning(deposit_threads=threads, deposit_pair=pair, deposit_split=False)
    a0 = plan.accelerations_f64(pos, mass, 1.0)
    d0 = plan.density()
    plan.set_tuning(deposit_threads=threads, deposit_pair=pair, deposit_split=True)
    for _ in range(2):
        a1 = plan.accelerations_f64(pos, mass, 1.0)
        assert np.array_equal(plan.density(), d0)
        assert np.array_equal(a1, a0)
    ref = oracle_mod.cic_assign(pos, mass, box, nm).reshape(nm, nm, nm)
    # the density is stored as FP32: half an ulp of each cell, and the
    # fixed-point unit (below 2^-40 of the largest sum) of each contribution
    assert np.abs(d0 - ref).max() <= 2.0 ** -24 * ref.max() * 1.01


@pytest.mark.parametrize("threads,pair", [(256, False), (512, False), (256, True), (512, True)])
@pytest.mark.parametrize("count,spread", [(5 * ITEMS + 3, 0.0), (8 * ITEMS, 0.0), (8 * ITEMS + 1, 0.0),
                                          (100 * ITEMS, 0.0), (100 * ITEMS, 1.0)])
def test_more_slices_wanted_than_there_are(pm, oracle_mod, count, spread, threads, pair):
    """Every particle in the cell just below a tile corner feeds eight tiles.
    5 * 8192 + 3 of them want 8 * 6 = 48 slices of 8192 particles, and the
    table's first half has (2 * 40963 // 8192 + 16) & ~7 = 24: some tiles run
    whole beside the sliced ones, in whatever order they ask.  From 8 * 8192 + 1
    on they take slices of the second half."""
    nm = 48
    print(f"case slices spent count={count} spread={spread} threads={threads} pair={pair}", flush=True)
    rng = np.random.default_rng(7)
    pos = rng.uniform(15.0 - spread, 16.0 + spread, (count, 3))
    mass = rng.uniform(0.5, 1.5, count).astype(np.float32).astype(np.float64)
    plan = pm.Plan(nm, float(nm), keep_density=True)
    plan.set_tuning(deposit_threads=threads, deposit_pair=pair, deposit_split=False)
    a0 = plan.accelerations_f64(pos, mass, 1.0)
    d0 = plan.density()
    plan.set_tuning(deposit_threads=threads, deposit_pair=pair, deposit_split=True)
    for _ in range(3):
        a1 = plan.accelerations_f64(pos, mass, 1.0)
        assert np.array_equal(plan.density(), d0)
        assert np.array_equal(a1, a0)
    ref = oracle_mod.cic_assign(pos, mass, float(nm), nm).reshape(nm, nm, nm)
    assert np.abs(d0 - ref).max() <= 2.0 ** -24 * ref.max() * 1.01


@pytest.mark.parametrize("nm,count", [(32, 1500000), (96, 1900000), (64, 1400001)])
def test_dense_sets(pm, oracle_mod, nm, count):
    """So many particles that an evenly loaded tile holds more than 8192 and the
    slices get longer with the load (only the clump's tile is split at 96^3)."""
    print(f"case dense nm={nm} count={count}", flush=True)
    rng = np.random.default_rng(nm)
    pos = rng.uniform(0.0, nm, (count, 3))
    pos[: count // 10] = (8.0 + rng.normal(0.0, 0.7, (count // 10, 3))) % nm
    mass = rng.uniform(0.5, 1.5, count).astype(np.float32).astype(np.float64)
    plan = pm.Plan(nm, float(nm), keep_density=True)
    got = []
    for split in (False, True, True):
        plan.set_tuning(deposit_split=split)
        got.append((plan.accelerations_f64(pos, mass, 1.0), plan.density(), plan.cell_moments()))
    for g in got[1:]:
        assert all(np.array_equal(x, y) for x, y in zip(g, got[0]))
    ref = oracle_mod.cic_assign(pos, mass, float(nm), nm).reshape(nm, nm, nm)
    assert np.abs(got[0][1] - ref).max() <= 2.0 ** -24 * ref.max() * 1.01


@pytest.mark.parametrize("nm,count", [(16, 32768), (16, 32769), (48, 3 * 32768 + 5)])
def test_moments_of_heavy_tiles(pm, nm, count):
    """Cell moments at and past the slice length, twice (the cleared words and
    counters are left as they were found), against sums in FP64: the fixed
    point has over 2^40 units per mass."""
    print(f"case moments nm={nm} count={count}", flush=True)
    rng = np.random.default_rng(count)
    box = float(nm)
    pos = (8.0 + rng.normal(0.0, 1.5, (count, 3)).clip(-7.5, 7.5)) % box
    pos = np.concatenate([pos, rng.uniform(0.0, box, (300, 3))])
    mass = rng.uniform(0.5, 1.5, pos.shape[0]).astype(np.float32).astype(np.float64)
    plan = pm.Plan(nm, box)
    plan.accelerations_f64(pos, mass, 1.0)
    i = np.floor(pos).astype(np.int64) % nm
    c = (i[:, 2] * nm + i[:, 1]) * nm + i[:, 0]
    f = pos - np.floor(pos) - 0.5
    vals = np.concatenate([mass[:, None] * f, (mass * (f ** 2).sum(1))[:, None], mass[:, None]], axis=1)
    ref = np.stack([np.bincount(c, weights=vals[:, k], minlength=nm ** 3) for k in range(5)], axis=1)
    for _ in range(2):
        got = plan.cell_moments().reshape(-1, 5)
        assert np.abs(got - ref).max() <= count * 2.0 ** -38


def test_boxes_of_an_ensemble(pm, oracle_mod):
    """Clumped boxes beside plain, small and empty ones of the same side in one
    launch per stage: the forces of one pipeline per box bit for bit, replayed,
    and the oracle's."""
    print("case slices of boxes", flush=True)
    rng = np.random.default_rng(3)
    boxes, parts = [], []
    for nm, count, centre in ((32, 30001, 8.0), (32, 0, 8.0), (32, 700, 8.0), (32, 90000, 15.5), (48, 40000, 24.0)):
        pos = (centre + rng.normal(0.0, 0.4, (count, 3))) % nm
        pos[count // 2:] = rng.uniform(0.0, nm, (count - count // 2, 3))
        pos = pos.astype(np.float32)
        pos[pos >= nm] = 0.0
        boxes.append({"grid_size": nm, "box_size": float(nm)})
        parts.append(pos)
    off = np.concatenate([[0], np.cumsum([len(p) for p in parts])])
    pos = np.concatenate(parts)
    mass = rng.uniform(0.5, 1.5, len(pos)).astype(np.float32)
    d = [pm.DeviceArray.from_host(np.ascontiguousarray(a)) for a in (pos[:, 0], pos[:, 1], pos[:, 2], mass)]
    out = [pm.DeviceArray((len(pos),), np.float32) for _ in range(3)]
    batch = pm.Batch(boxes)
    got = []
    for tables in (True, True, False, True):
        batch.set_box_tables(tables)
        for _ in range(2):
            batch.solve_device(*(a.ptr for a in d), off, 1.0, *(o.ptr for o in out))
            pm.device_synchronize()
            got.append(np.stack([o.numpy() for o in out], axis=1))
    for g in got[1:]:
        assert np.array_equal(g, got[0])
    for b, bx in enumerate(boxes):
        if off[b + 1] > off[b]:
            sel = slice(off[b], off[b + 1])
            ref = oracle_mod.pm_accelerations(pos[sel].astype(np.float64), mass[sel].astype(np.float64), bx["box_size"],
                                              bx["grid_size"], 1.0)
            assert np.sqrt(((got[0][sel] - ref) ** 2).sum() / (ref ** 2).sum()) < 1e-5
