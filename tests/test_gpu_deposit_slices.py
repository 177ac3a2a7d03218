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
