"""The autotuner keeps its defaults where the variants run the same work (the
deposit of a small problem does not sort, so the sorted deposit's choices do
nothing there)."""
import pytest

pytestmark = pytest.mark.gpu

DEPOSIT = ("deposit_threads", "deposit_split", "deposit_pair")


@pytest.mark.parametrize("nm", [24, 32, 48])
def test_deposit_choices_of_small_meshes_stay(pm, nm):
    print(f"case tuning nm={nm}", flush=True)
    plan = pm.Plan(nm, 1.0)
    default = {"deposit_threads": 512, "deposit_split": True, "deposit_pair": False}
    for _ in range(12):
        got = plan.autotune(reps=1)
        assert got["tuned"] and {k: got[k] for k in DEPOSIT} == default
