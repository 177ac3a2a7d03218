"""The autotuner keeps its defaults where the variants run the same work (the
deposit of a small problem does not sort, so the sorted deposit's choices do
nothing there), and a tuning file is read only if it was written for the
kernels that its choices select."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
DEPOSIT = ("deposit_threads", "deposit_split", "deposit_pair")


@pytest.mark.parametrize("nm", [24, 32, 48])
def test_deposit_choices_of_small_meshes_stay(pm, nm):
    print(f"case tuning nm={nm}", flush=True)
    plan = pm.Plan(nm, 1.0)
    default = {"deposit_threads": 512, "deposit_split": True, "deposit_pair": False}
    for _ in range(12):
        got = plan.autotune(reps=1)
        assert got["tuned"] and {k: got[k] for k in DEPOSIT} == default


@pytest.mark.parametrize("nm,threads", [(64, 512), (128, 256), (512, 256), (1024, 256)])
def test_default_deposit(pm, nm, threads):
    """One tile a workgroup on every mesh: two are slower for even sets, also at
    1024^3."""
    print(f"case default deposit nm={nm}", flush=True)
    got = pm.Plan(nm, 1.0, r_split=0.1).tuning()
    if not got["tuned"]:  # (an earlier autotune of this process holds otherwise)
        assert {k: got[k] for k in DEPOSIT} == {"deposit_threads": threads, "deposit_split": True, "deposit_pair": False}


SCRIPT = """
import sys
sys.path.insert(0, {pkg!r})
import gadget_ng_pm_hip as pm
t = pm.Plan(64, 1.0).tuning()
if {measure!r}:
    t = pm.Plan(64, 1.0).autotune(reps=1)
print("TUNING", t["tuned"], t["deposit_threads"], t["deposit_pair"], flush=True)
"""


def in_a_process(path, measure=False):
    """The tuning of a plan in a process with that tuning file."""
    env = dict(os.environ, GNG_PM_TUNE_FILE=str(path))
    code = SCRIPT.format(pkg=os.path.join(ROOT, "gadget-ng_amd"), measure=measure)
    r = subprocess.run([sys.executable, "-c", code], env=env, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr
    return next(line for line in r.stdout.splitlines() if line.startswith("TUNING")).split()[1:]


def test_tuning_files_of_other_kernels_are_not_read(pm, tmp_path):
    print("case tuning file", flush=True)
    line = "gfx950 64 0 0 0 0 0 0 1 1 1\n"  # 256 threads and two tiles, unlike the default
    default = ["False", "512", "False"]
    old = tmp_path / "old"
    old.write_text(line)
    assert in_a_process(old) == default
    (tmp_path / "other").write_text("gng_pm_tuning_1\n" + line)
    assert in_a_process(tmp_path / "other") == default
    (tmp_path / "empty").write_text("")
    assert in_a_process(tmp_path / "empty") == default
    (tmp_path / "new").write_text("gng_pm_tuning_2\n" + line)
    assert in_a_process(tmp_path / "new") == ["True", "256", "True"]
    # what one process measures, the next one reads
    assert in_a_process(old, measure=True)[0] == "True"
    assert old.read_text().startswith("gng_pm_tuning_2\n")
    assert in_a_process(old)[0] == "True"
