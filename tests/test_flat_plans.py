"""Plans of the flat and hold channels-last kernels against what the kernels assume of them, on the CPU."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "atex_amd", "csrc")


def test_flat_plans_cover_every_instance_once(tmp_path):
    exe = str(tmp_path / "flat_plan_check")
    subprocess.run(["g++", "-O1", "-std=c++17", "-I", CSRC, os.path.join(HERE, "flat_plan_check.cc"), "-o", exe],
                   check=True, capture_output=True, text=True)
    run = subprocess.run([exe], capture_output=True, text=True)
    assert run.returncode == 0, run.stdout[-4000:]
    plans, split, held = (int(v) for v in run.stdout.split()[1:])
    assert plans > 100_000 and split > 50_000 and held > 20_000
