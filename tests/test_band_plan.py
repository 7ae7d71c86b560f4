"""The band LU's plans (which block is updated in which launch, the sweeps) on
the CPU, for block bandwidths 0 to 8, 1 to 82 blocks and 0 to 5 cuts."""
import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_band_plans_solve_and_have_no_races(tmp_path):
    exe = str(tmp_path / "band_plan_check")
    subprocess.run(["g++", "-O2", "-std=c++17", os.path.join(HERE, "band_plan_check.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout
