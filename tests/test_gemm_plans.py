"""CPU checks of the wide-tile GEMM's plans (infer_amd/csrc/iq_plan.h),
compiled with g++ and run here."""
import os
import subprocess
import tempfile

HERE = os.path.dirname(os.path.abspath(__file__))


def test_gemmw_plans_cover_and_fit():
    with tempfile.TemporaryDirectory() as d:
        exe = os.path.join(d, "test_gemm_plans")
        subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-o", exe,
                        os.path.join(HERE, "cpp", "test_gemm_plans.cpp")], check=True)
        r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr
    assert "0 failures" in r.stdout
