"""CPU check of the one-launch f32 GEMM's rule and index maps (tests/gemm_f32_plan_sim.cpp, built with
g++ from rust-gpu_amd/csrc/gemm_f32_plan.h, the header the launcher and the kernel include): output
coverage, K pieces, and that every load is inside its operand or dropped by the range check."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_gemm_f32_plan_simulation(tmp_path):
    exe = str(tmp_path / "gemm_f32_plan_sim")
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Werror", "-o", exe,
                    os.path.join(HERE, "gemm_f32_plan_sim.cpp")], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout[-4000:]
    last = r.stdout.strip().splitlines()[-1]
    assert last.endswith(" 0 failures") and int(last.split()[0]) > 100000, r.stdout
