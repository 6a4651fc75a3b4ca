"""The plans that a thread keeps: each size planned once while no more than sixteen are in use, whatever they have in common."""
import subprocess
from pathlib import Path

HERE = Path(__file__).resolve().parent


def test_sizes_in_turn_are_planned_once(tmp_path):
    exe = tmp_path / "plan_cache_test"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", f"-I{HERE.parent / 'gemm-zoo_amd' / 'csrc'}", str(HERE / "plan_cache_test.cpp"),
                    "-o", str(exe)], check=True)
    p = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert p.returncode == 0 and p.stdout.strip() == "ok", p.stdout
