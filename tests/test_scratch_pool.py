"""The pool of the fused step's scratch (csrc/scratch_pool.hpp), compiled for
the CPU over counted blocks: sets are allocated whole or not at all, reused,
bounded, and given back to an allocation that fails."""
import subprocess
from pathlib import Path

ROOT = Path(__file__).resolve().parent.parent


def test_pool_on_counted_blocks(tmp_path):
    exe = tmp_path / "scratch_pool_check"
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Wextra", f"-I{ROOT / 'simplebubblyflowsolver_amd' / 'csrc'}",
                    str(ROOT / "tests" / "scratch_pool_check.cpp"), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr
