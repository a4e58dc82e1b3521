"""CPU model of how the launches of a Krylov solve learn of its stop
(tests/cpp/stop_check.cpp, xyst_amd/csrc/xg_stop.hpp)."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("seed", [1, 2, 3])
def test_a_workgroup_never_splits(tmp_path, seed):
    exe = str(tmp_path / "stop_check")
    subprocess.run(["g++", "-O1", "-std=c++17", "-o", exe,
                    os.path.join(ROOT, "tests", "cpp", "stop_check.cpp")], check=True)
    r = subprocess.run([exe, str(seed)], capture_output=True, text=True)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout
