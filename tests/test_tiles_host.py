"""CPU check of the SpMV row tiles (xyst_amd/csrc/xg_tiles.cpp)."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("tiles") / "tiles_check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-pthread", "-o", out,
                    os.path.join(ROOT, "tests", "cpp", "tiles_check.cpp"),
                    os.path.join(ROOT, "xyst_amd", "csrc", "xg_tiles.cpp")], check=True)
    return out


@pytest.mark.parametrize("nrow,ncol,mean,nlong", [
    (1, 1, 1, 0), (128, 128, 0, 0), (129, 300, 1, 0), (1000, 1000, 15, 0),
    (3001, 5000, 15, 3), (4000, 2048, 100, 4), (200000, 200000, 15, 2)])
def test_tiles_cover_the_matrix(exe, nrow, ncol, mean, nlong):
    for seed in (1, 2):
        r = subprocess.run([exe] + [str(v) for v in (nrow, ncol, mean, nlong, seed)],
                           capture_output=True, text=True)
        assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout


@pytest.mark.parametrize("mean,rows", [(3, 128), (3, 256), (15, 256)])
def test_tiles_of_given_rows(exe, mean, rows):
    r = subprocess.run([exe, "5001", "5001", str(mean), "2", "3", str(rows)],
                       capture_output=True, text=True)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout


def test_tiles_without_threads(tmp_path):
    """Where no thread can be created the caller's does all the work."""
    out = str(tmp_path / "tiles_check")
    cpp = os.path.join(ROOT, "tests", "cpp")
    subprocess.run(["g++", "-O2", "-std=c++17", "-pthread", "-o", out,
                    os.path.join(cpp, "tiles_check.cpp"), os.path.join(cpp, "no_threads.cpp"),
                    os.path.join(ROOT, "xyst_amd", "csrc", "xg_tiles.cpp")], check=True)
    r = subprocess.run([out, "200000", "200000", "15", "2", "1"], capture_output=True, text=True)
    assert r.returncode == 0 and r.stdout.strip() == "ok", (r.stdout, r.stderr)
