"""Layouts of meshes with a node of many neighbours, on the CPU
(tests/cpp/gather_layout_check.cpp): what the blocks' capacities hold is taken
whatever its degree."""
import os
import subprocess

import numpy as np
import pytest

from tests.meshes import hub_mesh
from xyst_amd import riemann as X

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("hub") / "gather_layout_check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-o", out,
                    os.path.join(ROOT, "tests", "cpp", "gather_layout_check.cpp"),
                    os.path.join(ROOT, "xyst_amd", "csrc", "xg_layout.cpp")], check=True)
    return out


def _check(exe, tmp_path, k, hub, *args):
    m = hub_mesh(k, hub)
    e, _ = X.mesh_domint(m["coord"], m["inpoel"])
    e = e.astype(np.int32)
    f = tmp_path / "hub.bin"
    with open(f, "wb") as fh:
        np.array([k + 1, len(e), len(m["triinpoel"]), len(m["inpoel"])], np.int64).tofile(fh)
        for a in (e[:, 0], e[:, 1], m["triinpoel"], m["inpoel"]):
            np.ascontiguousarray(a, np.int32).tofile(fh)
    r = subprocess.run([exe, str(f)] + [str(a) for a in args], capture_output=True, text=True)
    assert r.returncode == 0 and r.stdout.startswith("ok"), (args, r.stderr)


# a block of four lanes per node holds 256 nodes, one of one lane 768
@pytest.mark.parametrize("hub", ["first", "last"])
@pytest.mark.parametrize("k,lanes", [(255, 4), (256, 1), (300, 1), (511, 1), (767, 1)])
def test_gradient_rows(exe, tmp_path, k, lanes, hub):
    _check(exe, tmp_path, k, hub, "gradrows", 0, lanes)


# gather blocks (1) as long as one holds the hub's neighbours, then scatter
# blocks (0), whose nodes need not be with a hub that is numbered last
@pytest.mark.parametrize("kind,k,gather", [
    ("rhs", 311, 1), ("rhs", 312, 0), ("rhs", 400, 0), ("rhs", 1500, 0),
    ("tet", 511, 1), ("tet", 512, 0), ("tet", 1500, 0),
    ("cho", 615, 1), ("cho", 616, 0), ("cho", 1500, 0)])
def test_blocks(exe, tmp_path, kind, k, gather):
    _check(exe, tmp_path, k, "last", kind, 0, gather)


@pytest.mark.parametrize("kind,k", [("rhs", 311), ("tet", 511), ("cho", 615)])
def test_blocks_hub_first(exe, tmp_path, kind, k):
    _check(exe, tmp_path, k, "first", kind, 0, 1)
