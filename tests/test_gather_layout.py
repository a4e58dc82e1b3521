"""CPU check of the small meshes' block layouts and of the node rows
(tests/cpp/gather_layout_check.cpp)."""
import os
import subprocess

import numpy as np
import pytest

from xyst_amd import riemann as X
from xyst_amd.meshgen import box_mesh, renumber_mesh

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("gather") / "gather_layout_check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-o", out,
                    os.path.join(ROOT, "tests", "cpp", "gather_layout_check.cpp"),
                    os.path.join(ROOT, "xyst_amd", "csrc", "xg_layout.cpp")], check=True)
    return out


@pytest.mark.parametrize("n,order", [(1, "lex"), (2, "lex"), (9, "lex"), (9, "random"),
                                     (14, "rcm+block")])
def test_small_blocks_reach_every_node_once(exe, tmp_path, n, order):
    m = box_mesh(n, seed=n)
    N = m["coord"].shape[1]
    if order == "random":
        m = renumber_mesh(m, np.random.default_rng(3).permutation(N))
    elif order == "rcm+block":
        m = renumber_mesh(m, X.mesh_rcm(N, m["inpoel"]))
        m = renumber_mesh(m, X.mesh_block_order(m["coord"], 1024))
    e, _ = X.mesh_domint(m["coord"], m["inpoel"])
    e = e.astype(np.int32)
    flip = np.random.default_rng(n).random(len(e)) < 0.5     # both orientations
    e[flip] = e[flip][:, ::-1]
    f = tmp_path / "mesh.bin"
    with open(f, "wb") as fh:
        np.array([N, len(e), len(m["triinpoel"]), len(m["inpoel"])], np.int64).tofile(fh)
        for a in (e[:, 0], e[:, 1], m["triinpoel"], m["inpoel"]):
            np.ascontiguousarray(a, np.int32).tofile(fh)
    for kind in ("rhs", "cho", "tet", "rows"):
        for nodes in (1, 16, 31, 77):
            for gather in (1, 4) if kind == "rows" else (0, 1):
                r = subprocess.run([exe, str(f), kind, str(nodes), str(gather)],
                                   capture_output=True, text=True)
                assert r.returncode == 0 and r.stdout.startswith("ok"), \
                    (kind, nodes, gather, r.stderr)


@pytest.mark.parametrize("n,lanes", [(20, 1), (20, 4), (37, 1)])
def test_row_sums_round_less_than_in_input_order(tmp_path, n, lanes):
    """Numbered as bench.py numbers its meshes, the edges of a node ascend by
    neighbour, and terms that nearly cancel lie far apart in input order: the
    layout's order has to do better by a fifth (it does by a third)."""
    from tests.meshes import smooth_state
    exe = str(tmp_path / "row_sum_check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-o", exe,
                    os.path.join(ROOT, "tests", "cpp", "row_sum_check.cpp"),
                    os.path.join(ROOT, "xyst_amd", "csrc", "xg_layout.cpp")], check=True)
    m = box_mesh(n, seed=n)
    m = renumber_mesh(m, X.mesh_rcm(m["coord"].shape[1], m["inpoel"]))
    m = renumber_mesh(m, X.mesh_block_order(m["coord"], 1024))
    e, d = X.mesh_domint(m["coord"], m["inpoel"])
    u = smooth_state(m["coord"]).T
    f = tmp_path / "sums.bin"
    with open(f, "wb") as fh:
        np.array([u.shape[1], len(e), len(u)], np.int64).tofile(fh)
        np.ascontiguousarray(e.T, np.int32).tofile(fh)
        np.ascontiguousarray(d, np.float64).tofile(fh)
        np.ascontiguousarray(u).tofile(fh)
    r = subprocess.run([exe, str(f), str(lanes)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    rows, ordered = (float(v) for v in r.stdout.split())
    assert rows <= 0.8 * ordered, (rows, ordered)
