"""The row-tile SpMV of the CG kernels at the sizes where tiles end: rows as
long as a tile and longer, diagonal matrices, odd row counts, one-level and
two-level multigrid (needs an MI355X)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _arrow(n):
    """SPD: 4 on the diagonal, 1/sqrt(n) in the first row and column, whose
    squares sum to less than 1: eigenvalues between 3 and 5."""
    ia, ja, a = [0], [], []
    for r in range(n):
        c = np.arange(n) if r == 0 else np.array([0, r])
        v = np.full(c.size, 1.0 / np.sqrt(n))
        v[c == r] = 4.0
        ja.append(c)
        a.append(v)
        ia.append(ia[-1] + c.size)
    return np.array(ia), np.concatenate(ja), np.concatenate(a)


def _diagonal(n):
    return np.arange(n + 1), np.arange(n), 1.0 + np.arange(n) % 7


def _scattered(n, k=7):
    """Symmetric, k random entries a row and their mirror images of 1/(4 k), 2
    on the diagonal: rows of less than 4 k entries, so eigenvalues between 1
    and 3."""
    rng = np.random.default_rng(n)
    i, j = np.repeat(np.arange(n), k), rng.integers(0, n, n * k)
    i, j = i[i != j], j[i != j]
    key = np.unique(np.concatenate([i * n + j, j * n + i, np.arange(n) * (n + 1)]))
    r, c = key // n, key % n
    ia = np.searchsorted(r, np.arange(n + 1))
    assert np.diff(ia).max() <= 4 * k
    a = np.full(key.size, 0.25 / k)
    a[r == c] = 2.0
    return ia, c, a


def _band(n, k):
    """Symmetric, k entries of -1/(2 k) on either side of 2 on the diagonal:
    eigenvalues between 1 and 3."""
    i = np.arange(n)
    c = i[:, None] + np.arange(-k, k + 1)
    ok = (c >= 0) & (c < n)
    a = np.broadcast_to(np.where(np.arange(-k, k + 1) == 0, 2.0, -0.5 / k), c.shape)
    return np.concatenate([[0], np.cumsum(ok.sum(1))]), c[ok], a[ok]


def _multiply(ia, ja, a, x):
    row = np.repeat(np.arange(ia.size - 1), np.diff(ia))
    return np.bincount(row, a * x[ja], ia.size - 1)


@pytest.mark.parametrize("kind,n", [("arrow", 2047), ("arrow", 2048), ("arrow", 2049),
                                    ("arrow", 5001), ("diagonal", 1), ("diagonal", 255),
                                    ("diagonal", 257), ("diagonal", 2 ** 19 + 1),
                                    # lists of at most 700, of 768 to 1000 and of more columns
                                    ("scattered", 700), ("scattered", 1000),
                                    ("scattered", 5000),
                                    # 256 rows a tile up to 11 entries a row, 128 from 13 on
                                    ("band1", 513), ("band5", 4097), ("band6", 4097)])
def test_cg_at_the_edges_of_tiles(kind, n):
    """Condition at most 7, so a relative residual of 1e-12 (1e-10 with the
    FP32 recurrence) leaves at most seven times that error."""
    from xyst_amd import cg as X
    ia, ja, a = {"arrow": _arrow, "diagonal": _diagonal, "scattered": _scattered,
                 "band1": lambda n: _band(n, 1), "band5": lambda n: _band(n, 5),
                 "band6": lambda n: _band(n, 6)}[kind](n)
    print("tiles %s %d" % (kind, n), flush=True)
    x = np.sin(np.arange(n) + 1.0)
    b = _multiply(ia, ja, a, x) * 1e4
    cg = X.ConjugateGradients(X.CSR(1, ia, ja, a))
    nx = np.linalg.norm(x) * 1e4
    for pc in ("none", "jacobi"):
        cg.init(np.zeros(n), b, pc=pc)
        cg.solve(200, 1e-12)
        assert cg.converged
        assert np.linalg.norm(cg.solution() - 1e4 * x) <= 7e-12 * nx
    cg.init(np.zeros(n), b, pc="jacobi")
    cg.solve_reliable(400, 1e-10)
    assert cg.converged
    assert np.linalg.norm(cg.solution() - 1e4 * x) <= 7e-10 * nx
    cg.init(np.zeros(n), b, pc="jacobi")
    cg.solve_flexible(200, 1e-12, pc="jacobi")
    assert cg.converged
    assert np.linalg.norm(cg.solution() - 1e4 * x) <= 7e-12 * nx
    cg.ctx.close()


@pytest.mark.parametrize("n,levels", [(4, 1), (9, 2), (17, 2)])
def test_multigrid_levels(n, levels):
    """Flexible CG with multigrid on ChoCG's pressure matrix: the residual is
    recomputed on the host; a second solve on the same hierarchy gives the
    same bits, one stopped by the iteration limit reports it."""
    from xyst_amd import cg as X
    from xyst_amd.meshgen import box_mesh
    m = box_mesh(n, seed=4)
    A = X.CSR.poisson(m["coord"], m["inpoel"])
    N = A.nrow
    b = np.cos(3.0 * m["coord"][0]) * 1e3
    b[0] = 0.0
    cg = X.ConjugateGradients(A)
    got = []
    for _ in range(2):
        cg.init(np.zeros(N), b, dirbc={0: [(1, 0.0)]}, apply=True, pc="jacobi")
        cg.solve_flexible(100, 1e-10, pc="amg")
        assert cg.converged and cg.inner_total == cg.it
        got.append(cg.solution())
    assert np.array_equal(got[0], got[1])
    assert cg.amg_info()[0] >= levels
    x = got[0]
    r = b - _multiply(A.ia.astype(int), A.ja.astype(int), A.a, x)
    r[0] = 0.0
    assert np.linalg.norm(r) <= 1.01e-10 * np.linalg.norm(b)
    it = cg.it
    for cap in (1, it - 1, it):
        if cap < 1:
            continue
        cg.init(np.zeros(N), b, dirbc={0: [(1, 0.0)]}, apply=True, pc="jacobi")
        cg.solve_flexible(cap, 1e-10, pc="amg")
        assert cg.it == cap and cg.converged == (cap >= it)
    cg.ctx.close()


def test_multigrid_follows_a_new_matrix():
    """A second matrix on the same context gets a hierarchy of its own."""
    from xyst_amd import cg as X
    from xyst_amd.meshgen import box_mesh
    its, ctx = [], None
    for n in (17, 11, 17):
        m = box_mesh(n, seed=4)
        A = X.CSR.poisson(m["coord"], m["inpoel"])
        b = np.cos(3.0 * m["coord"][0]) * 1e3
        cg = X.ConjugateGradients(A, ctx=ctx)
        ctx = cg.ctx
        cg.init(np.zeros(A.nrow), b, dirbc={0: [(1, 0.0)]}, apply=True, pc="jacobi")
        cg.solve_flexible(100, 1e-10, pc="amg")
        assert cg.converged
        its.append(cg.it)
    assert its[0] == its[2]
    ctx.close()
