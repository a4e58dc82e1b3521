"""Parity of the block operators with the oracle on both sides of every size
at which the block layout changes (xg_layout.hpp, *_blocks), needs an MI355X.

Tolerance as in the operators' own tests: 1e-12 of the oracle's round-off
scale of the entry, 1e-11 of the component's maximum for a KozCG step."""
import numpy as np
import pytest

import oracle as O
from tests.meshes import Case, hub_mesh, smooth_state
from xyst_amd.meshgen import box_mesh, renumber_mesh

pytestmark = pytest.mark.gpu


def _case(n):
    """n odd: numbered as generated, n even: RCM and compact cells."""
    from xyst_amd import riemann as X
    m = box_mesh(n, seed=n)
    if n % 2 == 0:
        m = renumber_mesh(m, X.mesh_rcm(m["coord"].shape[1], m["inpoel"]))
        m = renumber_mesh(m, X.mesh_block_order(m["coord"], 1024))
    print("block sizes n=%d" % n, flush=True)
    return Case(m["coord"], m["inpoel"], m["triinpoel"], m["faceset"], (1, 2, 3, 4, 5, 6))


def _close(x, ref, A):
    assert np.all(np.abs(x - ref) <= 1e-12 * A + 1e-300)


# grad changes between 35 and 36, rhs between 29 and 30
@pytest.mark.parametrize("n", [19, 29, 30, 35, 36])
def test_riemann(n):
    from xyst_amd import riemann as X
    c = _case(n)
    U = smooth_state(c.coord)
    U[c.coord[0] < 0.4, 4] *= 3.0
    for flux in ("rusanov", "hllc"):
        ctx = X.Context(0, flux=flux)
        ctx.upload_mesh(c.coord, c.se.sup, c.se.int, c.tri, c.besym)
        G = ctx.grad(U)
        Go, A = O.grad(c.se, c.coord, c.tri, U, absacc=True)
        _close(G, Go, A)
        Gv = Go / c.vol[:, None]
        R = ctx.rhs(Gv, U)
        Ro, A = O.rhs(O.cfg(flux=flux), c.se, c.coord, c.tri, c.besym, Gv, U, absacc=True)
        _close(R, Ro, A)
        assert np.array_equal(R, ctx.rhs(Gv, U))
        ctx.close()


# gather to scatter blocks between 20 and 21, to full blocks between 39 and 40
@pytest.mark.parametrize("n", [20, 21, 39, 40])
def test_kozak(n):
    import torch
    from xyst_amd import kozak as K
    from xyst_amd import riemann as X
    c = _case(n)
    U0 = smooth_state(c.coord)
    U0[c.coord[0] < 0.4, 4] *= 3.0
    ctx = X.Context(0)
    K.upload(ctx, c.coord, c.inpoel)
    R = K.rhs(ctx, 1e-3, U0)
    Ro, A = O.kozak_rhs(O.cfg(), c.coord, c.inpoel, 1e-3, U0, absacc=True)
    _close(R, Ro, A)
    K.setup(ctx, c.vol, c.symnodes, c.symnorms, fctsys=(0, 4))
    U = torch.tensor(U0, device="cuda")
    Un = torch.empty_like(U)
    dt = K.dt_dev(ctx, U, 0.5)
    K.step_dev(ctx, dt, U, Un)
    Uo, _ = O.kozcg_step(O.cfg(), O.fctcfg(True, 1.0, False, [0, 4]), c.coord, c.inpoel, c.vol,
                         dt, c.symnodes, c.symnorms, np.zeros(0, np.int64),
                         np.zeros((0, 5)), U0)
    assert np.all(np.abs(U.cpu().numpy() - Uo) <= 1e-11 * np.abs(Uo).max(0))
    ctx.close()


# the node kernels of the step add the halo slots themselves: full blocks
# (halo slots) at 40, gather blocks (none) at 12; 5 and 6 components.  The
# kernels repeat the oracle's operations per tet; the order of a node's sums
# and the half step's rounding differ.
@pytest.mark.parametrize("n,ns,fct", [(12, 1, True), (40, 0, False), (40, 1, False),
                                      (40, 1, True)])
def test_kozcg_halo_sums(n, ns, fct):
    import torch
    from xyst_amd import kozak as K
    from xyst_amd import riemann as X
    c = _case(n)
    U0 = smooth_state(c.coord)
    U0[c.coord[0] < 0.4, 4] *= 3.0
    U0 = np.column_stack([U0] + [1.0 + 0.3 * np.sin(3.0 * c.coord[1] + i) for i in range(ns)])
    ctx = X.Context(0)
    K.upload(ctx, c.coord, c.inpoel)
    K.setup(ctx, c.vol, c.symnodes, c.symnorms, fct=fct, fctsys=(0, 4), ncomp=5 + ns)
    U = torch.tensor(U0, device="cuda")
    Un = torch.empty_like(U)
    dt = K.dt_dev(ctx, U, 0.5)
    K.step_dev(ctx, dt, U, Un)
    Uo, _ = O.kozcg_step(O.cfg(), O.fctcfg(fct, 1.0, False, [0, 4]), c.coord, c.inpoel, c.vol,
                         dt, c.symnodes, c.symnorms, np.zeros(0, np.int64),
                         np.zeros((0, 5 + ns)), U0)
    assert np.all(np.abs(U.cpu().numpy() - Uo) <= 1e-11 * np.abs(Uo).max(0))
    assert np.array_equal(Un.cpu().numpy(), U0)
    ctx.close()


# gather to full blocks between 29 and 30
@pytest.mark.parametrize("n", [17, 29, 30])
def test_chorin(n):
    from xyst_amd import chorin as X
    from xyst_amd import riemann as R
    c = _case(n)
    e, d = O.chocg_domint(c.coord, c.inpoel)
    se = O.domsuped(c.inpoel, e, d)
    ctx = R.Context(0)
    X.upload(ctx, c.coord, se.sup, se.int, c.tri)
    rng = np.random.default_rng(n)
    U, P = rng.standard_normal((c.npoin, 3)), rng.standard_normal(c.npoin)
    G9, Gp = rng.standard_normal((c.npoin, 9)), rng.standard_normal((c.npoin, 3))
    for flux in ("damp2", "damp4"):
        Ro, A = O.chorin_rhs(O.chocfg(flux=flux, stab=True, mu=0.05), se, c.coord, c.tri, P, U,
                             G9, absacc=True)
        _close(X.rhs(ctx, X.config(flux, stab=True, mu=0.05), P, U, G9), Ro, A)
    Do, A = O.chorin_div(se, c.coord, c.tri, 0.01, P, Gp, U, stab=True, absacc=True)
    _close(X.div(ctx, 0.01, P, Gp, U, np.zeros(c.npoin), stab=True), Do, A)
    Go, A = O.chorin_vgrad(se, c.coord, c.tri, U, absacc=True)
    _close(X.vgrad(ctx, U, np.zeros((c.npoin, 9))), Go, A)
    Fo, A = O.chorin_flux(se, c.coord, c.tri, U, G9, 0.02, absacc=True)
    _close(X.flux(ctx, 0.02, U, G9, np.zeros((c.npoin, 3))), Fo, A)
    ctx.close()


# a node of more neighbours than the small meshes' blocks hold, numbered last:
# one lane per node for the gradient (255, 256 around the change), scatter
# blocks for the rhs, the tet and the chorin operators
@pytest.mark.parametrize("k", [255, 256, 300, 400, 511])
def test_riemann_hub(k):
    from xyst_amd import riemann as X
    print("hub k=%d" % k, flush=True)
    m = hub_mesh(k)
    c = Case(m["coord"], m["inpoel"], m["triinpoel"], m["faceset"], (1,))
    U = smooth_state(c.coord)
    ctx = X.Context(0)
    ctx.upload_mesh(c.coord, c.se.sup, c.se.int, c.tri, c.besym)
    G = ctx.grad(U)
    Go, A = O.grad(c.se, c.coord, c.tri, U, absacc=True)
    _close(G, Go, A)
    Gv = Go / c.vol[:, None]
    R = ctx.rhs(Gv, U)
    Ro, A = O.rhs(O.cfg(), c.se, c.coord, c.tri, c.besym, Gv, U, absacc=True)
    _close(R, Ro, A)
    ctx.close()


@pytest.mark.parametrize("k", [511, 512, 1500])
def test_kozak_hub(k):
    from xyst_amd import kozak as K
    from xyst_amd import riemann as X
    print("hub k=%d" % k, flush=True)
    m = hub_mesh(k)
    U = smooth_state(m["coord"])
    ctx = X.Context(0)
    K.upload(ctx, m["coord"], m["inpoel"])
    Ro, A = O.kozak_rhs(O.cfg(), m["coord"], m["inpoel"], 1e-3, U, absacc=True)
    _close(K.rhs(ctx, 1e-3, U), Ro, A)
    ctx.close()


@pytest.mark.parametrize("k", [615, 616, 1500])
def test_chorin_hub(k):
    from xyst_amd import chorin as X
    from xyst_amd import riemann as R
    print("hub k=%d" % k, flush=True)
    m = hub_mesh(k)
    e, d = O.chocg_domint(m["coord"], m["inpoel"])
    se = O.domsuped(m["inpoel"], e, d)
    ctx = R.Context(0)
    X.upload(ctx, m["coord"], se.sup, se.int, m["triinpoel"])
    rng = np.random.default_rng(k)
    n = k + 1
    U, P = rng.standard_normal((n, 3)), rng.standard_normal(n)
    G9, Gp = rng.standard_normal((n, 9)), rng.standard_normal((n, 3))
    Ro, A = O.chorin_rhs(O.chocfg(flux="damp4", stab=True, mu=0.05), se, m["coord"],
                         m["triinpoel"], P, U, G9, absacc=True)
    _close(X.rhs(ctx, X.config("damp4", stab=True, mu=0.05), P, U, G9), Ro, A)
    Do, A = O.chorin_div(se, m["coord"], m["triinpoel"], 0.01, P, Gp, U, stab=True, absacc=True)
    _close(X.div(ctx, 0.01, P, Gp, U, np.zeros(n), stab=True), Do, A)
    ctx.close()
