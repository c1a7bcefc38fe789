"""Multigrid cycle of the mixed solver on lattices whose halving stops at an odd
element count above the dense limit: the further levels (last node kept) against
a direct solve and against the iterations of the nearest lattice that halves.

Bars: true residual 1e-8, solution within 1e-5 of a direct solve of the oracle's
system (those of the other mixed solves); at most 1.6 times the iterations of
the even neighbour (measured 1.0 to 1.3; the polynomial these levels replace
took 1.5 to 10 times on these lattices); repeated solves are bitwise equal.
"""
import numpy as np
import pytest
import scipy.sparse.linalg as spla

import mg_model as G
import oracle as O
from neopz_amd import _lib as L
from neopz_amd import problems as P
from neopz_amd.analysis import Context, TPZLinearAnalysis, TPZStepSolver

pytestmark = pytest.mark.gpu


def _box(nx, ny, nz, mat=P.POISSON, p=1, seed=0):
    dim = 3 if nz else 2
    pb = P.Problem(material=mat, dim=dim, p=p, nx=nx, ny=ny, nz=max(nz, 1), force_kind=P.FORCE_CONST,
                   force_const=(1.0, 0.2, -0.5), bc_type=[0, -1, 0, -1, 0 if nz else -1, -1])
    if mat != P.POISSON:
        pb.el_coef = np.exp(np.random.default_rng(seed).standard_normal(pb.nvol))
    return pb


# (odd lattice, the same with even counts): all odd, one direction odd, odd
# after one halving, odd on every level, short directions (2 nodes, 1 element)
CASES = {
    "plane_63x51": (lambda: _box(63, 51, 0), lambda: _box(64, 48, 0)),
    "plane_50x50_p2": (lambda: _box(50, 50, 0, P.DARCY, 2, 1), lambda: _box(48, 48, 0, P.DARCY, 2, 1)),
    "plane_127x17": (lambda: _box(127, 17, 0, P.DARCY), lambda: _box(128, 16, 0, P.DARCY)),
    "box_11": (lambda: _box(11, 11, 11, P.POISSON, 2), lambda: _box(12, 12, 12, P.POISSON, 2)),
    "box_13x12x15": (lambda: _box(13, 12, 15, P.DARCY), lambda: _box(12, 12, 16, P.DARCY)),
    "slab_31x31x1": (lambda: _box(31, 31, 1, P.DARCY), lambda: _box(32, 32, 1, P.DARCY)),
    "elast_9x8x7": (lambda: _box(9, 8, 7, P.ELAST3D, 2), lambda: _box(8, 8, 8, P.ELAST3D, 2)),
}


def _solve(ctx, pb):
    an = TPZLinearAnalysis(pb, False, ctx=ctx)
    st = TPZStepSolver()
    st.SetMixedFCG(200000, 1e-8, precond=L.PRECOND_MULTIGRID)
    an.SetSolver(st)
    an.Assemble()
    u = an.Solve()
    v = an.Solve()
    assert np.array_equal(u, v)
    assert st.info["converged"] and st.info["true_residual"] <= 1e-8 and not st.info["fallback"]
    return u, st.info["iterations"]


@pytest.mark.parametrize("name", list(CASES))
def test_odd_lattices_coarsen(name):
    odd, even = (f() for f in CASES[name])
    ctx = Context(0)
    u, it = _solve(ctx, odd)
    _, it_even = _solve(ctx, even)
    print(f"[gpu] {name}: {it} iterations, even neighbour {it_even}", flush=True)
    assert it <= 1.6 * it_even + 2
    o = O.Oracle(odd)
    ia, ja = o.pattern()
    a, rhs = o.assemble()
    x = spla.spsolve(G.full_from_upper(ia, ja, a, o.neq).tocsc(), rhs)
    assert np.linalg.norm(u - x) <= 1e-5 * np.linalg.norm(x)
    ctx.close()


def test_apply_and_solve_in_turn():
    """pzg_mg_apply keeps its own levels (a polynomial at the odd count) and
    the solver its: used in turn on one assembly they do not disturb each
    other."""
    pb = _box(11, 11, 11, P.POISSON, 2)
    ctx = Context(0)
    an = TPZLinearAnalysis(pb, False, ctx=ctx)
    st = TPZStepSolver()
    st.SetMixedFCG(200000, 1e-8, precond=L.PRECOND_MULTIGRID)
    an.SetSolver(st)
    an.Assemble()
    r = np.random.default_rng(1).standard_normal(an.mesh["neq"])
    zs, us = [], []
    for _ in range(2):
        z = np.zeros_like(r)
        L.check(ctx.lib.pzg_mg_apply(ctx.h, L.INNER_MATFREE, 0, 0.0, L.ptr(r, L.dp), L.ptr(z, L.dp), None, None,
                                     None))
        zs.append(z)
        us.append(an.Solve())
    assert np.array_equal(zs[0], zs[1]) and np.array_equal(us[0], us[1])
    ctx.close()
