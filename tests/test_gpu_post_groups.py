"""Error norms on meshes large enough for several elements per group of lanes,
against the oracle.

Bars: those of the error norms at small sizes: |e - e_ref| <= 1e-12 |e_ref| +
1e-13 max|e_ref| per element (sums of squares of FP64 values over the same
points).  Sizes: element counts that leave the last group partly filled, groups
whose elements have different table columns (a change of the vertices' order
inside the list), elements without equations on some sides (orders 1 and 2
mixed).
"""
import numpy as np
import pytest

import oracle as O
from neopz_amd import problems as P
from neopz_amd.analysis import Context, TLaplaceExample1, TPZLinearAnalysis

pytestmark = pytest.mark.gpu

CASES = {
    "tet_p2": lambda: P.darcy3d_tet(n=12, pmax=2, seed=1, hp=False),
    "tet_hp2": lambda: P.darcy3d_tet(n=15, pmax=2, seed=2, hp=True),
    "quad_p2": lambda: P.darcy2d(n=65, p=2, seed=3),
    "elast_hex_p1": lambda: P.elasticity3d(n=17, p=1, seed=4),
}


def _close(e, e_ref):
    floor = 1e-13 * np.max(np.abs(e_ref))
    assert np.all(np.abs(e - e_ref) <= 1e-12 * np.abs(e_ref) + floor)


@pytest.mark.parametrize("name", list(CASES))
def test_errors_match_oracle(name):
    pb = CASES[name]()
    porder = 6  # 64 points per element and more: a wavefront per group
    ctx = Context(0)
    an = TPZLinearAnalysis(pb, False, ctx=ctx)
    o = O.Oracle(pb)
    u = np.random.default_rng(7).standard_normal(o.neq)
    an.LoadSolution(u)
    if pb.nstate == 1:
        ex = TLaplaceExample1(TLaplaceExample1.ECosCos, center=(0.1, -0.2, 0.3))
        an.SetExact(ex.ExactSolution(), porder)
        ref = dict(kind=O.EXACT_COSCOS, center=(0.1, -0.2, 0.3))
    else:
        def exact(x):
            return np.sin(x), np.repeat(np.cos(x)[:, :, None], 3, axis=2)
        an.SetExact(exact, porder)
        uq, duq = exact(o.error_points(porder))
        ref = dict(kind=O.EXACT_POINTS, uq=uq, duq=duq)
    tot = an.PostProcessError(store_error=True)
    el_r, tot_r = o.evaluate_error(u, porder=porder, **ref)
    _close(an.ElementSolution(), el_r)
    _close(tot, tot_r)
    ctx.close()
