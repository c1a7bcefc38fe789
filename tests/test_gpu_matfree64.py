"""FP64 products on meshes of identical affine p = 2 hexahedra against the
oracle's assembled matrix: element by element on the large mesh, by the block CSR
on the small ones (fewer than 96 elements, 6000 with one unknown a node; both
sides of these limits are in test_gpu_element_product_sizes.py).

Bar: |K x - K_ref x| <= 1e-13 * sum_j |K_ij| |x_j| per row: both sums have at
most a few hundred terms of that size, added in another order (64 eps = 1.4e-14
times a small factor).  Element counts that are no multiple of the 16-element
tile, a single element, one and three wavefronts per tile (below and above the
split), several Dirichlet faces meeting in an edge, and coefficients for which
AddKel drops entries in some elements only (the block CSR is used then).
"""
import ctypes as C
import os

import numpy as np
import pytest

import oracle as O
from neopz_amd import _lib as L
from neopz_amd import mesh as M
from neopz_amd import problems as P
from neopz_amd.analysis import Context, TPZLinearAnalysis, TPZStepSolver

pytestmark = pytest.mark.gpu


def _elast(nx, ny, nz, faces, seed=0, scale=1.0):
    pb = P.Problem(material=P.ELAST3D, dim=3, p=2, nx=nx, ny=ny, nz=nz, E=1.0, nu=0.3,
                   force_kind=P.FORCE_CONST, force_const=(0.3, -1.0, 0.2),
                   bc_type=[0 if f in faces else -1 for f in range(6)])
    pb.el_coef = scale * np.exp(np.random.default_rng(seed).standard_normal(pb.nvol))
    return pb


def _scalar(n, seed=0):
    pb = P.Problem(material=P.DARCY, dim=3, p=2, nx=n, ny=n, nz=n, force_kind=P.FORCE_CONST,
                   force_const=(1.0, 0, 0), bc_type=[0] * 6)
    pb.el_coef = np.exp(np.random.default_rng(seed).standard_normal(pb.nvol))
    return pb


def _mixed_drop(n):
    # coefficients over 14 decades: AddKel keeps an entry in some elements only
    pb = _elast(n, n, n, (0,))
    pb.el_coef = 10.0 ** np.linspace(-12, 2, pb.nvol)
    return pb


CASES = {
    "one_element": lambda: _elast(1, 1, 1, (4,)),
    "elast_5x3x2": lambda: _elast(5, 3, 2, (0, 2, 5), 1),
    "elast_15_tiny": lambda: _elast(5, 3, 1, (0,), 2, 1e-3),
    "elast_all_faces": lambda: _elast(4, 4, 4, range(6), 3),
    "scalar_7": lambda: _scalar(7, 4),
    "drop_some": lambda: _mixed_drop(3),
}


@pytest.mark.parametrize("name", list(CASES))
def test_product_matches_oracle(name):
    pb = CASES[name]()
    o = O.Oracle(pb)
    ia, ja = o.pattern()
    a, rhs = o.assemble()
    ctx = Context(0)
    an = TPZLinearAnalysis(pb, False, ctx=ctx)
    st = TPZStepSolver()
    st.SetCG(5000, TPZStepSolver.jacobi(), 1e-10, 0)
    an.SetSolver(st)
    an.Assemble()
    rng = np.random.default_rng(5)
    x, y = rng.standard_normal(o.neq), rng.standard_normal(o.neq)
    z = an.K.MultAdd(x, y, 0.7, -0.4)
    ref = O.multadd(ia, ja, a, x, y, 0.7, -0.4)
    bound = O.multadd(ia, ja, np.abs(a), np.abs(x), np.abs(y), 0.7, 0.4)
    assert np.all(np.abs(z - ref) <= 1e-13 * bound)
    if name == "drop_some":  # 14 decades of coefficients: the product only, no solve converges
        ctx.close()
        return
    u = an.Solve()
    assert st.info["converged"]
    # the reported true residual is that of the assembled matrix
    r = rhs - O.multadd(ia, ja, a, u)
    rb = O.multadd(ia, ja, np.abs(a), np.abs(u))
    rel = np.linalg.norm(r) / np.linalg.norm(rhs)
    slack = 1e-13 * np.linalg.norm(rb) / np.linalg.norm(rhs)
    assert abs(st.info["true_residual"] - rel) <= 1e-6 * rel + slack
    v, w = C.c_double(), C.c_double()
    L.check(ctx.lib.pzg_true_residual(ctx.h, C.byref(v)))
    L.check(ctx.lib.pzg_true_residual_noalloc(ctx.h, C.byref(w)))
    assert v.value == w.value
    ctx.close()


def test_large_mesh_matches_block_csr():
    """Above the split (one wavefront per tile of 16 elements): the product
    against the block CSR of the same assembly (element scatter, separate
    environment switch read by pzg_struct_create)."""
    pb = _elast(41, 41, 41, (0, 4), 6)
    ctx = Context(0)
    md = M.build(pb)
    x = np.random.default_rng(8).standard_normal(md["neq"])
    # zero on the Dirichlet faces: their rows then hold no term 1e12 times the
    # others, and max |z| bounds every row's sum of |terms| within a factor 50
    bpos = md["blk_pos"][np.unique(md["bc_conn"])]
    x[(bpos[:, None] + np.arange(3)).ravel()] = 0.0
    zs = []
    for off in ("0", "1"):
        os.environ["PZG_NO_BLKASM"] = off
        try:
            an = TPZLinearAnalysis(md, False, ctx=ctx)
            an.Assemble()
            zs.append(an.K.Multiply(x))
        finally:
            del os.environ["PZG_NO_BLKASM"]
    # 64 eps on row sums of |terms| <= 50 max |z|
    assert np.max(np.abs(zs[0] - zs[1])) <= 1e-12 * np.max(np.abs(zs[1]))
    ctx.close()
