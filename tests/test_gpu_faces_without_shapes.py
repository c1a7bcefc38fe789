"""Dirichlet faces with a connect that carries no equations, on lattices of
identical p = 2 hexahedra: such a face leaves one of its functions unpenalized.
Products and solves against the oracle's assembled matrix.

Bars: FP64 product 1e-13 * |K| |x| per row, FP32 product 30 roundings relative
to |S| |x|, solutions 1e-8 (FP64 CG to 1e-11) and 1e-5 (mixed, true residual
1e-8) of a direct solve: those of these products and solvers elsewhere.
"""
import numpy as np
import pytest
import scipy.sparse as sp
import scipy.sparse.linalg as spla

import oracle as O
from neopz_amd import _lib as L
from neopz_amd import mesh as M
from neopz_amd import problems as P
from neopz_amd.analysis import Context, TPZLinearAnalysis, TPZStepSolver

pytestmark = pytest.mark.gpu


def _mesh(material):
    """The faces' middle connects replaced by one connect of size 0 on every
    second face."""
    pb = P.Problem(material=material, dim=3, p=2, nx=4, ny=3, nz=2, E=1.0, nu=0.3, force_kind=P.FORCE_CONST,
                   force_const=(0.3, -1.0, 0.2), bc_type=[0, -1, 0, -1, -1, -1])
    pb.el_coef = np.exp(np.random.default_rng(1).standard_normal(pb.nvol))
    md = M.build(pb)
    n = md["nconn"]
    bc = np.asarray(md["bc_conn"]).reshape(-1, 9).copy()
    bc[::2, 8] = n
    md["bc_conn"], md["nconn"] = bc, n + 1
    md["blk_pos"] = np.append(md["blk_pos"], md["neq"]).astype(np.int64)
    md["blk_size"] = np.append(md["blk_size"], 0).astype(np.int32)
    md["conn_order"] = np.full(n + 1, 2)  # (for the oracle)
    md["conn_order"][np.asarray(md["vol_conn"]).reshape(-1, 27)[:, :8]] = 1
    return pb, md


@pytest.mark.parametrize("material", [P.ELAST3D, P.DARCY])
def test_products_and_solves(material):
    pb, md = _mesh(material)
    o = O.Oracle(pb, mesh=md)
    ia, ja = o.pattern()
    a, rhs = o.assemble()
    U = sp.csr_matrix((a, ja, ia), shape=(o.neq, o.neq))
    F = (U + sp.triu(U, 1).T).tocsr()
    ctx = Context(0)
    an = TPZLinearAnalysis(md, False, ctx=ctx)
    an.Assemble()
    x = np.random.default_rng(3).standard_normal(o.neq)
    assert np.all(np.abs(an.K.MultAdd(x, None, 1.0, 0.0) - F @ x) <= 1e-13 * (abs(F) @ np.abs(x)))
    s = 1.0 / np.sqrt(U.diagonal())
    x = x.astype(np.float32).astype(np.float64)
    z = np.zeros_like(x)
    L.check(ctx.lib.pzg_scaled_apply(ctx.h, L.INNER_MATFREE, L.ptr(x, L.dp), L.ptr(z, L.dp)))
    bound = s * (abs(F) @ np.abs(s * x))
    assert np.linalg.norm(z - s * (F @ (s * x))) <= 30 * 2.0 ** -24 * np.linalg.norm(bound)
    ref = spla.spsolve(F.tocsc(), rhs)
    st = TPZStepSolver()
    an.SetSolver(st)
    st.SetCG(20000, TPZStepSolver.jacobi(), 1e-11, 0)
    assert np.linalg.norm(an.Solve() - ref) <= 1e-8 * np.linalg.norm(ref)
    st.SetMixedFCG(20000, 1e-8)
    assert np.linalg.norm(an.Solve() - ref) <= 1e-5 * np.linalg.norm(ref)
    assert not st.info["fallback"]
    ctx.close()
