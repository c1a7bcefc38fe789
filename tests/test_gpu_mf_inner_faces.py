"""Dirichlet faces inside the lattice: FP32 matrix-free product on lattices of
identical p = 2 boxes against the oracle's assembled matrix, and solves on it.

Bars: the product's is that of the tiles without such faces (30 roundings in a
row relative to |S| |x|); the solution within 1e-5 of a direct solve of the
oracle's system, the bar of the other mixed solves; no fallback.  Planes: inside
a tile of 4^3 cells, on the face between two tiles, both, a single face.
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

_EDGE = {frozenset(e): 8 + k for k, e in enumerate(M._HEX_EDGE)}


def _mesh(n, planes, single=False):
    """Clamped at x = 0 and, by further boundary elements of the same kind, on
    the planes x = i cells."""
    nx, ny, nz = n
    pb = P.Problem(material=P.ELAST3D, dim=3, p=2, nx=nx, ny=ny, nz=nz, E=1.0, nu=0.3, force_kind=P.FORCE_CONST,
                   force_const=(0.3, -1.0, 0.2), bc_type=[0, -1, -1, -1, -1, -1])
    pb.el_coef = np.exp(np.random.default_rng(nx).standard_normal(pb.nvol))
    md = M.build(pb)
    vn, vc = np.asarray(md["vol_nodes"]).reshape(-1, 8), np.asarray(md["vol_conn"]).reshape(-1, 27)
    side = M._HEX_FACE.index((0, 3, 7, 4))  # the side x = 0 of an element
    f = M._HEX_FACE[side]
    local = list(f) + [_EDGE[frozenset((f[k], f[(k + 1) % 4]))] for k in range(4)] + [20 + side]
    els = np.concatenate([np.flatnonzero(np.arange(pb.nvol) % nx == i) for i in planes])
    if single:
        els = els[len(els) // 2:][:1]
    md["bc_nodes"] = np.ascontiguousarray(np.concatenate([md["bc_nodes"], vn[els][:, f]]))
    md["bc_conn"] = np.ascontiguousarray(np.concatenate([md["bc_conn"], vc[els][:, local]]))
    md["bc_id"] = np.concatenate([md["bc_id"], np.zeros(len(els), np.int32)]).astype(np.int32)
    md["conn_order"] = np.full(md["nconn"], 2)  # (for the oracle)
    md["conn_order"][vc[:, :8]] = 1
    return pb, md


def _scaled_apply(ctx, x):
    z = np.zeros_like(x)
    L.check(ctx.lib.pzg_scaled_apply(ctx.h, L.INNER_MATFREE, L.ptr(x, L.dp), L.ptr(z, L.dp)))
    return z


@pytest.mark.parametrize("n,planes,single", [((4, 4, 4), (1,), False), ((8, 4, 4), (4,), False),
                                             ((8, 5, 4), (3, 4), False), ((6, 4, 4), (2,), True)])
def test_product_and_solve(n, planes, single):
    pb, md = _mesh(n, planes, single)
    o = O.Oracle(pb, mesh=md)
    ia, ja = o.pattern()
    a, rhs = o.assemble()
    U = sp.csr_matrix((a, ja, ia), shape=(o.neq, o.neq))
    F = (U + sp.triu(U, 1).T).tocsr()
    ctx = Context(0)
    an = TPZLinearAnalysis(md, False, ctx=ctx)
    an.Assemble()
    s = 1.0 / np.sqrt(U.diagonal())
    rng = np.random.default_rng(3)
    for x in (rng.standard_normal(o.neq), 1.0 / s):
        x = x.astype(np.float32).astype(np.float64)
        z = _scaled_apply(ctx, x)
        ref = s * (F @ (s * x))
        bound = s * (abs(F) @ np.abs(s * x))
        assert np.linalg.norm(z - ref) <= 30 * 2.0 ** -24 * np.linalg.norm(bound)
    x = spla.spsolve(F.tocsc(), rhs)
    for precond in (L.PRECOND_BLOCK_JACOBI, L.PRECOND_MULTIGRID):
        st = TPZStepSolver()
        st.SetMixedFCG(20000, 1e-8, precond=precond)
        an.SetSolver(st)
        u = an.Solve()
        assert st.info["converged"] and not st.info["fallback"]
        assert np.linalg.norm(u - x) <= 1e-5 * np.linalg.norm(x)
    ctx.close()
