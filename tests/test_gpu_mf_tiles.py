"""FP32 matrix-free product on lattices of identical p = 2 boxes (tiles of 4^3
cells) against the oracle's assembled matrix in FP64, and the multigrid cycle
whose level 0 runs inside it against the cycle over the stored block CSR.

Bars (written here, checked below):
  * product: |z - S x|_2 <= 30 * 2^-24 * | |S| |x| |_2: a value passes the two
    scalings, three transforms of two roundings on each side, a product of at
    most four coefficients, five terms and the sum over eight elements, about
    30 roundings in a row, each relative to terms of S x;
  * cycle: 2e-4 relative, the bar of the cycle against its FP64 model.

Element counts: one cell, less than a tile, whole tiles, one cell more than a
tile, different counts (and so edge lengths) per direction, more tiles than
workgroups of the tile kernel.
"""
import ctypes as C

import numpy as np
import pytest
import scipy.sparse as sp

import oracle as O
from neopz_amd import _lib as L
from neopz_amd import problems as P
from neopz_amd.analysis import Context, TPZLinearAnalysis

pytestmark = pytest.mark.gpu


def _elast(nx, ny, nz, faces, seed=0):
    pb = P.Problem(material=P.ELAST3D, dim=3, p=2, nx=nx, ny=ny, nz=nz, E=1.0, nu=0.3,
                   force_kind=P.FORCE_CONST, force_const=(0.3, -1.0, 0.2),
                   bc_type=[0 if f in faces else -1 for f in range(6)])
    pb.el_coef = np.exp(np.random.default_rng(seed).standard_normal(pb.nvol))
    return pb


def _scaled_apply(ctx, op, x):
    z = np.zeros_like(x)
    L.check(ctx.lib.pzg_scaled_apply(ctx.h, op, L.ptr(x, L.dp), L.ptr(z, L.dp)))
    return z


@pytest.mark.parametrize("renumber", [False, True])
@pytest.mark.parametrize("n,faces", [((1, 1, 1), (4,)), ((3, 2, 4), range(6)), ((4, 4, 4), (0, 2)),
                                     ((5, 9, 4), (1, 3, 5)), ((1, 8, 13), ())])
def test_product_matches_oracle(n, faces, renumber):
    pb = _elast(*n, faces, seed=sum(n))
    o = O.Oracle(pb)
    ia, ja = o.pattern()
    a, _ = o.assemble()
    ctx = Context(0)
    an = TPZLinearAnalysis(pb, renumber, ctx=ctx)
    an.Assemble()
    if renumber:  # the equations are the context's
        ia, ja, a = an.K.IA(), an.K.JA(), an.K.A()
    U = sp.csr_matrix((a, ja, ia), shape=(o.neq, o.neq))
    F = (U + sp.triu(U, 1).T).tocsr()
    s = 1.0 / np.sqrt(U.diagonal())
    rng = np.random.default_rng(3)
    for x in (rng.standard_normal(o.neq), 1.0 / s, np.where(rng.random(o.neq) < 0.02, 1.0, 0.0)):
        x = x.astype(np.float32).astype(np.float64)
        z = _scaled_apply(ctx, L.INNER_MATFREE, x)
        ref = s * (F @ (s * x))
        bound = s * (abs(F) @ np.abs(s * x))
        assert np.linalg.norm(z - ref) <= 30 * 2.0 ** -24 * np.linalg.norm(bound)
    ctx.close()


def test_large_lattice_matches_block_csr():
    """44 x 40 x 43 cells: 1210 tiles, more than the tile kernel's workgroups."""
    pb = _elast(44, 40, 43, (0, 5), 7)
    ctx = Context(0)
    an = TPZLinearAnalysis(pb, False, ctx=ctx)
    an.Assemble()
    x = np.random.default_rng(8).standard_normal(an.K.neq)
    # zero on the Dirichlet faces (their rows would hide all others in a norm)
    md = an.mesh
    bpos = md["blk_pos"][np.unique(md["bc_conn"])]
    x[(bpos[:, None] + np.arange(3)).ravel()] = 0.0
    z = [_scaled_apply(ctx, op, x) for op in (L.INNER_BSR, L.INNER_MATFREE)]
    free = np.ones(len(x), bool)
    free[(bpos[:, None] + np.arange(3)).ravel()] = False
    # the stored operator's rounding (256 terms a row) and the tiles'; the rows'
    # sums of |terms| are at most 6 times their root mean square here
    d = np.linalg.norm((z[0] - z[1])[free])
    assert d <= 6 * 60 * 2.0 ** -24 * np.linalg.norm(z[0][free])
    ctx.close()


@pytest.mark.parametrize("degree", [1, 2, 3])
@pytest.mark.parametrize("n", [(4, 4, 4), (6, 10, 4)])
def test_cycle_matches_stored_operator(n, degree):
    pb = _elast(*n, (0, 4), seed=degree)
    ctx = Context(0)
    an = TPZLinearAnalysis(pb, False, ctx=ctx)
    an.Assemble()
    r = np.random.default_rng(9).standard_normal(an.K.neq)
    zs = []
    for op in (L.INNER_BSR, L.INNER_MATFREE):
        z = np.zeros_like(r)
        nlev = C.c_int32(0)
        dims, lmax = np.zeros(48, dtype=np.int32), np.zeros(16)
        L.check(ctx.lib.pzg_mg_apply(ctx.h, op, degree, 0.0, L.ptr(r, L.dp), L.ptr(z, L.dp), C.byref(nlev),
                                     L.ptr(dims, L.i32p), L.ptr(lmax, L.dp)))
        zs.append(z)
    assert np.linalg.norm(zs[0] - zs[1]) <= 2e-4 * np.linalg.norm(zs[0])
    ctx.close()
