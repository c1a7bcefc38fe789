"""Error of the tiled FP32 product against FP64 beside the element-major
product's on the same lattice (PZG_NO_BLKASM leaves the lattice to it).

Bar: at random vectors, zero on the clamped face, the tiles' relative error is
not above the element-major product's (mean of four vectors; measured 0.75 to
0.97 of it).  Counts: cubes whose edge is no power of two, so that a factor of
the edge rounded into the rows' constants would show (1.01 to 1.12), and a box.
"""
import os

import numpy as np
import pytest

from neopz_amd import _lib as L
from neopz_amd import mesh as M
from neopz_amd import problems as P
from neopz_amd.analysis import Context, TPZLinearAnalysis

pytestmark = pytest.mark.gpu


def _error(n, element_major):
    pb = P.Problem(material=P.ELAST3D, dim=3, p=2, nx=n[0], ny=n[1], nz=n[2], E=1.0, nu=0.3,
                   force_kind=P.FORCE_CONST, force_const=(1.0, 0.0, 0.0), bc_type=[-1, -1, -1, -1, 0, -1])
    pb.el_coef = np.exp(np.random.default_rng(2).standard_normal(pb.nvol))
    md = M.build(pb)
    ctx = Context(0)
    os.environ["PZG_NO_BLKASM"] = "1" if element_major else "0"
    try:
        an = TPZLinearAnalysis(md, False, ctx=ctx)
        an.Assemble()
        s = 1.0 / np.sqrt(an.K.A()[an.K.IA()[:-1]])
        free = np.ones(md["neq"], bool)
        free[(md["blk_pos"][np.unique(md["bc_conn"])][:, None] + np.arange(3)).ravel()] = False
        out = []
        for seed in range(4):
            x = np.where(free, np.random.default_rng(seed).standard_normal(md["neq"]), 0.0)
            x = x.astype(np.float32).astype(np.float64)
            z = np.zeros_like(x)
            L.check(ctx.lib.pzg_scaled_apply(ctx.h, L.INNER_MATFREE, L.ptr(x, L.dp), L.ptr(z, L.dp)))
            ref = s * an.K.Multiply(s * x)
            out.append(np.linalg.norm((z - ref)[free]) / np.linalg.norm(ref[free]))
    finally:
        del os.environ["PZG_NO_BLKASM"]
        ctx.close()
    return np.mean(out)


@pytest.mark.parametrize("n", [(5, 5, 5), (10, 10, 10), (15, 15, 15), (21, 21, 21), (4, 6, 8)])
def test_error_not_above_element_major(n):
    tiles, elements = _error(n, False), _error(n, True)
    print(f"[gpu] {n}: tiles {tiles:.3e}, element-major {elements:.3e}", flush=True)
    assert tiles <= elements
