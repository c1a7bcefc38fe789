"""Solves of several meshes in one context, graphs on: the batch that a context
keeps from one solve to the next is used only for the system it was captured on.

Every mesh is solved once in a context of its own; then all of them, in turn
and back, in one context.  Bar: the same iterations and the same solution bit
for bit (same kernels in the same order), no fallback.  The meshes have equal
counts of elements, equations and Dirichlet faces where they can: other edge
lengths, permuted counts, moved nodes (no lattice), the faces on one side and
on two.
"""
import numpy as np
import pytest

from neopz_amd import mesh as M
from neopz_amd import problems as P
from neopz_amd.analysis import Context, TPZLinearAnalysis, TPZStepSolver

pytestmark = pytest.mark.gpu


def _lattice(nx, ny, nz, faces=(0,), keep=None, stretch=(1.0, 1.0, 1.0), warp=0.0, E=1.0):
    """keep: the Dirichlet faces per side that stay."""
    pb = P.Problem(material=P.ELAST3D, dim=3, p=2, nx=nx, ny=ny, nz=nz, E=E, nu=0.3, force_kind=P.FORCE_CONST,
                   force_const=(0.3, -1.0, 0.2), bc_type=[0 if f in faces else -1 for f in range(6)])
    md = M.build(pb)
    if keep is not None:
        ids = np.asarray(md["bc_id"])
        on = np.concatenate([np.flatnonzero(ids == f)[:keep] for f in np.unique(ids)])
        for k in ("bc_nodes", "bc_conn", "bc_id"):
            md[k] = np.ascontiguousarray(md[k][on])
    x = np.asarray(md["xyz"]).reshape(-1, 3) * np.array(stretch)
    x = x + warp * np.sin(np.pi * x[:, [1, 2, 0]])
    md["xyz"] = np.ascontiguousarray(x.ravel())
    return md


MESHES = {
    "box": lambda: _lattice(4, 6, 8),
    "other_edges": lambda: _lattice(4, 6, 8, stretch=(1.0, 2.0, 0.5)),
    "permuted": lambda: _lattice(4, 8, 6),
    "moved_nodes": lambda: _lattice(4, 6, 8, warp=0.03),
    "other_modulus": lambda: _lattice(4, 6, 8, E=3.0),
    "half_a_side": lambda: _lattice(4, 6, 8, keep=24),
    "two_half_sides": lambda: _lattice(4, 6, 8, faces=(0, 1), keep=12),
    "larger": lambda: _lattice(9, 5, 8, faces=(0, 3)),
}
ORDER = ["box", "other_edges", "box", "permuted", "moved_nodes", "other_modulus", "half_a_side", "two_half_sides",
         "larger", "half_a_side", "box"]


def _solve(ctx, md, kind):
    an = TPZLinearAnalysis(md, False, ctx=ctx)
    st = TPZStepSolver()
    an.SetSolver(st)
    if kind == "mixed":
        st.SetMixedFCG(20000, 1e-8)
    else:
        pre = an.BuildPreconditioner(an.EBlockJacobi, True) if kind == "pcg_block" else TPZStepSolver.jacobi()
        st.SetCG(20000, pre, 1e-10, 0)
    assert st.use_graph
    out = []
    for _ in range(2):  # the second solve replays the first one's graph
        an.Assemble()
        u = an.Solve()
        out.append((st.info["iterations"], st.info["fallback"], st.info["converged"], u))
    return out


@pytest.mark.parametrize("kind", ["mixed", "pcg", "pcg_block"])
def test_meshes_in_turn_equal_fresh_contexts(kind):
    mds = {k: f() for k, f in MESHES.items()}
    ref = {}
    for k, md in mds.items():
        ctx = Context(0)
        ref[k] = _solve(ctx, md, kind)[0]
        ctx.close()
        assert ref[k][2] and not ref[k][1], k
    ctx = Context(0)
    for k in ORDER:
        print(f"[gpu] {kind} {k}", flush=True)
        for it, fallback, converged, u in _solve(ctx, mds[k], kind):
            assert (it, fallback, converged) == ref[k][:3], k
            assert np.array_equal(u, ref[k][3]), k
    ctx.close()
