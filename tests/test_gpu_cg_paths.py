"""FP64 CG on its three device paths (one workgroup in LDS, direction inside the
product, direction apart) against the oracle's CG, around the sizes where the
path changes.

Bars: the iterates after 1, 2, 7 and 20 steps within 1e-8 of the oracle's CG
(rounding differences grow with the steps, from 1e-15 times the ratio of the
penalty rows to the others); the converged solution within 1e-8 of the oracle's.
The number of steps to 1e-11 is not compared: the penalty of 6.7e16 on the
boundary rows makes the last digits of the recursion depend on the order of the
sums (377 against 416 steps on 91^2 elements).  The iteration limit is kept on
every path (the one-workgroup kernel resumes after its own 2000 iterations).
"""
import numpy as np
import pytest

import oracle as O
from neopz_amd import _lib as L
from neopz_amd import problems as P
from neopz_amd.analysis import Context, TPZLinearAnalysis, TPZStepSolver, TPZSYsmpMatrixHIP

pytestmark = pytest.mark.gpu

CASES = {
    "lds_one_element": lambda: P.poisson2d(n=1, p=2, seed=1),
    "lds_largest": lambda: P.poisson2d(n=13, p=2, seed=1),       # 11,025 entries: 149 KB
    "merged_smallest": lambda: P.poisson2d(n=14, p=2, seed=1),   # 12,769 entries: past the LDS
    "merged_largest": lambda: P.poisson2d(n=90, p=2, seed=1),    # 519,841 entries
    "apart_smallest": lambda: P.poisson2d(n=91, p=2, seed=1),    # 531,441 entries
    "lds_blocks": lambda: P.elasticity3d(n=3, p=1, seed=2),      # 1000 blocks of 9
    "merged_blocks": lambda: P.elasticity3d(n=6, p=1, seed=2),
}


@pytest.mark.parametrize("precond", ["jacobi", "block"])
@pytest.mark.parametrize("name", list(CASES))
def test_pcg64_paths_match_oracle(name, precond):
    pb = CASES[name]()
    o = O.Oracle(pb)
    ia, ja = o.pattern()
    a, rhs = o.assemble()
    ctx = Context(0)
    an = TPZLinearAnalysis(pb, False, ctx=ctx)
    st = TPZStepSolver()
    an.SetSolver(st)
    pre = TPZStepSolver.jacobi() if precond == "jacobi" else an.BuildPreconditioner(an.EBlockJacobi, True)
    st.SetCG(20000, pre, 1e-11, 0)
    for graph in (True, False, True):
        st.use_graph = graph
        an.Assemble()
        u = an.Solve()
        ref = (O.pcg(ia, ja, a, rhs, maxit=20000, tol=1e-11, wasted_spmv=False) if precond == "jacobi" else
               O.pcg_block(ia, ja, a, rhs, np.full(o.neq // pb.nstate, pb.nstate), maxit=20000, tol=1e-11))
        assert st.info["converged"]
        assert np.linalg.norm(u - ref["x"]) <= 1e-8 * np.linalg.norm(ref["x"])
    # the iteration limit, odd and even
    for maxit in (1, 2, 7, 20):
        st.SetCG(maxit, pre, 1e-30, 0)
        u = an.Solve()
        ref = (O.pcg(ia, ja, a, rhs, maxit=maxit, tol=1e-30, wasted_spmv=False) if precond == "jacobi" else
               O.pcg_block(ia, ja, a, rhs, np.full(o.neq // pb.nstate, pb.nstate), maxit=maxit, tol=1e-30))
        if name != "lds_one_element":  # (nine equations, all of them penalized: exact after one step)
            assert st.info["iterations"] == maxit and not st.info["converged"]
            assert np.linalg.norm(u - ref["x"]) <= 1e-8 * np.linalg.norm(ref["x"])
    ctx.close()


def test_one_workgroup_resumes():
    """Ill-conditioned tridiagonal system whose CG needs more iterations than
    one launch of the one-workgroup kernel runs."""
    n = 800
    d = 10.0 ** np.linspace(0, 7, n)
    ia = np.arange(n + 1) * 2
    ia[-1] = 2 * n - 1
    ja = np.empty(2 * n - 1, np.int64)
    a = np.empty(2 * n - 1)
    ja[0::2], a[0::2] = np.arange(n), 2.0 + 1e-5 * d / d[-1]
    ja[1::2], a[1::2] = np.arange(1, n), -1.0
    f = np.random.default_rng(3).standard_normal(n)
    ctx = Context(0)
    K = TPZSYsmpMatrixHIP(ctx, n)
    K.SetData(ia, ja, a, f)
    st = TPZStepSolver(K)
    st.SetCG(5000, TPZStepSolver.jacobi(K), 0.0, 0)  # never met: every iteration is run
    st.Solve(f)
    assert st.info["iterations"] == 5000
    st.SetCG(5000, TPZStepSolver.jacobi(K), 1e-12, 0)
    u = st.Solve(f)
    assert st.info["converged"]
    import scipy.sparse as sp
    import scipy.sparse.linalg as spla
    U = sp.csr_matrix((a, ja, ia), shape=(n, n))
    x = spla.spsolve((U + sp.triu(U, 1).T).tocsc(), f)
    # condition number at most 4 / (smallest eigenvalue of the Laplacian, 1.5e-5): 1e-12 * 2.6e5
    assert np.linalg.norm(u - x) <= 1e-6 * np.linalg.norm(x)
    ctx.close()
