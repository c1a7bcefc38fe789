"""What a user of this framework has it do, as timed cases.

Every case goes through the public classes of ``neopz_amd``: assemble and
solve (``TPZLinearAnalysis``), products with the assembled matrix
(``TPZSYsmpMatrixHIP.MultAdd``), error norms (``PostProcessError``) and the
training of the learned preconditioner (``train_on_seeds``).  A solve case is
one step of a parameter study on a fixed mesh: a new coefficient field (where
the material has one), an assembly and a solve whose solution comes back to the host.
The mesh, the device context, the pattern and trained weights are what such a
program keeps between the steps.

``exact`` restates the quadrilateral and hexahedral problems on uniform
lattices in plain torch, in 64 bits: element matrices as products of
one-dimensional ones, conjugate gradients over the elements.
"""
import numpy as np
import torch

from neopz_amd import _lib as L
from neopz_amd import mesh as M
from neopz_amd import problems as P
from neopz_amd.analysis import (Context, TLaplaceExample1, TPZLinearAnalysis, TPZSSpStructMatrixHIP,
                                TPZStepSolver)
from neopz_amd.learned import LearnedSmoother, train_on_seeds


def listed():
    return [
        # the smallest problem a user runs (the smoke test): launches and latency only
        dict(name="poisson_8_pcg", kind="poisson2d", n=8, p=2, solver="pcg", tol=1e-12),
        # 2D Poisson, 64 x 64, p = 2, FP64 Jacobi-PCG to 1e-10: the plain reference method
        dict(name="poisson_64_pcg", kind="poisson2d", n=64, p=2, solver="pcg", tol=1e-10),
        # 2D Darcy flow, a new permeability field on the 256 x 256 mesh, multigrid FCG
        dict(name="darcy_256_p1_mg", kind="darcy2d", n=256, p=1, solver="mg", tol=1e-8),
        # the same at p = 2 with an odd number of elements (the lattice does not halve)
        dict(name="darcy_255_p2_mg", kind="darcy2d", n=255, p=2, solver="mg", tol=1e-8),
        # 3D elasticity, plain FP64 PCG with the connect-block Jacobi (BuildPreconditioner)
        dict(name="elast_24_pcg_block", kind="elast3d", n=24, p=2, load="traction", solver="pcg_block", tol=1e-10),
        # 3D elasticity on an hp mesh (orders 1 and 2): stored FP32 operator, block Jacobi
        dict(name="elast_hp_21_bj", kind="elast_hp", n=21, p=2, load="traction", solver="bj", tol=1e-8),
        # 3D elasticity 48^3, i.i.d. modulus, traction: multigrid FCG without a trained smoother
        dict(name="elast_48_mg", kind="elast3d", n=48, p=2, load="traction", solver="mg", tol=1e-8),
        # the headline workload: 64^3, random-field modulus, body load, learned smoother
        dict(name="elast_64_learned", kind="elast3d", n=64, p=2, load="body", solver="learned", tol=1e-8),
        # hp Darcy flow on 6 x 32^3 tetrahedra, orders 1 to 5, connect-block Jacobi FCG
        dict(name="tet_32_hp5_bj", kind="tet", n=32, p=5, solver="bj", tol=1e-8),
        # training of the learned smoother on one field (assembly, pairs, fit, Adam steps)
        dict(name="train_12", kind="train", n=12, p=2, steps=100),
        # error norms of a solution on hp tetrahedra against a manufactured one
        dict(name="errors_tet_24", kind="errors_tet", n=24, p=5, order=14),
        # product of the assembled matrix with a vector of the caller
        dict(name="matvec_48", kind="matvec", n=48, p=2, load="body"),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    kind = rng.choice(["poisson2d", "poisson2d", "darcy2d", "darcy2d", "elast_pcg", "elast_hp", "elast_mg",
                       "elast_learned", "tet", "train", "errors_tet", "errors_quad", "matvec"])
    if kind == "poisson2d":
        return dict(kind=kind, n=_log_int(rng, 6, 120), p=rng.choice([1, 2]), solver="pcg",
                    tol=rng.choice([1e-10, 1e-12]))
    if kind == "darcy2d":
        return dict(kind=kind, n=_log_int(rng, 40, 400), p=rng.choice([1, 2]), solver="mg", tol=1e-8)
    if kind == "elast_pcg":
        return dict(kind="elast3d", n=_log_int(rng, 3, 28), p=rng.choice([1, 2]), load="traction",
                    solver=rng.choice(["pcg", "pcg_block"]), tol=1e-10)
    if kind == "elast_hp":
        return dict(kind=kind, n=_log_int(rng, 6, 26), p=2, load="traction", solver="bj", tol=1e-8)
    if kind == "elast_mg":
        return dict(kind="elast3d", n=_log_int(rng, 8, 56), p=2, load=rng.choice(["traction", "body"]),
                    solver="mg", tol=1e-8)
    if kind == "elast_learned":
        return dict(kind="elast3d", n=_log_int(rng, 12, 60), p=2, load=rng.choice(["traction", "body"]),
                    solver="learned", tol=1e-8)
    if kind == "tet":
        return dict(kind=kind, n=_log_int(rng, 4, 30), p=rng.randint(2, 5), solver="bj", tol=1e-8)
    if kind == "train":
        return dict(kind=kind, n=_log_int(rng, 5, 14), p=2, steps=_log_int(rng, 20, 150))
    if kind == "errors_tet":
        return dict(kind=kind, n=_log_int(rng, 3, 26), p=rng.randint(2, 5), order=rng.randint(4, 14))
    if kind == "errors_quad":
        return dict(kind=kind, n=_log_int(rng, 16, 512), p=rng.choice([1, 2]), order=rng.randint(4, 14))
    return dict(kind="matvec", n=_log_int(rng, 6, 48), p=2, load=rng.choice(["traction", "body"]))


# ---- the problems -------------------------------------------------------------
def _orders(n, p, nvol):
    """Orders of an hp mesh: part of the mesh, the same for every coefficient field on it."""
    return np.random.default_rng(100 * n + p).integers(1, p + 1, nvol).astype(np.int32)


def _problem(case, seed):
    kind, n, p = case["kind"], case["n"], case["p"]
    if kind in ("poisson2d", "errors_quad"):
        return P.poisson2d(n=n, p=p, seed=seed)
    if kind == "darcy2d":
        return P.darcy2d(n=n, p=p, seed=seed)
    if kind in ("tet", "errors_tet"):
        pb = P.darcy3d_tet(n=n, pmax=p, seed=seed)
        pb.el_porder = _orders(n, p, pb.nvol)
        return pb
    if kind == "train":
        return P.elasticity3d(n=n, p=p, seed=seed, field_kind="grf", corr_len=0.1 * 64 / n, load="body")
    pb = P.elasticity3d(n=n, p=p, seed=seed, field_kind="grf" if case["load"] == "body" else "iid",
                        load=case["load"])
    if kind == "elast_hp":
        pb.el_porder = _orders(n, p, pb.nvol)
    return pb


def _trained(case):
    """Weights of the learned smoother from two seeded 8^3 systems of the same family."""
    def make(seed):
        return _problem(dict(case, n=8), seed)
    ctx = Context(0)
    sm = TPZSSpStructMatrixHIP(ctx, M.build(make(1000)))
    K = sm.Create()
    sm.Assemble(K)
    ls, _, _ = train_on_seeds(ctx, sm, K, lambda s: make(s).el_coef, [1001, 1002], nrhs=4, steps=40, lr=3e-3)
    w = ls.get_weights()
    ctx.close()
    return w


def _vector(seed, n):
    return np.random.default_rng(seed + 5).standard_normal(n)


def prepare(case, seed):
    pb = _problem(case, seed)
    md = M.build(pb)
    ctx = Context(0)
    kind = case["kind"]
    if kind in ("errors_tet", "errors_quad"):
        an = TPZLinearAnalysis(md, False, ctx=ctx)
        an.LoadSolution(_vector(seed, md["neq"]))
        an.SetExact(TLaplaceExample1(TLaplaceExample1.ESinSin), case["order"])
        return dict(kind=kind, an=an)
    sm = TPZSSpStructMatrixHIP(ctx, md)
    K = sm.Create()
    if kind == "matvec":
        sm.Assemble(K)
        return dict(kind=kind, K=K, sm=sm, x=_vector(seed, md["neq"]))
    coef = md["vol_coef"]
    if kind == "train":
        return dict(kind=kind, ctx=ctx, sm=sm, K=K, coef=coef, steps=case["steps"])
    an = TPZLinearAnalysis(md, False, ctx=ctx)
    an.fStructMatrix, an.K = sm, K
    st = TPZStepSolver(K)
    an.SetSolver(st)
    solver = case["solver"]
    if solver in ("pcg", "pcg_block"):
        pre = TPZStepSolver.jacobi() if solver == "pcg" else an.BuildPreconditioner(an.EBlockJacobi, True)
        st.SetCG(200000, pre, case["tol"], 0)
        st.check_every = 100
    else:
        st.SetMixedFCG(200000, case["tol"], precond={"bj": L.PRECOND_BLOCK_JACOBI, "mg": L.PRECOND_MULTIGRID,
                                                     "learned": L.PRECOND_LEARNED}[solver])
        st.check_every = 100 if solver == "bj" else 0
    if solver == "learned":
        ls = LearnedSmoother(ctx)
        ls.setup(seed=0)
        ls.set_weights(_trained(case))
    return dict(kind="solve", ctx=ctx, an=an, coef=coef)


def run(state):
    kind = state["kind"]
    if kind == "matvec":
        return state["K"].MultAdd(state["x"], None, 1.0, 0.0)
    if kind == "train":
        coef = state["coef"]
        ls, first, last = train_on_seeds(state["ctx"], state["sm"], state["K"], lambda s: coef, [1], nrhs=4,
                                         steps=state["steps"], lr=3e-3)
        return dict(first=first, last=last, weights=ls.get_weights())
    if kind in ("errors_tet", "errors_quad"):
        an = state["an"]
        totals = an.PostProcessError(store_error=True)
        return dict(totals=totals, elements=an.ElementSolution())
    ctx, an, coef = state["ctx"], state["an"], state["coef"]
    if coef is not None:
        L.check(ctx.lib.pzg_mesh_set_coef(ctx.h, L.ptr(coef, L.dp)))
    an.Assemble()
    return an.Solve()


def _sizes(case):
    """(elements, equations, stored entries of the upper triangle)."""
    kind, n, p = case["kind"], case["n"], case["p"]
    dim = 2 if kind in ("poisson2d", "darcy2d", "errors_quad") else 3
    if kind in ("tet", "errors_tet"):
        # orders uniform in 1..p, the lowest on shared sides; unknowns
        # per cube and stored entries per row as counted on such meshes
        per, row = {2: (1.7, 7), 3: (4.3, 9), 4: (10.3, 12), 5: (20.6, 16)}[p]
        return 6 * n ** 3, int(per * n ** 3), int(per * n ** 3 * row)
    ns = 3 if dim == 3 else 1
    nb = (p * n + 1) ** dim
    full = (8 * n + 1 if p == 2 else 3 * n + 1) ** dim
    if kind == "elast_hp":  # a side keeps its function when none of its elements has order 1
        nb, full = int(0.31 * nb), int(0.13 * full)
    return n ** dim, nb * ns, (full * ns * ns + nb * ns) // 2


def work(case):
    nel, neq, nnz = _sizes(case)
    kind = case["kind"]
    if kind == "matvec":
        return {"bytes": 8 * (nnz + 2 * neq), "flops": 4 * nnz}
    if kind in ("errors_tet", "errors_quad"):
        nerr = 6 if kind == "errors_tet" else 3
        npts = 512 if kind == "errors_tet" else 64
        return {"bytes": 8 * (neq + nerr * nel), "flops": 40 * npts * nel}
    if kind == "train":  # the pairs read by every step, and the network on the element graph
        return {"bytes": case["steps"] * nel * 4 * 81 * 4 * 2,
                "flops": nel * (case["steps"] * 3 * 3 * 2 * 2 * 32 * 32 + 4 * 4 * 81 * 81)}
    # coefficients in, the stored matrix written and read for the FP64 residual, solution out
    return {"bytes": 8 * (nel + 2 * nnz + 2 * neq), "flops": 4 * nnz}


def tolerance(case):
    """About four times what another order of sums was seen to change over 45 drawn cases."""
    if case["kind"] == "train":  # Adam steps follow the sign of small FP32 gradients: 6e-4 after 140 steps
        return {"rel": 2.5e-3, "max": 2e-2}
    if "solver" not in case:  # FP64 sums: 1e-14, largest entry 5e-14
        return {"rel": 4e-14, "max": 1e-12}
    if case["solver"] in ("pcg", "pcg_block"):  # stopped at 1e-10: 1e-11 from the exact solution
        return {"rel": 1e-10, "max": 1e-8}
    return {"rel": 2e-8, "max": 1e-6}  # stopped at 1e-8: 3e-9 from the exact solution


# ---- the same in plain torch, 64 bits -------------------------------------------
# side -> (function per direction: 0 and 1 the linear ones, 2 the bubble), in
# the order of the mesh's element connect lists
_QUAD = [(0, 0), (1, 0), (1, 1), (0, 1), (2, 0), (1, 2), (2, 1), (0, 2), (2, 2)]
_HEX = ([(0, 0, 0), (1, 0, 0), (1, 1, 0), (0, 1, 0), (0, 0, 1), (1, 0, 1), (1, 1, 1), (0, 1, 1),
         (2, 0, 0), (1, 2, 0), (2, 1, 0), (0, 2, 0), (0, 0, 2), (1, 0, 2), (1, 1, 2), (0, 1, 2),
         (2, 0, 1), (1, 2, 1), (2, 1, 1), (0, 2, 1), (2, 2, 0), (2, 0, 2), (1, 2, 2), (2, 1, 2),
         (0, 2, 2), (2, 2, 1), (2, 2, 2)])


def _basis1d(x):
    """Values and derivatives [3, q] on [0, 1] of 1-x, x, 4x(1-x)."""
    return np.stack([1 - x, x, 4 * x * (1 - x)]), np.stack([-1 + 0 * x, 1 + 0 * x, 4 - 8 * x])


def _gauss(q):
    x, w = np.polynomial.legendre.leggauss(q)
    return (x + 1) / 2, w / 2


def _tensor1d(h):
    """M[d][e][i, j] = integral of the d-th and e-th derivatives over an interval of length h."""
    x, w = _gauss(4)
    v, g = _basis1d(x)
    f = [v, g / h]
    return [[np.einsum("iq,jq,q->ij", f[d], f[e], w) * h for e in (0, 1)] for d in (0, 1)]


def _grams(sides, h):
    """G[a][b][i, j] = integral of d_a phi_i d_b phi_j over a cell with edges h."""
    t, dim = _tensor1d(h), len(sides[0])
    s = np.array(sides)
    out = []
    for a in range(dim):
        row = []
        for b in range(dim):
            g = np.ones((len(s), len(s)))
            for d in range(dim):
                g = g * t[int(d == a)][int(d == b)][s[:, d][:, None], s[:, d][None, :]]
            row.append(g)
        out.append(row)
    return out


class _Plain:
    """Operator and load of a lattice problem in 64 bits."""

    def __init__(self, pb, md):
        dev = "cuda" if torch.cuda.is_available() else "cpu"
        self.dev, self.ns, self.neq = dev, md["nstate"], md["neq"]
        self.nall = self.neq
        h, dim = 1.0 / pb.nx, pb.dim
        sides = (_QUAD if dim == 2 else _HEX)
        if pb.p == 1:
            sides = sides[:2 ** dim]
        self.sides, self.h, self.dim, ns = sides, h, dim, self.ns
        G = _grams(sides, h)
        if ns == 1:
            K = sum(G[a][a] for a in range(dim)) * (pb.scale if pb.material == P.POISSON else 1.0)
        else:
            mu, lam = 1 / (2 * (1 + pb.nu)), pb.nu / ((1 + pb.nu) * (1 - 2 * pb.nu))
            K = np.zeros((len(sides), 3, len(sides), 3))
            for a in range(3):
                for b in range(3):
                    K[:, a, :, b] = lam * G[a][b] + mu * G[b][a]
                    if a == b:
                        K[:, a, :, b] += mu * sum(G[c][c] for c in range(3))
            K = K.reshape(3 * len(sides), -1)
        self.K = torch.from_numpy(K).to(dev)
        coef = md["vol_coef"] if md["vol_coef"] is not None else np.ones(len(md["vol_nodes"]))
        self.coef = torch.from_numpy(np.ascontiguousarray(coef)).to(dev)[:, None]
        self.conn = self._dofs(md, md["vol_conn"][:, :len(sides)])
        # boundary: [(type, value, dofs)] of every face in use
        ids, t = md["bc_id"], np.asarray(md["bc_type"])
        self.bsides = ([(0,), (1,), (2,)] if dim == 2 else _QUAD)
        if pb.p == 1:
            self.bsides = self.bsides[:2 ** (dim - 1)]
        self.faces = [(int(t[f]), np.asarray(md["bc_val"]).reshape(-1, 3)[f],
                       self._dofs(md, md["bc_conn"][ids == f][:, :len(self.bsides)])) for f in np.unique(ids)]
        self.big = md["big_number"]
        self.b = self._load(pb, md)

    def _dofs(self, md, conn):
        """Equations [element, shape * state]; a place of its own behind them for a side without a function."""
        pos = np.where(md["blk_size"] > 0, md["blk_pos"], -1)[conn]
        own = self.neq + np.arange(pos.size * self.ns).reshape(*pos.shape, self.ns)
        d = np.where(pos[:, :, None] >= 0, pos[:, :, None] + np.arange(self.ns), own)
        self.nall = max(self.nall, int(d.max()) + 1)
        return torch.from_numpy(d.reshape(len(conn), -1)).to(self.dev)

    def _load(self, pb, md):
        b = torch.zeros(self.nall, dtype=torch.float64, device=self.dev)
        if pb.force_kind != P.FORCE_NONE:
            x, w = _gauss(int(0.51 * (md["rule_order_vol"] + 2)))
            v, _ = _basis1d(x)
            corner = np.asarray(md["xyz"]).reshape(-1, 3)[np.asarray(md["vol_nodes"])[:, 0]][:, :self.dim]
            pts = np.stack(np.meshgrid(*[x] * self.dim, indexing="ij"), -1).reshape(-1, self.dim)
            wt = np.prod(np.stack(np.meshgrid(*[w] * self.dim, indexing="ij"), -1).reshape(-1, self.dim), 1)
            idx = np.stack(np.meshgrid(*[np.arange(len(x))] * self.dim, indexing="ij"), -1).reshape(-1, self.dim)
            phi = np.array([np.prod([v[s[d], idx[:, d]] for d in range(self.dim)], 0) for s in self.sides])
            W = torch.from_numpy(phi * wt * self.h ** self.dim).to(self.dev)          # [shape, q]
            X = torch.from_numpy(corner[:, None] + self.h * pts[None]).to(self.dev)   # [el, q, dim]
            if pb.force_kind == P.FORCE_CONST:
                f = torch.tensor(pb.force_const[:self.ns], dtype=torch.float64, device=self.dev).expand(
                    X.shape[0], X.shape[1], self.ns)
            else:
                f = 0
                for row in pb.bumps:
                    c = torch.from_numpy(row[:self.dim].copy()).to(self.dev)
                    a = torch.from_numpy(row[3:3 + self.ns].copy()).to(self.dev)
                    f = f + torch.exp(-((X - c) ** 2).sum(-1) / (2 * pb.bump_width ** 2))[..., None] * a
            fe = torch.matmul(W, f)  # [el, shape, state]
            if pb.material == P.POISSON:
                fe = fe * pb.scale
            b.index_add_(0, self.conn.reshape(-1), fe.reshape(-1))
        one = np.array([0.5, 0.5, 2 / 3]) * self.h  # integrals of the 1D functions
        m = np.array([np.prod([one[k] for k in s]) for s in self.bsides])
        for t, val, dofs in self.faces:
            if t == 1:
                fe = torch.from_numpy(np.outer(m, val[:self.ns]).ravel()).to(self.dev)
                b.index_add_(0, dofs.reshape(-1), fe.repeat(dofs.shape[0]))
        return b[:self.neq]

    def mult(self, x, penalty=False):
        xe = torch.cat([x, x.new_zeros(self.nall - self.neq)])
        y = torch.zeros_like(xe)
        y.index_add_(0, self.conn.reshape(-1), (torch.matmul(xe[self.conn], self.K) * self.coef).reshape(-1))
        if penalty:
            t = _tensor1d(self.h)[0][0]
            s = np.array(self.bsides)
            m = np.ones((len(s), len(s)))
            for d in range(s.shape[1]):
                m = m * t[s[:, d][:, None], s[:, d][None, :]]
            m = torch.from_numpy(np.kron(m, np.eye(self.ns)) * self.big).to(self.dev)
            for kind, _, dofs in self.faces:
                if kind == 0:
                    y.index_add_(0, dofs.reshape(-1), torch.matmul(xe[dofs], m).reshape(-1))
        return y[:self.neq]

    def solve(self):
        """Conjugate gradients with the Dirichlet equations held at zero (the penalty 1e12 and more
        leaves less than 1e-9 there)."""
        free = torch.ones(self.nall, dtype=torch.float64, device=self.dev)
        for kind, _, dofs in self.faces:
            if kind == 0:
                free[dofs.reshape(-1)] = 0
        free = free[:self.neq]
        diag = torch.zeros(self.nall, dtype=torch.float64, device=self.dev)
        diag.index_add_(0, self.conn.reshape(-1), (torch.diagonal(self.K)[None] * self.coef).reshape(-1))
        minv = free / diag[:self.neq]
        x, r = torch.zeros_like(free), self.b * free
        z = minv * r
        p, rho, stop = z.clone(), torch.dot(r, z), 1e-13 * float(torch.linalg.norm(r))
        for it in range(40000):
            q = self.mult(p) * free
            alpha = rho / torch.dot(p, q)
            x += alpha * p
            r -= alpha * q
            z = minv * r
            new = torch.dot(r, z)
            p = z + (new / rho) * p
            rho = new
            if it % 50 == 49 and float(torch.linalg.norm(r)) <= stop:
                break
        return x


def _plain_errors(case, seed):
    """H1 norm, L2 norm and H1 semi-norm of the error per element and of the mesh."""
    pb = _problem(case, seed)
    md = M.build(pb)
    u = _vector(seed, md["neq"])
    h, n = 1.0 / pb.nx, int(0.51 * (max(md["rule_order_vol"], case["order"]) + 2))
    x, w = _gauss(n)
    v, g = _basis1d(x)
    sides = _QUAD if pb.p == 2 else _QUAD[:4]
    ue = u[md["blk_pos"][md["vol_conn"][:, :len(sides)]]]
    corner = np.asarray(md["xyz"]).reshape(-1, 3)[np.asarray(md["vol_nodes"])[:, 0]]
    f = [np.stack([np.outer(a[i], b[j]).ravel() for i, j in sides]) for a, b in ((v, v), (g / h, v), (v, g / h))]
    X, Y = corner[:, :1] + h * np.repeat(x, n), corner[:, 1:2] + h * np.tile(x, n)
    wt = np.outer(w, w).ravel() * h * h
    d0 = (ue @ f[0] - np.sin(np.pi * X) * np.sin(np.pi * Y)) ** 2 @ wt
    d1 = ((ue @ f[1] - np.pi * np.cos(np.pi * X) * np.sin(np.pi * Y)) ** 2 +
          (ue @ f[2] - np.pi * np.sin(np.pi * X) * np.cos(np.pi * Y)) ** 2) @ wt
    e = np.stack([d0 + d1, d0, d1], 1)
    return dict(totals=np.sqrt(e.sum(0)), elements=np.sqrt(e))


def exact(case, seed):
    kind = case["kind"]
    if kind == "errors_quad":
        return _plain_errors(case, seed)
    if kind in ("tet", "errors_tet", "train"):
        # tetrahedra: the oriented side functions up to order 5 in plain torch take longer than the limit;
        # training: its pairs come from the library's own generator
        return None
    pb = _problem(case, seed)
    plain = _Plain(pb, M.build(pb))
    if kind == "matvec":
        return plain.mult(torch.from_numpy(_vector(seed, plain.neq)).to(plain.dev), penalty=True).cpu().numpy()
    return plain.solve().cpu().numpy()
