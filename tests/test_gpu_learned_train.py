"""Training steps of the learned smoother: all weight gradients in one launch,
the features formed once per call, no gradient of the fitted matrix.

Bars: those of the gradient check at three pairs (loss 1e-4, blocks 2e-3
relative, FP32 kernels), here at pair counts that are no multiple of the four
that the forward kernel takes at a time; two training calls of one step against
one call of two steps: equal, bit for bit (same kernels in the same order).
"""
import numpy as np
import pytest

import les_ref as R
from neopz_amd import mesh as M
from neopz_amd import problems as P
from neopz_amd.analysis import Context, TPZSSpStructMatrixHIP
from neopz_amd.learned import LearnedSmoother

pytestmark = pytest.mark.gpu


def _learned(pb, nrhs):
    c = Context(0)
    sm = TPZSSpStructMatrixHIP(c, M.build(pb))
    K = sm.Create()
    sm.Assemble(K)
    ls = LearnedSmoother(c)
    ls.setup(seed=7)
    ls.collect(nrhs=nrhs, seed=11)
    return c, K, ls


@pytest.mark.parametrize("nrhs", [1, 4, 6])
@pytest.mark.parametrize("name", ["hex_p2", "quad_p1"])
def test_gradient_at_pair_counts(name, nrhs):
    pb = P.elasticity3d(n=4, p=2, seed=2, field_kind="grf", load="body") if name == "hex_p2" else \
        P.darcy2d(n=17, p=1, seed=3)
    c, K, ls = _learned(pb, nrhs)
    w = ls.get_weights()
    w = w + 0.05 * np.random.default_rng(5).standard_normal(len(w)).astype(np.float32)
    ne = [k for k in range(1, 200) if R.offsets(k)["n"] == len(w)][0]
    G = w[: ne * ne].reshape(ne, ne)
    w[: ne * ne] = (0.5 * (G + G.T)).ravel()
    ls.set_weights(w)
    cia, cja, X, _ = ls.graph(K.neq)
    Rr, E, Mk = ls.samples(len(cia) - 1)
    loss, g = ls.loss_grad()
    loss_r, g_r = R.loss_grad(w, ne, X, cia, cja, Rr, E, Mk)
    assert abs(loss - loss_r) <= 1e-4 * abs(loss_r)
    o = R.offsets(ne)
    blocks = [(o["g"], ne * ne), (o["w0"], R.NF * R.NH), (o["w"], R.NH)]
    blocks += [(o[k][l], R.NH * R.NH) for l in range(R.NL) for k in ("a", "b")]
    for off, k in blocks:
        a, b = g[off:off + k].astype(np.float64), g_r[off:off + k]
        assert np.linalg.norm(a - b) <= 2e-3 * max(np.linalg.norm(b), 1e-12)
    c.close()


def test_steps_of_one_call_equal_single_calls():
    pb = P.elasticity3d(n=6, p=2, seed=2, field_kind="grf", load="body")
    out = []
    for calls in ((2,), (1, 1)):
        c, _, ls = _learned(pb, 4)
        for n in calls:
            last = ls.train(steps=n, lr=2e-3)[1]
        out.append((last, ls.get_weights()))
        c.close()
    assert out[0][0] == out[1][0] and np.array_equal(out[0][1], out[1][1])
