"""The sums of folded scalar steps are those of the launches of their own, bit
for bit: a product called by itself returns its dots through a launch that adds
up the same partial sums, and alpha and omega made of them have to give a
solve's x exactly.  b holds small integers, so that rho = b.b is exact in any
order.  Sizes: the tiles per load step of the folded sums (one load per thread,
four, eight), and beyond the rule, where the steps are launches of their own.
"""
import numpy as np
import pytest

import fpga_amd as fa
from test_gpu_folded_steps import SIZES

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bs", [3, 4])
@pytest.mark.parametrize("name", list(SIZES))
def test_folded_sums(name, bs):
    print(f"case {name} bs={bs}", flush=True)
    nx, ny, nz = SIZES[name]
    s = fa.generate(fa.GridSpec(nx, ny, nz, bs=bs, seed=5, perm_sigma=1.5))
    b = np.random.default_rng(2).integers(-8, 9, s.N).astype(np.float64)
    g = fa.BicgstabSolver(bs, s.n, s.nnzb)
    try:
        g.upload_system(s)
        g.analyse()
        g.factor()
        perm = g.colouring()[1]
        sp = lambda v: v.reshape(s.n, bs)[perm].ravel()
        r = sp(b)
        rho = float((b * b).sum())
        # first half-iteration: alpha = rho / (r.v)
        phat = g.precond_apply_perm(r)
        v, dots = g.spmv_perm_ex(phat, 0, w=r, red=1)
        alpha = rho / dots[0]
        x, res = g.solve(b, tol=0.0, maxit=0)
        assert res.max_iter_reached
        x1 = alpha * phat
        np.testing.assert_array_equal(sp(x), x1)
        # second: omega = (t.s) / (t.t); a tolerance that stops the run there
        sv = r + -alpha * v
        shat = g.precond_apply_perm(sv)
        _, dots = g.spmv_perm_ex(shat, 0, w=sv, red=3)
        omega = dots[0] / dots[1]
        g.set_history(8)
        g.solve(b, tol=0.0, maxit=1)
        hist = g.history()
        g.set_history(0)
        assert hist[0] == np.sqrt(rho) and hist[1] > hist[2] * 1.000001
        x, res = g.solve(b, tol=float(hist[2] / hist[0]) * 1.0000001, maxit=5)
        assert res.converged and res.half_iterations == 1 and res.final_norm == hist[2]
        np.testing.assert_array_equal(sp(x), x1 + omega * shat)
    finally:
        g.close()
