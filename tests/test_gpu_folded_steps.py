"""Scalar steps folded into the vector updates (few reduction partials) against
the CPU oracle and against themselves at the limits of the rule: one to a few
hundred product tiles (one load per thread in the folded sums), above 1,024
(four), above 4,096 (four more), and above 8,192 (launches of their own).  What has to hold on every
side: the iteration counts, flags and norms of the oracle's solve, the same
bits when a solve is repeated, and the stops around the folded
steps: an iteration cap (which stops after a first half), a convergence in the
first half, and the watchdog.
"""
import numpy as np
import pytest

import fpga_amd as fa
import oracle

pytestmark = pytest.mark.gpu

# product tiles (3x3: 48 rows of 7 blocks each, 4x4: 36): below, at and above the lines
SIZES = {"one_tile": (5, 3, 2), "few": (16, 15, 12), "over_1024": (48, 41, 31), "over_4096": (70, 64, 56),
         "over_8192": (101, 80, 52)}


@pytest.mark.parametrize("bs", [3, 4])
@pytest.mark.parametrize("name", list(SIZES))
def test_folded_solves(name, bs):
    print(f"case {name} bs={bs}", flush=True)
    nx, ny, nz = SIZES[name]
    s = fa.generate(fa.GridSpec(nx, ny, nz, bs=bs, seed=5, perm_sigma=1.5))
    g = fa.BicgstabSolver(s.bs, s.n, s.nnzb)
    try:
        g.upload_system(s)
        g.analyse()
        g.factor()
        o = oracle.OracleSystem(bs, s.rowptr, s.colidx, s.values)
        o.factor()
        for tol in (1e-2, 1e-6):
            x, r = g.solve(s.b, tol=tol)
            xo, ro = o.solve(s.b, tol=tol)
            # the dots are summed in another order: the counts agree, the norms
            # to rounding grown over a solve this short
            assert r.converged and r.half_iterations == ro["half_iterations"]
            np.testing.assert_allclose(x, xo, rtol=0, atol=1e-9 * np.abs(xo).max())
            x2, r2 = g.solve(s.b, tol=tol)
            np.testing.assert_array_equal(x, x2)
            assert r2.norms == r.norms
            # the true residual is the one the run stopped at
            res = g.residual()
            assert abs(np.linalg.norm(res) - r.final_norm) <= 1e-12 * r.norms[0] + 1e-9 * r.final_norm
        for maxit in (0, 1, 3):
            x, r = g.solve(s.b, tol=0.0, maxit=maxit)
            xo, ro = o.solve(s.b, tol=0.0, maxit=maxit)
            assert r.max_iter_reached and not r.converged and r.half_iterations == ro["half_iterations"]
            np.testing.assert_allclose(x, xo, rtol=0, atol=1e-9 * np.abs(xo).max())
        # a stop in a first half and one in a second: a cut of the history at each
        g.set_history(100)
        x, r = g.solve(s.b, tol=1e-9)
        hist = g.history()
        g.set_history(0)
        for k in (1, 2):
            if len(hist) > k:
                x, r = g.solve(s.b, tol=float(hist[k] / hist[0]) * 1.0000001, maxit=50)
                assert r.converged and r.half_iterations == k - 1 and r.final_norm == hist[k]
    finally:
        g.close()


def test_folded_watchdog():
    """Past its deadline a folded run stops as aborted, with a consistent x."""
    s = fa.generate(fa.GridSpec(16, 15, 12, seed=5))
    g = fa.BicgstabSolver(s.bs, s.n, s.nnzb)
    try:
        g.upload_system(s)
        g.analyse()
        g.factor()
        g.set_options(timeout_s=1e-7)
        x, r = g.solve(s.b, tol=0.0, maxit=2000)
        assert r.aborted and not r.converged and np.isfinite(x).all()
        g.set_options(timeout_s=0.0)
        x, r = g.solve(s.b, tol=1e-8)
        assert r.converged and not r.aborted
    finally:
        g.close()
