"""Runs that end in the middle, in the paths of small systems.

Waiting sweeps: an entry that equals the mark of an unwritten one.  The mark is
put into a caller's own factors (a block of L, U or D^-1 of an early level, b is
finite), so that it comes out of the sweeps' arithmetic: the sweeps have to end
and the run to stop on the NaN.  The launches per level, which store what they
compute as it is, show that the mark does come out.

Folded scalar steps: a deadline that passes in mid-run.  The run stops as
aborted after some half-iterations, with the x and the residual norm of the last
one that was completed.
"""
import numpy as np
import pytest

import fpga_amd as fa
from test_gpu_sweep_product import links, random_system

pytestmark = pytest.mark.gpu

MARK64, MARK32 = 0x7FF8BDA5BDA5BDA5, 0x7FC0BDA5
# the double that converts to the FP32 mark
MARK32_AS_64 = 0x7FF817B4A0000000
SIGN = 1 << 63


def damaged(bs, factors, rowptr, colidx, vals, where, bits):
    """lu_values, dinv of a chain's factors with one entry of row 5 replaced."""
    (_, _, lv), (_, _, uv), dinv = factors
    n = len(rowptr) - 1
    rows = np.repeat(np.arange(n), np.diff(rowptr))
    lu = vals.reshape(-1, bs, bs).copy()
    lu[colidx < rows] = lv.reshape(-1, bs, bs)
    lu[colidx > rows] = uv.reshape(-1, bs, bs)
    dinv = dinv.reshape(-1, bs, bs).copy()
    nan = np.array([bits], np.uint64).view(np.float64)[0]
    at = {"L": np.flatnonzero((rows == 5) & (colidx < rows)), "U": np.flatnonzero((rows == 5) & (colidx > rows))}
    if where == "Dinv":
        dinv[5, 0, 0] = nan
    else:
        lu[at[where][0], 0, 0] = nan
    return lu, dinv


@pytest.mark.parametrize("bs", [3, 4])
@pytest.mark.parametrize("vec", ["f64", "f32"])
def test_mark_as_a_result(vec, bs):
    print(f"case {vec} bs={bs}", flush=True)
    n = 60
    rowptr, colidx, vals, b = random_system(bs, links(n, [(i, i + 1) for i in range(n - 1)]), 3)
    g, h = fa.BicgstabSolver(bs, n, len(colidx)), fa.BicgstabSolver(bs, n, len(colidx))
    seen = 0
    try:
        g.upload_bcsr(rowptr, colidx, vals)
        g.analyse(True)
        g.factor()
        np.testing.assert_array_equal(g.colouring()[1], np.arange(n))  # a level per row, in order
        factors = g.factors()
        for where in ("Dinv", "L", "U"):
            for sign in (0, SIGN):
                lu, dinv = damaged(bs, factors, rowptr, colidx, vals, where,
                                   (MARK64 if vec == "f64" else MARK32_AS_64) | sign)
                h.upload_factored(np.arange(n + 1, dtype=np.int32), rowptr, colidx, vals, lu, dinv)
                if vec == "f64":
                    seen += int((h.precond_apply_perm(b).view(np.uint64) == MARK64).sum())
                    runs = (h.solve, h.adjoint_solve)
                else:
                    z = h.precond_apply_perm_ex(b, 1)
                    seen += int((np.ascontiguousarray(z, np.float32).view(np.uint32) == MARK32).sum())
                    runs = (h.solve_mixed, h.adjoint_solve_mixed)
                for run in runs:
                    x, r = run(b, tol=1e-8)
                    assert r.nan_detected and not r.converged
        assert seen > 0
        h.upload_factored(np.arange(n + 1, dtype=np.int32), rowptr, colidx, vals,
                          *damaged(bs, factors, rowptr, colidx, vals, "U", 0))
        x, r = h.solve(b, tol=1e-8)
        assert r.converged
    finally:
        g.close()
        h.close()


@pytest.mark.parametrize("bs", [3, 4])
def test_folded_deadline_in_mid_run(bs):
    s = fa.generate(fa.GridSpec(48, 41, 31, bs=bs, seed=5, perm_sigma=1.5))
    g = fa.BicgstabSolver(s.bs, s.n, s.nnzb)
    rows = np.repeat(np.arange(s.n), np.diff(s.rowptr))

    def norm(x):
        ax = np.zeros((s.n, bs))
        np.add.at(ax, rows, np.einsum("qrc,qc->qr", s.values, x.reshape(s.n, bs)[s.colidx]))
        return np.linalg.norm(s.b - ax.ravel())

    try:
        g.upload_system(s)
        g.analyse()
        g.factor()
        x, r = g.solve(s.b, tol=1e-8)
        assert r.converged
        stopped = set()
        for ms in (0.6, 0.75, 0.9, 1.05, 1.2, 1.35, 1.5, 2.0, 3.0):
            g.set_options(timeout_s=ms * 1e-3, poll_iters=3)
            x, r = g.solve(s.b, tol=0.0, maxit=30000)
            assert r.aborted and not r.converged
            if r.half_iterations > 0:
                stopped.add(r.half_iterations)
                # the true residual drifts from the recurrence's by roundings of a
                # few dozen iterations; the step left out would be of its own size
                assert abs(norm(x) - r.final_norm) <= 1e-11 * np.linalg.norm(s.b) + 1e-6 * r.final_norm
        print("stopped after", sorted(stopped), flush=True)
        assert len(stopped) > 1, stopped
        g.set_options()
        x, r = g.solve(s.b, tol=1e-8)
        assert r.converged and not r.aborted
    finally:
        g.close()
