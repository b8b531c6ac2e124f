"""Sweeps whose tiles wait for one another (a solve's sweeps over many small
levels, or several small colours) against the launches per level that apply the preconditioner by itself
(which other tests hold to the oracle bit for bit).  A solve that stops after
its first half-iteration returns x = alpha phat, each entry rounded once, so
phat = M^-1 b shows in x up to the one number alpha: some double next to
x_k / phat_k must give every entry.  FP64, the two precision forms, and the
adjoint; level sets of grids, a chain (as many levels as rows), rows without
lower blocks, colourings on either side of the rule (2 to 5 colours, forward
and transposed launches differing).  Then whole solves: converged, and the same
bits when repeated.
"""
import numpy as np
import pytest

import fpga_amd as fa
from fpga_amd.configs import GRID_128x128x64, scaled
from test_gpu_sweep_product import grid_case, links, random_system

pytestmark = pytest.mark.gpu


def path(n):
    return lambda bs: random_system(bs, links(n, [(i, i + 1) for i in range(n - 1)]), 3)


def bands(bs):
    """40 levels of very different widths, with couplings over several levels."""
    rng = np.random.default_rng(12)
    widths = rng.integers(1, 400, 40)
    start = np.concatenate([[0], np.cumsum(widths)])
    pairs = []
    for k in range(1, 40):
        for r in range(start[k], start[k + 1]):
            pairs.append((int(rng.integers(start[k - 1], start[k])), r))
            pairs.append((int(rng.integers(0, start[k])), r))
    return random_system(bs, links(int(start[-1]), pairs), 4)


def clique_rows(bs):
    """Nine colours, most of one or two rows."""
    return random_system(bs, links(300, [(i, i + 1) for i in range(299)] +
                                   [(i, j) for i in range(100, 109) for j in range(100, i)]), 5)


CASES = {  # system, level sets
    "grid": (grid_case(scaled(GRID_128x128x64, 17, 14, 9)), True),
    "grid_wide": (grid_case(fa.GridSpec(40, 36, 12, seed=3)), True),
    "chain": (path(700), True),
    "bands": (bands, True),
    "levels_3": (path(3), True),
    "levels_4": (path(4), True),
    "colours_2": (grid_case(fa.GridSpec(9, 8, 7, seed=3)), False),
    "colours_4": (grid_case(scaled(GRID_128x128x64, 16, 15, 8)), False),
    "colours_wide": (grid_case(scaled(GRID_128x128x64, 37, 41, 19)), False),
    "colours_9": (clique_rows, False),
}


def check_scaled(x, phat, dtype):
    """x == dtype(alpha * phat) for one double alpha: every entry's rounding
    interval gives bounds on it, and a double between them must do."""
    x, p = x.astype(dtype), phat.astype(np.float64)
    assert np.array_equal(x[p == 0], p[p == 0].astype(dtype))
    x, p = x[p != 0], p[p != 0]
    half = np.spacing(np.abs(x)).astype(np.longdouble) / 2
    ends = np.sort(np.stack([(x - half) / p, (x + half) / p]), axis=0)
    lo, hi = ends[0].max(), ends[1].min()
    a = float((lo + hi) / 2)
    for m in range(-4, 5):
        if np.array_equal((p * (a + m * np.spacing(a))).astype(dtype), x):
            return
    raise AssertionError(f"no alpha in [{lo}, {hi}] gives x from phat")


@pytest.mark.parametrize("bs", [3, 4])
@pytest.mark.parametrize("name", list(CASES))
def test_waiting_sweeps(name, bs):
    print(f"case {name} bs={bs}", flush=True)
    make, level = CASES[name]
    rowptr, colidx, vals, b = make(bs)
    n = len(rowptr) - 1
    g = fa.BicgstabSolver(bs, n, len(colidx))
    try:
        g.upload_bcsr(rowptr, colidx, vals)
        g.analyse(level)
        g.factor()
        perm = g.colouring()[1]
        sp = lambda v: v.reshape(n, bs)[perm].ravel()
        x, _ = g.solve(b, tol=0.0, maxit=0)
        check_scaled(sp(x), g.precond_apply_perm(sp(b)), np.float64)
        x, _ = g.adjoint_solve(b, tol=0.0, maxit=0)
        check_scaled(sp(x), g.precond_apply_perm(sp(b), True), np.float64)
        for prec, vec32, dt in ((1, True, np.float32), (2, False, np.float64)):
            x, _ = g.solve_mixed(b, tol=0.0, max_outer=1, inner_tol=0.0, inner_maxit=0, vec32=vec32)
            check_scaled(sp(x), g.precond_apply_perm_ex(sp(b), prec), dt)
            x, _ = g.adjoint_solve_mixed(b, tol=0.0, max_outer=1, inner_tol=0.0, inner_maxit=0, vec32=vec32)
            check_scaled(sp(x), g.precond_apply_perm_ex(sp(b), prec, True), dt)
        for solve in ("solve", "solve_mixed", "adjoint_solve", "adjoint_solve_mixed"):
            x1, r1 = getattr(g, solve)(b, tol=1e-8)
            x2, r2 = getattr(g, solve)(b, tol=1e-8)
            assert r1.converged and r1.half_iterations == r2.half_iterations and r1.norms == r2.norms
            np.testing.assert_array_equal(x1, x2)
    finally:
        g.close()


def test_nan_right_hand_side_ends():
    """NaN entries, the mark of an unwritten entry among them, are results like
    any other: the sweeps end and the run stops on the NaN."""
    rowptr, colidx, vals, b = bands(3)
    n = len(rowptr) - 1
    g = fa.BicgstabSolver(3, n, len(colidx))
    try:
        g.upload_bcsr(rowptr, colidx, vals)
        g.analyse(True)
        g.factor()
        for bits in (0x7FF8BDA5BDA5BDA5, 0x7FF8000000000000):
            c = b.copy()
            c[5:50:7] = np.array([bits], np.uint64).view(np.float64)[0]
            x, r = g.solve(c, tol=1e-8)
            assert r.nan_detected and not r.converged
            x, r = g.solve_mixed(c, tol=1e-8)
            assert r.nan_detected and not r.converged
        x, r = g.solve(b, tol=1e-8)
        assert r.converged
    finally:
        g.close()
