"""Factorising again on one handle: new values on the same pattern, after the
precision form and the adjoint have been used (the factorisation then writes
the FP32 copies itself), against a fresh handle that makes them from its
finished factors.  L, U, D^-1, the product and the preconditioner in all three
kernel forms, forward and transposed, and the solves, bit for bit: both sides
round the same values.  Patterns: rows whose L blocks update only the diagonal
(a grid), rows with fill in other blocks (a clique in a grid, which takes the
search), level sets, a tile filled to its last block, one colour; and the
factors themselves against the oracle.
"""
import numpy as np
import pytest

import fpga_amd as fa
import oracle
from test_gpu_sweep_product import grid_case, links, random_system

pytestmark = pytest.mark.gpu


def clique(bs):
    pairs = [(i, i + 1) for i in range(499)] + [(i, j) for i in range(200, 212) for j in range(i)
                                                if j >= 200]
    return random_system(bs, links(500, pairs), 3)


def full_tile(bs):
    """Rows of 42 (3x3) or 32 (4x4) blocks: eight fill a wide tile exactly."""
    w, n = (42, 800) if bs == 3 else (32, 800)
    nb = [set() for _ in range(n)]
    for i in range(n // 2):
        for j in range(w - 1):
            k = n // 2 + (i + j * 9) % (n // 2)
            nb[i].add(k)
            nb[k].add(i)
    return random_system(bs, nb, 4)


CASES = {
    "grid": (grid_case(fa.GridSpec(11, 10, 9, seed=4, perm_sigma=2.0, inactive_frac=0.1, nnc_frac=0.05)), False),
    "levels": (grid_case(fa.GridSpec(8, 9, 5, seed=4)), True),
    "clique": (clique, False),
    "full_tile": (full_tile, False),
    "one_colour": (lambda bs: random_system(bs, links(70, []), 5), False),
}


def handle(bs, rowptr, colidx, vals, level):
    g = fa.BicgstabSolver(bs, len(rowptr) - 1, len(colidx))
    g.upload_bcsr(rowptr, colidx, vals)
    g.analyse(level)
    g.factor()
    return g


@pytest.mark.parametrize("bs", [3, 4])
@pytest.mark.parametrize("name", list(CASES))
def test_second_factorisation(name, bs):
    print(f"case {name} bs={bs}", flush=True)
    make, level = CASES[name]
    rowptr, colidx, vals, b = make(bs)
    vals2 = vals * np.random.default_rng(6).uniform(0.9, 1.1, (len(colidx), 1, 1))
    g, f = handle(bs, rowptr, colidx, vals, level), None
    try:
        g.solve_mixed(b, tol=1e-6)
        g.adjoint_solve_mixed(b, tol=1e-6)
        g.update_values(vals2)
        g.factor()
        f = handle(bs, rowptr, colidx, vals2, level)
        o = oracle.OracleSystem(bs, rowptr, colidx, vals2, level_scheduling=level)
        o.factor()
        p = np.random.default_rng(7).standard_normal(len(b))
        for a, c, e in zip(g.factors(), f.factors(), o.factors()):
            for u, v, w in zip(*(x if isinstance(x, tuple) else (x,) for x in (a, c, e))):
                np.testing.assert_array_equal(u, v)
                np.testing.assert_array_equal(u, w)
        for prec in (0, 1, 2):
            for tr in (False, True):
                np.testing.assert_array_equal(g.spmv_perm_ex(p, prec, tr), f.spmv_perm_ex(p, prec, tr))
                np.testing.assert_array_equal(g.precond_apply_perm_ex(p, prec, tr), f.precond_apply_perm_ex(p, prec, tr))
        for solve in ("solve", "solve_mixed", "adjoint_solve", "adjoint_solve_mixed"):
            xg, rg = getattr(g, solve)(b, tol=1e-8)
            xf, rf = getattr(f, solve)(b, tol=1e-8)
            assert rg.converged and rg.half_iterations == rf.half_iterations
            np.testing.assert_array_equal(xg, xf)
    finally:
        g.close()
        if f is not None:
            f.close()


@pytest.mark.parametrize("bs", [3, 4])
def test_values_survive_another_analysis(bs):
    """Device values given to an analysed handle, then another ordering: the
    second analysis must find them (the handle keeps them in colour order)."""
    import torch
    rowptr, colidx, vals, b = clique(bs)
    vals2 = vals * 1.5
    g, f = handle(bs, rowptr, colidx, vals, False), None
    try:
        d = torch.from_numpy(vals2).cuda()
        g.update_values_dev(d.data_ptr())
        g.analyse(True)
        g.factor()
        f = handle(bs, rowptr, colidx, vals2, True)
        xg, rg = g.solve(b, tol=1e-8)
        xf, rf = f.solve(b, tol=1e-8)
        assert rg.converged and rg.half_iterations == rf.half_iterations
        np.testing.assert_array_equal(xg, xf)
        with pytest.raises(fa.BdaError):
            g.update_values_dev(0)
    finally:
        g.close()
        if f is not None:
            f.close()
