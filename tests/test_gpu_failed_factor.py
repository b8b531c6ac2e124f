"""A factorisation that meets a singular block reports it, and the handle is
not factored afterwards, whatever it held before (a caller's own factors, which
the new ones have overwritten by then, or none); new values or factors make it
usable again.
"""
import numpy as np
import pytest

import fpga_amd as fa
from fpga_amd import wire

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bs", [3, 4])
def test_failed_factorisation_leaves_no_factors(bs):
    s = fa.generate(fa.GridSpec(12, 11, 5, bs=bs, seed=5))
    g = fa.BicgstabSolver(bs, s.n, s.nnzb)
    h = None
    try:
        g.upload_system(s)
        g.analyse()
        g.factor()
        _, perm, cptr = g.colouring()
        w = wire.export_handle(g, s.b, None)
        rowptr, colidx, vals, lu, dinv, _, b, _ = wire.import_arrays(bs, w)
        h = fa.BicgstabSolver(bs, s.n, len(colidx))
        h.upload_factored(cptr, rowptr, colidx, vals, lu, dinv)
        x, r = h.solve(b, tol=1e-8)
        xm, rm = h.solve_mixed(b, tol=1e-8)
        assert r.converged and rm.converged
        singular = vals.copy().reshape(-1, bs, bs)
        singular[rowptr[0] + int(np.searchsorted(colidx[rowptr[0]:rowptr[1]], 0))] = 0.0
        h.upload_factored(cptr, rowptr, colidx, singular, lu, dinv)
        with pytest.raises(fa.BdaError, match="singular"):
            h.factor()
        for call in (h.solve, h.solve_mixed, h.adjoint_solve, h.precond_apply_perm):
            with pytest.raises(fa.BdaError, match="bda_factor has not been called"):
                call(b)
        h.update_values(vals)
        h.factor()
        x2, r2 = h.solve(b, tol=1e-8)
        assert r2.half_iterations == r.half_iterations
        np.testing.assert_array_equal(x2, x)
        x2, r2 = h.solve_mixed(b, tol=1e-8)
        np.testing.assert_array_equal(x2, xm)
    finally:
        g.close()
        if h is not None:
            h.close()
