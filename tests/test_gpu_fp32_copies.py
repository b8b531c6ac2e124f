"""The FP32 copies of a factored system are made for those who use them: after
a factorisation whose copies nobody asked for, the next one writes none (seen
in the device memory that it takes on a larger pattern), and steps that use the
precision form and steps that do not may follow one another in any order, each
with the bits of a handle of its own.
"""
import ctypes as C

import numpy as np
import pytest

import fpga_amd as fa
from test_zz_no_alloc import _hip, free_bytes

pytestmark = pytest.mark.gpu


def factor_bytes(g, hip):
    before = free_bytes(hip)
    g.factor()
    return before - free_bytes(hip)


def test_no_copies_unasked():
    hip = _hip()
    if hip is None:
        pytest.skip("no HIP runtime to ask for the free memory")
    large = fa.generate(fa.GridSpec(64, 64, 40, seed=2))
    taken = {}
    for name in ("never", "once"):
        g = fa.BicgstabSolver(3, large.n, large.nnzb)
        try:
            # a pattern of the handle's size with few blocks, then one with all
            rows = np.arange(large.n, dtype=np.int32)
            diag = np.repeat(np.eye(3)[None], large.n, axis=0) * 2.0
            g.upload_bcsr(np.arange(large.n + 1, dtype=np.int32), rows, diag)
            g.analyse()
            g.factor()
            if name == "once":
                g.spmv_perm_ex(np.ones(large.N), 1)
            g.factor()
            g.solve(large.b, tol=1e-6)
            g.upload_system(large)
            g.analyse()
            taken[name] = factor_bytes(g, hip)
        finally:
            g.close()
    # A32 alone has 9 floats for each of 1.1 million blocks: 40 MB
    assert abs(taken["once"] - taken["never"]) < 8 << 20, taken


@pytest.mark.parametrize("bs", [3, 4])
def test_steps_in_any_order(bs):
    spec = fa.GridSpec(24, 21, 12, bs=bs, seed=3, perm_sigma=1.5)
    s = fa.generate(spec)
    g = fa.BicgstabSolver(bs, s.n, s.nnzb)
    rng = np.random.default_rng(4)
    try:
        g.upload_system(s)
        g.analyse()
        for mixed in (True, False, True, True, False, False, True):
            vals = s.values * rng.uniform(0.9, 1.1, (s.nnzb, 1, 1))
            g.update_values(vals)
            g.factor()
            f = fa.BicgstabSolver(bs, s.n, s.nnzb)
            f.upload_bcsr(s.rowptr, s.colidx, vals)
            f.analyse()
            f.factor()
            solve = "solve_mixed" if mixed else "solve"
            xg, rg = getattr(g, solve)(s.b, tol=1e-8)
            xf, rf = getattr(f, solve)(s.b, tol=1e-8)
            f.close()
            assert rg.converged and rg.norms == rf.norms
            np.testing.assert_array_equal(xg, xf)
    finally:
        g.close()
