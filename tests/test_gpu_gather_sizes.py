"""Values on their way into the solver's order, for counts on either side of the
line between the two forms of the gather (2^20 entries), a block more or less,
and for the smallest: diagonal systems whose blocks are a unit matrix with one
integer beside the diagonal, so that every inverse, its transpose and its FP32
form are exact and every block differs from its neighbours.
"""
import numpy as np
import pytest

import fpga_amd as fa

pytestmark = pytest.mark.gpu

LINE = 1 << 20


@pytest.mark.parametrize("bs,n", [(3, 1), (3, 57), (3, 58), (4, 1), (4, 32), (4, 33), (3, LINE // 9), (3, LINE // 9 + 1),
                                  (4, LINE // 16 - 1), (4, LINE // 16), (4, LINE // 16 + 1)])
def test_gathered_blocks(bs, n):
    print(f"case bs={bs} n={n}", flush=True)
    vals = np.tile(np.eye(bs), (n, 1, 1))
    k = np.arange(n)
    vals[:, 0, bs - 1] = k % 4093 + 1
    p = ((np.arange(n * bs) * 7) % 31 - 15).astype(np.float64)
    g = fa.BicgstabSolver(bs, n, n)
    try:
        g.upload_bcsr(np.arange(n + 1, dtype=np.int32), np.arange(n, dtype=np.int32), np.ones_like(vals) + 4 * np.eye(bs))
        g.analyse()
        g.update_values(vals)
        g.factor()
        pb = p.reshape(n, bs)
        inv = np.tile(np.eye(bs), (n, 1, 1))
        inv[:, 0, bs - 1] = -vals[:, 0, bs - 1]
        np.testing.assert_array_equal(g.factors()[2].reshape(n, bs, bs), inv)
        np.testing.assert_array_equal(g.spmv_perm(p), np.einsum("krc,kc->kr", vals, pb).ravel())
        np.testing.assert_array_equal(g.spmv_perm(p, True), np.einsum("krc,kr->kc", vals, pb).ravel())
        np.testing.assert_array_equal(g.spmv_perm_ex(p, 1), np.einsum("krc,kc->kr", vals, pb).ravel())
        np.testing.assert_array_equal(g.precond_apply_perm(p, True), np.einsum("krc,kr->kc", inv, pb).ravel())
    finally:
        g.close()
