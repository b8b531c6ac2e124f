"""The kernel times a handle reports, by kind, where scalar steps are folded
into other launches (small systems).  Both halves of an iteration run the same
lower sweep, so their bracketed times agree; what the second half's first
launch takes along when nobody looks (the ||s|| test, a launch's worth of about
3 us) counts with the vector updates.
"""
import numpy as np
import pytest

import fpga_amd as fa
from fpga_amd.configs import GRID_128x128x64, scaled

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("spec,level", [(fa.GridSpec(16, 15, 12, seed=5), False),
                                        (fa.GridSpec(16, 15, 12, bs=4, seed=5), False),
                                        (scaled(GRID_128x128x64, 16, 15, 8), False),
                                        (scaled(GRID_128x128x64, 16, 15, 8), True)],
                         ids=["colours_2", "colours_2_bs4", "colours_4", "levels"])
def test_lower_sweep_times_of_both_halves(spec, level):
    print(f"case {spec} level={level}", flush=True)
    s = fa.generate(spec)
    g = fa.BicgstabSolver(s.bs, s.n, s.nnzb)
    try:
        g.upload_system(s)
        g.analyse(level)
        g.factor()
        x0, r0 = g.solve(s.b, tol=0.0, maxit=12)
        first, second, vec = [], [], []
        for _ in range(15):
            g.set_profiling(True)
            x, r = g.solve(s.b, tol=0.0, maxit=12)
            t = g.kernel_times(fa.KIND_LOWER)
            v = g.kernel_times(fa.KIND_VEC)
            g.set_profiling(False)
            # the same solve, and a bracket per half-iteration for each kind
            np.testing.assert_array_equal(x, x0)
            assert r.half_iterations == r0.half_iterations and len(t) == 25 and len(v) == 25
            first += list(t[0:24:2])
            second += list(t[1:24:2])
        # a launch takes 2.8 us or more; the medians of 180 agree far better
        assert abs(np.median(first) - np.median(second)) * 1e3 < 1.5, (np.median(first), np.median(second))
    finally:
        g.close()
