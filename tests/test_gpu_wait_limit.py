"""A solve whose waiting sweep gives up (fpga_amd/csrc/wait_bound.hpp): it
reports an error, leaves the caller's x as it was, and the handle solves as
before afterwards.  The limit is set so low that a healthy sweep runs into it:
near a chain's end the last tiles wait for one another, some microseconds each
with no further tile to start, and a limit of one poll is then exceeded.
"""
import numpy as np
import pytest
import torch

import fpga_amd as fa
from fpga_amd.solver import BdaError
from test_gpu_sweep_product import links, random_system

pytestmark = pytest.mark.gpu

KINDS = {
    "solve": lambda g, b, x: g.solve_dev(b, x, 1e-8, 200),
    "adjoint_solve": lambda g, b, x: g.adjoint_solve_dev(b, x, 1e-8, 200),
    "solve_mixed": lambda g, b, x: g.solve_mixed_dev(b, x, 1e-8, vec32=True),
    "solve_mixed_x64": lambda g, b, x: g.solve_mixed_dev(b, x, 1e-8, vec32=False),
    "adjoint_solve_mixed": lambda g, b, x: g.adjoint_solve_mixed_dev(b, x, 1e-8),
}


@pytest.mark.parametrize("bs", [3, 4])
@pytest.mark.parametrize("kind", list(KINDS))
def test_given_up_sweep(kind, bs):
    print(f"case {kind} bs={bs}", flush=True)
    n = 700
    rowptr, colidx, vals, b = random_system(bs, links(n, [(i, i + 1) for i in range(n - 1)]), 3)
    x0 = 0.1 * np.random.default_rng(1).standard_normal(n * bs)
    g = fa.BicgstabSolver(bs, n, len(colidx))
    try:
        g.upload_bcsr(rowptr, colidx, vals)
        g.analyse(True)  # as many levels as rows
        g.factor()
        db, dx = torch.from_numpy(b).cuda(), torch.from_numpy(x0).cuda()
        ref = dx.clone()
        r1 = KINDS[kind](g, db.data_ptr(), ref.data_ptr())
        assert r1.converged
        g.set_wait_limit(1)
        with pytest.raises(BdaError, match="wait did not end"):
            KINDS[kind](g, db.data_ptr(), dx.data_ptr())
        np.testing.assert_array_equal(dx.cpu().numpy(), x0)
        with pytest.raises(BdaError, match="no solve has run"):
            g.residual()
        with pytest.raises(BdaError, match="wait did not end"):
            getattr(g, kind.replace("_x64", ""))(b, x0, tol=1e-8)
        g.set_wait_limit()
        r2 = KINDS[kind](g, db.data_ptr(), dx.data_ptr())
        assert r2.converged and r2.norms == r1.norms
        assert torch.equal(dx, ref)
    finally:
        g.close()
