"""The second sweep of colour 0 and the product's colour-0 rows in one pass
(factors made by the library) against the separate launches (the same factors
handed in with upload_factored, of which the library assumes nothing): x, the
iteration counts and the residual norms bit for bit, in FP64 and in both
precision forms, below and above the number of colour-0 tiles (640) from which
the pass is taken: patterns of two colours (ragged last tiles), three colours,
a colour-0 row that fills a tile, many colours, level sets, one colour (nothing
to merge), and a start vector that is not zero.  Both sides add the same products in the same order, so the tolerance is zero.
"""
import numpy as np
import pytest

import fpga_amd as fa
from fpga_amd.configs import GRID_128x128x64, scaled

pytestmark = pytest.mark.gpu


def random_system(bs, nb, seed):
    """Block CSR of the symmetric neighbour sets nb, diagonally dominant."""
    rng = np.random.default_rng(seed)
    n = len(nb)
    cols = [sorted(nb[i] | {i}) for i in range(n)]
    rowptr = np.concatenate([[0], np.cumsum([len(c) for c in cols])]).astype(np.int32)
    colidx = np.concatenate(cols).astype(np.int32)
    vals = rng.uniform(-0.5, 0.5, (len(colidx), bs, bs))
    rows = np.repeat(np.arange(n), np.diff(rowptr))
    off = np.zeros((n, bs))
    np.add.at(off, rows[colidx != rows], np.abs(vals).sum(axis=2)[colidx != rows])
    d = np.flatnonzero(colidx == rows)
    vals[d] = rng.normal(0.0, 0.05, (n, bs, bs)) + (off + 1.0)[:, :, None] * np.eye(bs)
    return rowptr, colidx, vals, rng.uniform(-1, 1, n * bs)


def links(n, pairs):
    nb = [set() for _ in range(n)]
    for i, j in pairs:
        nb[i].add(j)
        nb[j].add(i)
    return nb


def grid_case(spec):
    def make(bs):
        d = dict(spec.__dict__)
        d.update(bs=bs)
        s = fa.generate(fa.GridSpec(**d))
        return s.rowptr, s.colidx, s.values, s.b
    return make


def three_colours(n):
    """Triangles along a line: colours 0, 1, 2, the last of few rows."""
    pairs = [(2 * i, 2 * i + 1) for i in range(n // 2)] + [(2 * i + 1, 2 * i + 2) for i in range(n // 2 - 1)]
    pairs += [(40 * i, 40 * i + 2) for i in range(min(n // 40, 30))]
    return lambda bs: random_system(bs, links(n, pairs), 7)


def full_row(bs):
    """Row 0 fills a sweep's tile on its own; the rest is a chain."""
    w, n = 168 if bs == 3 else 128, 83000
    return random_system(bs, links(n, [(0, j) for j in range(1, w)] + [(i, i + 1) for i in range(1, n - 1)]), 8)


def star_rows(bs):
    """Every colour-0 row couples to many later rows: tiles of few rows, their
    block capacity used up to the last block or nearly."""
    n, w = 2000 if bs == 3 else 1400, 100 if bs == 3 else 96
    m = 4 * n
    return random_system(bs, links(n + m, [(i, n + (i * 37 + 7 * j) % m) for i in range(n) for j in range(w)]), 11)


CASES = {
    "two_colours_few": (grid_case(fa.GridSpec(13, 9, 7, seed=2)), False),
    "two_colours": (grid_case(fa.GridSpec(47, 43, 33, seed=2)), False),
    "grid_nnc": (grid_case(scaled(GRID_128x128x64, 51, 49, 37)), False),
    "star_rows": (star_rows, False),
    "three_few": (three_colours(3000), False),
    "three_many": (three_colours(150000), False),
    "full_row": (full_row, False),
    "one_colour": (lambda bs: random_system(bs, links(130, []), 9), False),
    "two_rows": (lambda bs: random_system(bs, links(2, [(0, 1)]), 10), False),
    "levels": (grid_case(scaled(GRID_128x128x64, 9, 8, 7)), True),
}


def with_own_factors(g, n, bs, rowptr, colidx, vals):
    """A second handle holding g's colour-ordered system and factors as the caller's own."""
    _, perm, cptr = g.colouring()
    iperm = np.empty(n, np.int64)
    iperm[perm] = np.arange(n)
    rows = np.repeat(np.arange(n), np.diff(rowptr))
    pr, pc = iperm[rows], iperm[colidx]
    order = np.lexsort((pc, pr))
    prow, pcol = pr[order], pc[order].astype(np.int32)
    prp = np.searchsorted(prow, np.arange(n + 1)).astype(np.int32)
    (_, _, lv), (_, _, uv), dinv = g.factors()
    lu = np.zeros((len(pcol), bs, bs))
    lu[pcol < prow] = lv
    lu[pcol > prow] = uv
    h = fa.BicgstabSolver(bs, n, len(pcol))
    h.upload_factored(cptr, prp, pcol, vals[order], lu, dinv)
    return h, perm


@pytest.mark.parametrize("bs", [3, 4])
@pytest.mark.parametrize("name", list(CASES))
def test_same_bits_as_separate_launches(name, bs):
    print(f"case {name} bs={bs}", flush=True)
    make, level = CASES[name]
    rowptr, colidx, vals, b = make(bs)
    n = len(rowptr) - 1
    g = fa.BicgstabSolver(bs, n, len(colidx))
    h = None
    try:
        g.upload_bcsr(rowptr, colidx, vals)
        g.analyse(level)
        g.factor()
        h, perm = with_own_factors(g, n, bs, rowptr, colidx, vals)
        sp = lambda v: v.reshape(n, bs)[perm].ravel()
        x0 = np.random.default_rng(1).standard_normal(n * bs)
        for start in (None, x0):
            xg, rg = g.solve(b, start, tol=1e-8, maxit=300)
            xh, rh = h.solve(sp(b), None if start is None else sp(start), tol=1e-8, maxit=300)
            assert rg.converged and rg.half_iterations == rh.half_iterations and rg.norms == rh.norms
            np.testing.assert_array_equal(sp(xg), xh)
        for vec32 in (True, False):
            xg, rg = g.solve_mixed(b, tol=1e-8, vec32=vec32)
            xh, rh = h.solve_mixed(sp(b), tol=1e-8, vec32=vec32)
            assert rg.converged and rg.inner_half_iterations == rh.inner_half_iterations and rg.norms == rh.norms
            np.testing.assert_array_equal(sp(xg), xh)
    finally:
        g.close()
        if h is not None:
            h.close()
