"""The bytes behind bench.py's rates: where a solve reads colour 0's blocks once
for the upper sweep and the product, they count once (CPU only)."""
import importlib.util
from pathlib import Path

import pytest

import fpga_amd as fa

ROOT = Path(__file__).resolve().parent.parent


@pytest.mark.parametrize("bs", [3, 4])
@pytest.mark.parametrize("fp32", [False, True])
def test_merged_blocks_count_once(bs, fp32):
    spec = importlib.util.spec_from_file_location("bench", ROOT / "bench.py")
    bench = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(bench)
    s = fa.generate(fa.GridSpec(7, 6, 5, bs=bs, seed=1))  # two colours
    colour, perm, cptr = fa.colour_pattern(s.rowptr, s.colidx)
    assert len(cptr) == 3

    class Handle:
        def algorithmic_bytes(self, kind, fp32=False):
            return 0.0

        def colouring(self):
            return colour, perm, cptr

    apart = bench.iteration_bytes(Handle(), fa, s, fp32, False)
    once = bench.iteration_bytes(Handle(), fa, s, fp32, True)
    # with two colours half of the off-diagonal blocks are colour 0's; two half-iterations
    assert apart - once == (s.nnzb - s.n) * (bs * bs * (4 if fp32 else 8) + 4)


@pytest.mark.parametrize("upper,lower,merged", [(40, 20, True), (20, 20, False), (0, 0, False)])
def test_merged_launch_seen_in_the_brackets(upper, lower, merged):
    spec = importlib.util.spec_from_file_location("bench", ROOT / "bench.py")
    bench = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(bench)

    class Handle:
        def kernel_stats(self, kind):
            return ({fa.KIND_UPPER: upper, fa.KIND_LOWER: lower}[kind], 1.0)

    assert bench.merged_sweeps(Handle(), fa) == merged
