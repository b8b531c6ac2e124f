"""When a tile of a waiting sweep gives up (fpga_amd/csrc/wait_bound.hpp), on
the CPU: never while tiles are started, however slowly and however long one
wait takes; never because of time in which the wave did not run, which no clock
it could read would leave out; and after a bounded number of its own looks once
nothing moves.
"""
import shutil
import subprocess
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parent.parent / "fpga_amd" / "csrc"

PROGRAM = r"""
#include "wait_bound.hpp"
#include <cstdio>
#include <initializer_list>
using namespace bda;
int main() {
    int bad = 0;
    for (uint32_t patience : {0u, 1u, 5u, kWaitPatience}) {
        // one long wait of a healthy sweep: a tile started every `patience` looks
        WaitCount c;
        const uint32_t every = patience > 0 ? patience : 1;
        for (uint32_t look = 0; look < 40u * every; ++look)
            if (wait_over(c, (int32_t)(look / every), patience) && patience > 0) ++bad;
        // nothing moves: over at the look after `patience` equal ones, not before
        WaitCount d;
        uint32_t looks = 0;
        while (!wait_over(d, 7, patience)) ++looks;
        if (looks != patience + 1) ++bad;
        // a tile started just before that: the count begins again
        WaitCount e;
        for (uint32_t i = 0; i <= patience; ++i)
            if (wait_over(e, 7, patience)) ++bad;
        if (wait_over(e, 8, patience) || e.looks != 0) ++bad;
    }
    // usable in constant expressions: nothing it reads but its arguments (no clock)
    constexpr bool pure = [] { WaitCount c; return !wait_over(c, 3, 0) && wait_over(c, 3, 0); }();
    static_assert(pure && (kWaitLook & (kWaitLook - 1)) == 0, "");
    std::printf("%d\n", bad);
    return bad;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not found")
def test_wait_bound(tmp_path):
    src, exe = tmp_path / "wait_bound.cpp", tmp_path / "wait_bound"
    src.write_text(PROGRAM)
    b = subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-I", str(CSRC), str(src), "-o", str(exe)],
                       capture_output=True, text=True, timeout=300)
    assert b.returncode == 0, b.stderr[-3000:]
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "0"
