"""The reverse sweep's memory budget over repeated calls, compiled from its
header: a sequence of equal calls asks for the same blocks and takes no more
memory after the first, and all together stay within a quarter of what was free."""
import os
import shutil
import subprocess

import pytest

from conftest import ROOT

SRC = r"""
#include <cstdio>
#include <cstdlib>
#include "adjoint_budget.hpp"
int main(int, char **v) {
  // free memory, bytes of a state, blocks, steps per block, calls
  size_t free_b = strtoull(v[1], 0, 10), state = strtoull(v[2], 0, 10);
  const int nblocks = atoi(v[3]), every = atoi(v[4]), limit = atoi(v[5]), calls = atoi(v[6]);
  size_t held = 0;
  for (int i = 0; i < calls; ++i) {
    const size_t fixed = size_t(nblocks + 1 + every) * state, block = 10 * size_t(every) * state;
    const int kept = gocfd::capi::kept_blocks(free_b, held, fixed, block, limit);
    const size_t need = fixed + size_t(kept) * block;
    if (need > held) { free_b -= need - held; held = need; }
    printf("%d %zu\n", kept, held);
  }
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    if not shutil.which("g++"):
        pytest.skip("needs g++")
    d = tmp_path_factory.mktemp("budget")
    (d / "b.cpp").write_text(SRC)
    subprocess.run(["g++", "-std=c++17", "-I", os.path.join(ROOT, "gocfd_amd", "csrc"), "-o", str(d / "b"), str(d / "b.cpp")],
                   check=True)
    return str(d / "b")


@pytest.mark.parametrize("free,state,steps,every,limit", [
    (288 * 10**9, 32_000_000, 2000, 45, None),   # more records than fit
    (288 * 10**9, 32_000_000, 20, 5, None),      # all fit
    (288 * 10**9, 32_000_000, 2000, 45, 1),      # a spacing of the caller's
    (4 * 10**9, 32_000_000, 210, 15, None),      # not even the checkpoints' quarter
])
def test_equal_calls_take_no_more_memory(program, free, state, steps, every, limit):
    nblocks = -(-steps // every)
    out = subprocess.run([program] + [str(x) for x in (free, state, nblocks, every, limit or nblocks, 12)], check=True,
                         capture_output=True, text=True).stdout.split("\n")
    calls = [tuple(int(x) for x in line.split()) for line in out if line]
    assert len(set(calls)) == 1
    kept, held = calls[0]
    assert kept <= (limit or nblocks)
    assert kept == 0 or held <= free // 4
