"""When the SOR sweep's copy of the matrices may take device memory (csrc/memrule.hpp, host code): it
leaves three times its size and 16 KB a cell; checked against the same rule in Python at its edges."""
from __future__ import annotations

import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "dndsr_amd", "csrc")
MAIN = r"""
#include <cstdio>
#include <cstdlib>
#include "memrule.hpp"
int main(int n, char **a)
{
    for (int i = 1; i + 2 < n; i += 3)
        std::printf("%d", (int)dndsr::roomForCopy(strtoull(a[i], nullptr, 10), strtoull(a[i + 1], nullptr, 10),
                                                  strtoull(a[i + 2], nullptr, 10)));
}
"""


@pytest.mark.parametrize("nCell,M,K", [(2, 2, 3), (151_949, 9, 6), (262_144, 19, 6), (2_000_000, 3, 4),
                                       (10_000_000, 19, 6)])
def test_copy_leaves_room(tmp_path, nCell, M, K):
    (tmp_path / "m.cpp").write_text(MAIN)
    subprocess.run(["g++", "-std=c++17", "-I", CSRC, str(tmp_path / "m.cpp"), "-o", str(tmp_path / "m")], check=True)
    copy = 8 * K * M * (M + 1) * nCell
    edges = (4 * copy, copy + 16384 * nCell)
    frees = [0, copy - 1, copy, 288 << 30] + [e + d for e in edges for d in (-1, 0, 1)]
    want = "".join(str(int(f >= max(edges))) for f in frees)
    args = [str(x) for f in frees for x in (f, copy, nCell)]
    assert subprocess.run([str(tmp_path / "m"), *args], capture_output=True, text=True, check=True).stdout == want
