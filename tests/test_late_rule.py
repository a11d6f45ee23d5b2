"""The rule that asks a late point (3D cone search, first radius only) in a
round, against its definition: an unknown candidate has a squared distance
beyond the point's reach and not below the bound that an earlier search left,
and it can be the component's edge while that is at most the edge's own (at
equal distances the ids decide).  Compiled for the host from the header that
the kernels use."""
import os
import subprocess

import pytest

import __graft_entry__ as ge

NONE = 0xffffffff
SOURCE = r"""
#include "emst_internal.h"
#include <cstdio>
int main()
{
    long long reach, lo;
    while (std::scanf("%lld %lld", &reach, &lo) == 2)
        std::printf("%u\n", emst::late_least((int32_t)reach, (uint32_t)lo));
}
"""


@pytest.fixture(scope="module")
def least(tmp_path_factory):
    d = tmp_path_factory.mktemp("late_rule")
    (d / "rule.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + os.path.join(ge.PKG_DIR, "csrc"), "-o", str(d / "rule"), str(d / "rule.cpp")], check=True)

    def run(pairs):
        text = "".join(f"{r} {lo}\n" for r, lo in pairs)
        out = subprocess.run([str(d / "rule")], input=text, capture_output=True, text=True, check=True).stdout
        return [int(x) for x in out.split()]
    return run


@pytest.mark.parametrize("base", [0, 0x3f800000, 0x7f000000])
def test_asked_while_a_candidate_can_be_the_edge(least, base):
    vals = [base + k for k in range(8)]
    pairs = [(r, lo) for r in [-1] + vals for lo in vals + [NONE]]
    for (r, lo), got in zip(pairs, least(pairs)):
        possible = [d for d in range(base, base + 12) if d > r and (lo == NONE or d >= lo)]
        for edge in vals + [NONE]:
            asked = got <= edge
            assert asked == (any(d <= edge for d in possible) or r < 0 and lo == NONE), (r, lo, edge)
