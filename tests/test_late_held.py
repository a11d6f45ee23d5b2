"""The smallest edge key (d2, smaller id) that a candidate yet unknown can give
a late point (3D cone search, first radius only), against its definition: such
a candidate lies beyond the point's reach; the earlier search left the key
(d2, id) of the nearest one, so that none comes before it, or a d2 up to and
with which there is none, or nothing.  Compiled for the host from the header
that the kernels use."""
import os
import subprocess

import pytest

import __graft_entry__ as ge

ALL = 0xffffffff
SOURCE = r"""
#include "emst_internal.h"
#include <cstdio>
int main()
{
    long long reach;
    unsigned long long key;
    unsigned pid;
    while (std::scanf("%lld %llu %u", &reach, &key, &pid) == 3)
        std::printf("%llu\n", (unsigned long long)emst::late_first((int32_t)reach, (uint64_t)key, pid));
    for (int32_t q : {0, 1, 5, 0x7ffffff0})
        if (emst::late_held(q) > -3 || emst::late_held(emst::late_held(q)) != q) return 1;
}
"""


@pytest.mark.parametrize("base", [0, 0x3f800000, 0x7f000000])
def test_first_key_of_unknown_candidates(tmp_path, base):
    (tmp_path / "rule.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    "-I" + os.path.join(ge.PKG_DIR, "csrc"), "-o", str(tmp_path / "rule"), str(tmp_path / "rule.cpp")],
                   check=True)
    ids, pids = range(4), (0, 2, 9)
    rows = [(r, (d, i), pid) for r in (-1, base, base + 2, base + 3) for d in (base, base + 2, base + 4, ALL)
            for i in ((0, 1, 3, ALL) if d != ALL else (ALL,)) for pid in pids]
    text = "".join(f"{r} {d << 32 | i} {pid}\n" for r, (d, i), pid in rows)
    out = subprocess.run([str(tmp_path / "rule")], input=text, capture_output=True, text=True, check=True).stdout
    for (r, left, pid), got in zip(rows, map(int, out.split())):
        nothing = left == (ALL, ALL)
        can = [(d, i) for d in range(0 if nothing and r < 0 else base, base + 8) for i in ids
               if d > r and (nothing or (d, i) >= left)] if base == 0 or not (nothing and r < 0) else [(0, 0)]
        least = min((d, min(i, pid)) for d, i in can)
        assert got >> 32 == least[0], (r, left, pid)
        # never above what a candidate can give; that key itself where the id is known
        assert got <= least[0] << 32 | least[1]
        if left[0] > r and left[1] != ALL:
            assert got == least[0] << 32 | least[1]
