"""Where pinned host memory is refused, results are copied the plain way: the
same trees and weights as with it.  The refusal is made in a process of its own
by a library that answers hipHostMalloc first."""
import os
import subprocess
import sys

import pytest

import __graft_entry__ as ge

pytestmark = pytest.mark.gpu

REFUSE = """
static int calls = 0;
int hipHostMalloc(void** p, unsigned long bytes, unsigned int flags)
{
    (void)bytes; (void)flags;
    ++calls;
    *p = 0;
    return 2;       /* hipErrorOutOfMemory */
}
int refused(void) { return calls; }
"""
PROGRAM = """
import ctypes, sys, zlib
shim = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL) if len(sys.argv) > 1 else None
import numpy as np
import __graft_entry__ as ge
pkg = ge.load_package()
for n, dim, rs in ((1000, 2, 0), (300_000, 3, 0), (300_000, 2, 1)):
    with pkg.Calculateur(dim=dim, round_search=rs) as c:
        c.initialize(pkg.synth(1, n, dim, 5))
        c.run()
        u, v, d = c.getLinks()
        w, m = c.evaluate()
        print(n, dim, m, repr(w), *(zlib.crc32(x.tobytes()) for x in (u, v, d, c.labels())))
with pkg.Calculateur(dim=2, round_search=1) as c:
    c.initialize_clouds([pkg.synth(0, n, 2, n) for n in (2000, 3000, 4000)])
    c.run()
    w, e, r = c.cloud_results()
    print(w.tolist(), e.tolist(), r.tolist())
if shim is not None:
    print("refused", shim.refused() > 0, file=sys.stderr)
"""


def run(args):
    r = subprocess.run([sys.executable, "-c", PROGRAM] + args, cwd=ge.ROOT, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr[-2000:]
    return r


def test_results_without_pinned_memory(tmp_path):
    print("case no pinned memory", flush=True)
    (tmp_path / "refuse.c").write_text(REFUSE)
    lib = str(tmp_path / "refuse.so")
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", lib, str(tmp_path / "refuse.c")], check=True)
    without, usual = run([lib]), run([])
    assert "refused True" in without.stderr
    assert without.stdout == usual.stdout and "300000" in usual.stdout
