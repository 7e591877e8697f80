"""Reads that take several chunks, and generations enqueued kernel by kernel
and as graphs in any order of step sizes, against the oracle, bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

KEYS = ("genome", "obj", "idx", "pql", "sorted", "front_of")


def same(a, b, keys=KEYS):
    for k in keys:
        assert np.array_equal(a[k], b[k]), k


@pytest.mark.parametrize("N,m,L", [(1100, 4, 1001), (1024, 2, 1024), (1025, 4, 1024)])
def test_chunks(cdp, orc, N, m, L):
    print("read", N, m, L, flush=True)
    T = cdp.tables
    aa, tab = T.synth_protein(L - 1, L), T.synth_tables(L)
    gj = cdp.Job(aa, tab, m, N, 2, 0.1, 5).init()
    oj = orc.Job(aa, tab, m, N, 2, 0.1, 5)
    oj.init()
    want = oj.read()
    for _ in range(2):
        same(gj.read(), want, ("genome", "obj", "idx", "pql"))
    gj.close()


@pytest.mark.parametrize("steps", [(1, 15, 1, 7, 9), (17, 8, 3), (16, 16, 1), (40,), (3, 30)])
def test_steps(cdp, orc, steps):
    print("steps", steps, flush=True)
    T = cdp.tables
    aa, tab = T.synth_protein(40, 4), T.synth_tables(4)
    gj = cdp.Job(aa, tab, 3, 20, 2, 0.2, 6).init()
    oj = orc.Job(aa, tab, 3, 20, 2, 0.2, 6)
    oj.init()
    for n in steps:
        gj.step(n)
        oj.step(n)
        same(gj.read(), oj.read())
    gj.close()
