"""The stem kernels on each side of the lines between them, against the oracle,
bit for bit: offspring with a workgroup per CDS (up to 16384 CDS), with the
list of changed CDS (more, in at most and in over 64 sublists), with two waves
a CDS (over 65536); evaluation of up to 2048 CDS and of more; lengths around a
word of the change mask and around 3072 bases; repeats, whose words match
everywhere, so that the search gives up and the tiles are scanned."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

KEYS = ("genome", "obj", "idx", "pql")


def generations(cdp, orc, aa, tab, m, N, gens, seed):
    gj = cdp.Job(aa, tab, m, N, 2, 0.1, seed).init()
    oj = orc.Job(aa, tab, m, N, 2, 0.1, seed)
    oj.init()
    for gen in range(gens):
        gj.step(1)
        oj.step(1)
        a, b = gj.read(), oj.read()
        for k in KEYS:
            assert np.array_equal(a[k], b[k]), (gen, k, np.argwhere(a[k] != b[k])[:5])
    gj.close()


@pytest.mark.parametrize("N,m,L", [(1024, 16, 24), (1025, 16, 24), (4097, 4, 20), (4097, 16, 20)])
def test_launch_sizes(cdp, orc, N, m, L):
    print("launch", N, m, L, flush=True)
    T = cdp.tables
    generations(cdp, orc, T.synth_protein(L - 1, N), T.synth_tables(N), m, N, 2, N + m)


@pytest.mark.parametrize("L", [1024, 1025])
def test_listed_lengths(cdp, L):
    """(the children's records against the same designs evaluated anew: the
    oracle's stems of 16400 such CDS take half a minute)"""
    print("listed", L, flush=True)
    T = cdp.tables
    aa, tab = T.synth_protein(L - 1, L), T.synth_tables(L)
    j = cdp.Job(aa, tab, 16, 1025, 2, 0.1, L).init()
    j.step(3)
    r = j.read()
    j.close()
    for a, b in zip(cdp.evaluate(aa, tab, r["genome"]), (r["obj"], r["idx"], r["pql"])):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("L", [32, 64, 65, 1024, 1025])
def test_lengths(cdp, orc, L):
    print("length", L, flush=True)
    T = cdp.tables
    generations(cdp, orc, T.synth_protein(L - 1, L), T.synth_tables(L), 2, 24, 4, L)


@pytest.mark.parametrize("unit,L", [("K", 300), ("F", 700), ("FK", 1100)])
def test_repeats(cdp, orc, unit, L):
    print("repeats", unit, L, flush=True)
    T = cdp.tables
    aa = np.array([T.AMINO.index(c) for c in (unit * L)[:L - 1]] + [T.STOP], np.int8)
    generations(cdp, orc, aa, T.synth_tables(1), 2, 12, 3, L)


@pytest.mark.parametrize("m,count", [(2, 1024), (2, 1025)])
def test_evaluation_sizes(cdp, orc, m, count):
    print("evaluate", m, count, flush=True)
    T = cdp.tables
    aa, tab = T.synth_protein(39, 3), T.synth_tables(3)
    pop = T.random_population(aa, m, count, 5)
    for a, b in zip(cdp.evaluate(aa, tab, pop), orc.evaluate(aa, tab, pop)):
        assert np.array_equal(a, b)
