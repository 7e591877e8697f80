"""k_design's code rows at the edges of their words, against the oracle, bit for
bit: lengths around 4 codons (a word), 16 (a 16-byte word, no padding), 32 (a
plane group) and 256 (a wave's words), 2 to 16 CDS, both workgroup sizes; the
pool as the caller reads it, before and after the first generation."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

KEYS = ("genome", "obj", "idx", "pql", "sorted", "front_of")


@pytest.mark.parametrize("L", [3, 4, 5, 15, 16, 17, 31, 32, 33, 48, 63, 64, 65, 255, 256, 257])
def test_evaluation_lengths(cdp, orc, L):
    print("evaluate", L, flush=True)
    T = cdp.tables
    aa, tab = T.synth_protein(L - 1, L), T.synth_tables(L)
    pop = T.random_population(aa, 3, 9, L)
    for a, b in zip(cdp.evaluate(aa, tab, pop), orc.evaluate(aa, tab, pop)):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("L,m,threads", [(4, 2, 256), (16, 3, 512), (17, 16, 256), (33, 11, 512), (64, 2, 512),
                                         (65, 7, 256), (256, 2, 256), (257, 3, 512)])
def test_generations(cdp, orc, L, m, threads):
    print("generations", L, m, threads, flush=True)
    T = cdp.tables
    aa, tab = T.synth_protein(L - 1, L), T.synth_tables(L)
    gj = cdp.Job(aa, tab, m, 37, 2, 0.2, L).init()
    sh = gj.shapes()
    sh["design_threads"] = threads
    gj.shapes(set=sh)
    oj = orc.Job(aa, tab, m, 37, 2, 0.2, L)
    oj.init()
    for gen in range(5):
        a, b = gj.read(), oj.read()
        for k in KEYS:
            assert np.array_equal(a[k], b[k]), (gen, k, np.argwhere(a[k] != b[k])[:5])
        if gen == 2:  # reading converts the rows in the idle buffer: twice gives the same
            assert np.array_equal(a["genome"], gj.read()["genome"])
        gj.step(1)
        oj.step(1)
    gj.close()
