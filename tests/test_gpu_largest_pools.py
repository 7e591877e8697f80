"""The largest pools a job, a sort and a selection accept (16384 designs,
and the first whose keys do not fit beside the small pools' niching arrays), against the oracle, bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def pool(P, seed):
    obj = np.random.default_rng(seed).normal(size=(P, 6)).astype(np.float32)
    obj[:, 5] = np.round(obj[:, 5] * 2) / 2
    return obj


@pytest.mark.parametrize("P", [15750, 16384])
def test_sort_and_selection(cdp, orc, P):
    print("pool", P, flush=True)
    obj, ext = pool(P, P), np.ones((6, 6), np.float32)
    a, b = cdp.nds(obj, P // 2), orc.nds(obj, P // 2)
    assert a[1] == b[1] and np.array_equal(a[0], b[0])
    g, o = cdp.select(obj, P // 2, 4, 1, 9, ext), orc.select(obj, P // 2, 4, 1, 9, ext)
    for k in ("sorted", "front_of", "extremes", "ideal", "worst", "nadir"):
        assert np.array_equal(g[k], o[k]), k


def test_job(cdp, orc):
    print("job of 8192 designs", flush=True)
    T = cdp.tables
    aa, tab = T.synth_protein(9, 3), T.synth_tables(3)
    gj = cdp.Job(aa, tab, 2, 8192, 3, 0.1, 4).init()
    oj = orc.Job(aa, tab, 2, 8192, 3, 0.1, 4)
    oj.init()
    gj.step(2)
    oj.step(2)
    a, b = gj.read(), oj.read()
    for k in ("genome", "obj", "idx", "pql", "sorted", "front_of"):
        assert np.array_equal(a[k], b[k]), k
    small = cdp.Job(aa, tab, 2, 64, 3, 0.1, 4).init()  # (the small pools' niching beside it)
    batch = cdp.Batch([gj, small])
    batch.step(1)
    batch.sync()
    oj.step(1)
    assert np.array_equal(gj.read()["sorted"], oj.read()["sorted"])
    batch.close()
    small.close()
    gj.close()
