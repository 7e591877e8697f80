"""The selection kernels at the edges of their tiles, against the oracle, bit
for bit: pools around the words of 64 designs, the workgroups' shares and the
line between the one-launch fronts and association (k_front_associate, at most
2048 designs a job and 4096 in all) and the three-launch one; few, 792 and more
than 1024 reference points; every association shape."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

KEYS = ("genome", "obj", "idx", "pql", "sorted", "front_of", "extremes", "ideal", "worst", "nadir")


def run_pair(cdp, orc, residues, m, N, H, gens, assoc=None, seed=77):
    T = cdp.tables
    aa, tab = T.synth_protein(residues, seed), T.synth_tables(seed)
    gj = cdp.Job(aa, tab, m, N, H, 0.1, seed).init()
    if assoc:
        sh = gj.shapes()
        sh["assoc_designs"] = assoc
        gj.shapes(set=sh)
    oj = orc.Job(aa, tab, m, N, H, 0.1, seed)
    oj.init()
    gj.step(gens)
    oj.step(gens)
    a, b = gj.read(), oj.read()
    gj.close()
    for k in KEYS:
        assert np.array_equal(a[k], b[k]), (k, np.argwhere(a[k] != b[k])[:5])


@pytest.mark.parametrize("N,H", [(1, 1), (5, 2), (31, 3), (32, 2), (33, 7), (127, 4), (129, 9), (257, 3), (511, 5),
                                 (1023, 2), (1024, 5), (1025, 2)])
def test_pool_edges(cdp, orc, N, H):
    print("pool", 2 * N, "H", H, flush=True)
    run_pair(cdp, orc, 30, 2, N, H, 4)


@pytest.mark.parametrize("assoc", [4, 8, 16, 32, 64])
def test_association_shapes(cdp, orc, assoc):
    print("association", assoc, flush=True)
    run_pair(cdp, orc, 40, 2, 150, 4, 3, assoc)


def test_reinitialised_job_starts_over(cdp, orc):
    # an odd number of generations, so that the latest selection sits in the
    # second half of the state when the job is initialised again
    T = cdp.tables
    aa, tab = T.synth_protein(30, 3), T.synth_tables(3)
    j = cdp.Job(aa, tab, 2, 40, 3, 0.1, 3).init()
    j.step(3)
    before = j.read()
    j.init()
    again = j.read()
    for k in ("ideal", "worst", "nadir"):
        assert np.array_equal(before[k], again[k]), k
    j.step(3)
    after = j.read()
    for k in KEYS:
        assert np.array_equal(before[k], after[k]), k
    j.close()
