"""Batches whose changed CDS are listed in more than 64 sublists, with a CDS of
over 1024 codons among them, on both sides of 65536 CDS: the listed stem
kernel's two shapes on their prefix sums in LDS, with a few entries a workgroup
and (beside a CDS that leaves one workgroup a CU) with more than the 64 it
fetches at once.  Every job ends as it does alone, where each CDS has its own
workgroup."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

KEYS = ("genome", "obj", "idx", "pql", "sorted", "front_of")


# (jobs, N and m of the short jobs; N and codons of the long one): 4160, 4160,
# 16370 and 8194 children, 16640, 66560, 65480 and 131104 CDS
@pytest.mark.parametrize("jobs,N,m,long_N,long_L", [(16, 256, 4, 64, 1025), (16, 256, 16, 64, 1025),
                                                    (16, 1023, 4, 2, 20000), (8, 1024, 16, 2, 20000)])
def test_many_sublists(cdp, jobs, N, m, long_N, long_L):
    T = cdp.tables
    specs = [(20, m, N, s + 1) for s in range(jobs)] + [(long_L, 2, long_N, 99)]

    def job(L, m, N, seed):
        return cdp.Job(T.synth_protein(L - 1, seed), T.synth_tables(seed), m, N, 2, 0.2, seed).init()

    print("batch", jobs, N, m, long_N, long_L, flush=True)
    held = [job(*s) for s in specs]
    batch = cdp.Batch(held)
    batch.step(2)
    batch.sync()
    if long_L == 20000:  # more than 64 entries for each of 256 workgroups, twice
        assert sum(j.cds_scanned() for j in held) > 2 * 64 * 256
    for s, j in zip(specs, held):
        alone = job(*s)
        alone.step(2)
        a, b = alone.read(), j.read()
        alone.close()
        for k in KEYS:
            assert np.array_equal(a[k], b[k]), (s, k)
    batch.close()
    for j in held:
        j.close()
