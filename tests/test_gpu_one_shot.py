"""Evaluations and selections from shared idle streams and buffers, against the
oracle, bit for bit: sizes that grow and shrink from call to call, a last chunk
of packed rows that is short, rows at every alignment, and calls from several
threads at once."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def evaluation(cdp, orc, L, m, count):
    T = cdp.tables
    aa, tab = T.synth_protein(L - 1, L), T.synth_tables(L)
    pop = T.random_population(aa, m, count, count)
    return (aa, tab, pop), orc.evaluate(aa, tab, pop)


@pytest.mark.parametrize("L,m,count", [(51, 2, 3), (402, 3, 871), (30, 2, 1), (1023, 5, 410), (7, 16, 1000)])
def test_chunks(cdp, orc, L, m, count):
    print("evaluate", L, m, count, flush=True)
    args, want = evaluation(cdp, orc, L, m, count)
    for _ in range(2):
        for a, b in zip(cdp.evaluate(*args), want):
            assert np.array_equal(a, b)


def test_threads(cdp, orc):
    work = []
    for t in range(6):
        rng = np.random.default_rng(t)
        obj = rng.random((2 * (40 + 70 * t), 6)).astype(np.float32)
        ext = np.full((6, 6), 1e9, np.float32)
        work.append((evaluation(cdp, orc, 40 + 111 * t, 2 + t % 3, 30 + 40 * t),
                     (obj, len(obj) // 2, 3), cdp.select(obj, len(obj) // 2, 3, 0, t, ext), orc.nds(obj, len(obj) // 2), ext))
    bad = []

    def run(t):
        (args, want), (obj, N, H), sel, fronts, ext = work[t]
        for _ in range(5):
            ok = all(np.array_equal(a, b) for a, b in zip(cdp.evaluate(*args), want))
            got = cdp.select(obj, N, H, 0, t, ext)
            ok &= all(np.array_equal(got[k], sel[k]) for k in sel)
            fo, nf = cdp.nds(obj, N)
            ok &= nf == fronts[1] and np.array_equal(fo, fronts[0])
            if not ok:
                bad.append(t)

    threads = [threading.Thread(target=run, args=(t,)) for t in range(len(work))]
    print("threads", len(threads), flush=True)
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


def test_windows(cdp):
    """More rows than one window: the designs on each side of its end."""
    print("windows", flush=True)
    T = cdp.tables
    L, m, count = 1001, 16, 2200
    aa, tab = T.synth_protein(L - 1, 9), T.synth_tables(9)
    pop = T.random_population(aa, m, count, 9)
    got = cdp.evaluate(aa, tab, pop)
    per = (32 << 20) // (m * L)
    assert 0 < per < count
    for a, b in ((0, 3), (per - 3, per + 3), (count - 3, count)):
        for x, y in zip(got, cdp.evaluate(aa, tab, pop[a:b])):
            assert np.array_equal(x[a:b], y)
