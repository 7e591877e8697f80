"""The chain of searches for a CDS's longest stem (csrc/cd_seek.h), compiled for
the host with the address sanitizer, against the oracle's closed form with its
tie rule: guesses that are right, too long and too short, seeds, budgets that
run out, repeats whose stems are far longer than the first guess, and CDS
without a stem."""
import os
import shutil
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "protein_encoding_v2_nsga-iii_amd", "csrc")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.fixture(scope="module")
def harness(tmp_path_factory):
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not available")
    out = str(tmp_path_factory.mktemp("chain") / "seek_chain_check")
    subprocess.run([HIPCC, "-O1", "-std=c++17", "--offload-host-only", "-x", "hip", "-Xarch_host",
                    "-fsanitize=address", "-I", CSRC, os.path.join(HERE, "seek_chain_check.cpp"), "-o", out],
                   check=True, capture_output=True)
    return out


def run(harness, lines, budget=None):
    r = subprocess.run([harness] + ([] if budget is None else [str(budget)]), input="\n".join(lines) + "\n",
                       capture_output=True, text=True, check=True)
    out = [tuple(map(int, x.split())) for x in r.stdout.strip().split("\n")]
    assert len(out) == len(lines)
    return out


def text(s):
    return "".join(map(str, s))


def sequences(rng, count):
    out = []
    for _ in range(count):
        n = 3 * int(rng.integers(2, 420))
        kind = int(rng.integers(0, 4))
        if kind == 0:
            s = rng.integers(0, 4, n)
        elif kind == 1:
            s = rng.choice(4, size=n, p=[0.42, 0.08, 0.08, 0.42])
        else:
            u = rng.integers(0, 4, int(rng.integers(1, 40)))
            if kind == 3:
                u = np.concatenate([u, 3 - u[::-1]])  # pairs with itself along whole diagonals
            s = np.resize(u, n)
            f = rng.random(n) < rng.choice([0.0, 0.01, 0.1])
            s[f] = rng.integers(0, 4, int(f.sum()))
        out.append(s.astype(np.uint8))
    return out


@pytest.mark.parametrize("budget", [None, 0, 1, 7])
def test_initialisation(orc, harness, budget):
    seqs = sequences(np.random.default_rng(3), 120)
    got = run(harness, [text(s) for s in seqs], budget)
    for s, g in zip(seqs, got):
        assert g[:3] == orc.sl(s, 0), len(s)
    assert budget != 0 or all(g[4] or g[0] == 0 for g in got)  # (no step: no search ends with a stem)


@pytest.mark.parametrize("budget", [None, 1])
@pytest.mark.parametrize("off", [-3, 0, 4])
def test_children(orc, harness, off, budget):
    """Children whose parent's stem pairs still (the search of the changed part)
    or not (a guess from its length, off by `off`)."""
    rng = np.random.default_rng(off + 9)
    lines, want, whole = [], [], 0
    for s in sequences(rng, 100):
        L = len(s) // 3
        l, p, q = orc.sl(s, 0)
        t, mask = s.copy(), np.zeros(L, int)
        for k in np.flatnonzero(rng.random(L) < 0.05):
            mask[k] = 1
            t[3 * k:3 * k + 3] = rng.integers(0, 4, 3)
        broken = any(int(t[p + i]) + int(t[q + l - 1 - i]) != 3 for i in range(l))
        if off and not broken:
            continue  # (a stem that pairs is the parent's own)
        whole += broken
        lines.append(f"{text(t)} {max(0, l + off) if broken else l} {p} {q} {text(mask)}")
        want.append(orc.sl(t, 0))
    assert whole > 10
    for g, w, x in zip(run(harness, lines, budget), want, lines):
        assert g[:3] == w, x.split()[1:4]


def test_long_repeats_are_searched_again(orc, harness):
    """A repeat whose stems run along whole diagonals stops the first search and
    is found by one at the length met, not by the tiles."""
    rng = np.random.default_rng(2)
    fk = np.concatenate([np.stack([np.full(250, 3), np.full(250, 3), rng.choice([1, 3], 250)], 1),
                         np.stack([np.zeros(250, int), np.zeros(250, int), rng.choice([0, 2], 250)], 1)], 1).ravel()
    seqs = [np.resize([3, 3, 3, 0, 0, 0], 1500), np.resize([0, 1, 2, 3], 1500), np.resize([3, 3, 1, 2, 0, 0], 3300), fk]
    for s, g in zip(seqs, run(harness, [text(s) for s in seqs])):
        assert g[:3] == orc.sl(np.asarray(s, np.uint8), 0)
        assert g[3] > 1 and not g[4], g


def test_no_stem_two_guesses(orc, harness):
    """CDS without a pair, or with pairs too short to search: two searches."""
    for u in ([0, 0, 2], [1, 0, 2], [2]):
        s = np.resize(u, 1800).astype(np.uint8)
        (g,) = run(harness, [text(s)])
        assert g[:3] == orc.sl(s, 0) and g[3] == 2 and g[4] == 1


def test_the_chain_ends(harness):
    """Whatever a search returns, the next one is shorter, or at least half as
    long again, or none; and after a longer one none is shorter."""
    cases = [(n, K, a, f, s, p) for n in (30, 600, 5000) for K in (5, 6, 9, 14) for a in (0, 1)
             for f in (0, K - 1, K, 2 * K) for s in (0, 4, K - 1, K, K + 1) for p in (0, 1)]
    for (n, K, a, f, s, p), (k,) in zip(cases, run(harness, ["after %d %d %d %d %d %d" % c for c in cases])):
        assert k < K or (not a and 2 * k >= 3 * K), (n, K, a, f, s, p, k)
        assert not (a and s >= K) or k == 0, (n, K, a, f, s, p, k)
