"""The engine's word search for stems (csrc/cd_seek.h), compiled for the host
with the address sanitizer, against the oracle's closed form with its tie rule:
whole searches at every length from 5 to the longest stem, and searches of the
changed part of children whose parent's longest stem still pairs, on random,
A/U rich (many ties), repetitive and planted sequences, with few and many
changed codons."""
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
    out = str(tmp_path_factory.mktemp("seek") / "seek_host_check")
    subprocess.run([HIPCC, "-O1", "-std=c++17", "--offload-host-only", "-x", "hip", "-Xarch_host",
                    "-fsanitize=address", "-I", CSRC, os.path.join(HERE, "seek_host_check.cpp"), "-o", out],
                   check=True, capture_output=True)
    return out


def run(harness, lines):
    r = subprocess.run([harness], input="\n".join(lines) + "\n", capture_output=True, text=True, check=True)
    f = r.stderr.split()
    return [tuple(map(int, o.split())) for o in r.stdout.strip().split("\n")], int(f[1]), int(f[3])


def sequence(rng, L):
    kind = int(rng.integers(0, 4))
    n = 3 * L
    if kind == 0:
        return rng.integers(0, 4, n)
    if kind == 1:
        return rng.choice(4, size=n, p=[0.42, 0.08, 0.08, 0.42])
    if kind == 2:
        s = np.resize(rng.integers(0, 4, int(rng.integers(5, 60))), n)
        f = rng.random(n) < 0.2
        s[f] = rng.integers(0, 4, int(f.sum()))
        return s
    s = rng.integers(0, 4, n)
    k = int(rng.integers(5, max(6, min(40, n // 3))))
    i = int(rng.integers(0, max(1, n - 2 * k - 8)))
    if i + 2 * k + 5 <= n:
        s[i + k + 5:i + 2 * k + 5] = 3 - s[i:i + k][::-1]
    return s


def text(s):
    return "".join(map(str, s))


def test_whole_search_every_length(orc, harness):
    rng = np.random.default_rng(1)
    lines, want = [], []
    for L in [5, 6, 7, 10, 11, 21, 22, 32, 43, 64, 100, 333, 501, 800, 1024, 1025]:
        for _ in range(3):
            s = sequence(rng, L).astype(np.uint8)
            w = orc.sl(s, 0)
            for K in range(5, w[0] + 1):
                if 3 * L > 3072 and K < 6:
                    continue  # (long CDS are searched from 6 on)
                lines.append(f"{text(s)} {K}")
                want.append(w if (3 * L - 4) // 2 >= K else (0, 0, 0))
    got, _, _ = run(harness, lines)
    assert len(got) == len(want) > 100
    for g, w, x in zip(got, want, lines):
        assert g == w, (len(x), x.split()[1])


@pytest.mark.parametrize("rate", [0.01, 0.05, 0.1, 0.4])
def test_changed_part(orc, harness, rate):
    rng = np.random.default_rng(int(rate * 1000))
    lines, want = [], []
    while len(lines) < 150:
        L = int(rng.choice([8, 11, 22, 33, 64, 101, 170, 400, 700, 1100]))
        s = sequence(rng, L).astype(np.uint8)
        l, p, q = orc.sl(s, 0)
        if l < 6:
            continue
        t = s.copy()
        mask = np.zeros(L, int)
        for k in np.flatnonzero(rng.random(L) < rate):
            mask[k] = 1  # (a marked codon may come out unchanged)
            t[3 * k:3 * k + 3] = rng.integers(0, 4, 3)
        if any(int(t[p + i]) + int(t[q + l - 1 - i]) != 3 for i in range(l)):
            continue  # the parent's stem does not pair any more
        lines.append(f"{text(t)} {l} {p} {q} {text(mask)}")
        want.append(orc.sl(t, 0))
    got, looked, total = run(harness, lines)
    for g, w, x in zip(got, want, lines):
        assert g == w, x.split()[1:4]
    assert looked <= total and (rate > 0.01 or looked < total)
