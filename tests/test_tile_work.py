"""The stem scans (csrc/cd_tile.h, csrc/cd_scan.h) on repeats, compiled for the
host: the tiles follow a run of pairs once, not again in every tile that it
crosses, so the work a tile takes does not grow with the length of the CDS; the
anti-diagonals measure the first run of a length, not every one; and the
longest stem is the oracle's."""
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
    out = str(tmp_path_factory.mktemp("tiles") / "tile_work_check")
    subprocess.run([HIPCC, "-O1", "-std=c++17", "--offload-host-only", "-x", "hip", "-finstrument-functions",
                    "-I", CSRC, os.path.join(HERE, "tile_work_check.cpp"), "-o", out], check=True, capture_output=True)
    return out


def scan(harness, seqs, mode="tile"):
    text = "\n".join("".join(map(str, s)) for s in seqs) + "\n"
    r = subprocess.run([harness, mode], input=text, capture_output=True, text=True, check=True)
    return [tuple(map(int, x.split())) for x in r.stdout.strip().split("\n")]


# (A0 C1 G2 U3: repeats of units that are their own reverse complement pair
# along every diagonal of their period)
@pytest.mark.parametrize("unit", ["03", "333000", "0123"])
def test_work_a_tile(harness, unit):
    u = np.array(list(unit), np.uint8).astype(int)
    short, long_ = scan(harness, [np.resize(u, 3000), np.resize(u, 6000)])
    # twice the length: the share of tiles at the edges falls, each run is
    # followed over at most its own rows -- a tenth covers both
    assert long_[3] / long_[4] <= 1.1 * short[3] / short[4]


# (repeats with a pair at every few positions and no long run: CAG, AUG UGG)
@pytest.mark.parametrize("unit", ["102", "032322"])
def test_work_a_diagonal(harness, unit):
    u = np.array(list(unit), np.uint8).astype(int)
    pairs, none = scan(harness, [np.resize(u, 3000), np.zeros(3000, int)], "diag")
    # a run measured takes three calls and comes once or twice a diagonal of 24
    # chunks on average, of at least eight calls each
    assert 0 < pairs[0] < 4 and none[0] == 0
    assert pairs[3] <= 1.1 * none[3]


@pytest.mark.parametrize("mode", ["tile", "diag"])
def test_stems_of_repeats(orc, harness, mode):
    rng = np.random.default_rng(8)
    seqs = []
    for k in range(60):
        n = 3 * int(rng.integers(20, 400))
        s = np.resize(rng.integers(0, 4, int(rng.integers(1, 70))), n)
        f = rng.random(n) < rng.choice([0.0, 0.005, 0.05])
        s[f] = rng.integers(0, 4, int(f.sum()))
        seqs.append(s.astype(np.uint8))
    for s, g in zip(seqs, scan(harness, seqs, mode)):
        w = orc.sl(s, 0)
        if mode == "diag" or w[0] >= 4:  # (the tiles find runs of 4 and more)
            assert g[:3] == w, len(s)
