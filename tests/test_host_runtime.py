"""The engine's host code on a stand-in for the HIP runtime (fake_hip.cpp: two
devices, rules on streams, events and memory, kernels that do nothing), each
case in a process of its own."""
import os
import shutil
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))

SETUP = """
import ctypes as C, importlib, sys
F = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
F.fake_used.restype = F.fake_host.restype = C.c_size_t
sys.path.insert(0, sys.argv[2])
import numpy as np
cdp = importlib.import_module("protein_encoding_v2_nsga-iii_amd")
T = cdp.tables
def job(residues=30, m=2, N=16, seed=1):
    return cdp.Job(T.synth_protein(residues, seed), T.synth_tables(seed), m, N, 2, 0.1, seed).init()
"""


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    if not shutil.which("g++"):
        pytest.skip("g++ not available")
    out = str(tmp_path_factory.mktemp("hip") / "fake_hip.so")
    subprocess.run(["g++", "-O1", "-shared", "-fPIC", "-std=c++17", os.path.join(HERE, "fake_hip.cpp"), "-o", out],
                   check=True, capture_output=True)
    return out


def run(fake, code):
    r = subprocess.run([sys.executable, "-c", SETUP + code, fake, os.path.dirname(HERE)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]


@pytest.mark.parametrize("batched", [False, True])
def test_another_device_is_current(fake, batched):
    """A job or batch of device 0 is stepped (by graph and kernel by kernel) and
    read while device 1 is the thread's, which it stays."""
    run(fake, f"""
jobs = [job(seed=1), job(seed=2)]
work = cdp.Batch(jobs) if {batched} else jobs[0]
work.step(30)
F.hipSetDevice(1)
work.step(11)
jobs[0].read()
dev = C.c_int()
F.hipGetDevice(C.byref(dev))
assert dev.value == 1 and F.fake_launches(0) > 0 and F.fake_launches(1) == 0
job(seed=3).read()
assert F.fake_launches(1) > 0
""")


def test_memory_of_a_closed_job_can_be_had_again(fake):
    """With the call that ends it, as a server counts it."""
    run(fake, """
before = F.fake_used()
j = job()
assert F.fake_used() > before
j.step(3)
j.close()
assert F.fake_used() == before
""")


def test_idle_buffers_are_given_back(fake):
    """What a one-shot call keeps for the next one leaves no job, and no larger
    call, without memory; and what is kept is bounded."""
    run(fake, """
aa, tab = T.synth_protein(300, 1), T.synth_tables(1)
pop = T.random_population(aa, 2, 4000, 1)
cdp.evaluate(aa, tab, pop)
kept = F.fake_used()
assert 0 < kept <= 64 << 20 and F.fake_host() <= 64 << 20
need = cdp.device_bytes(301, 2, 500, 2)
F.fake_limit.argtypes = [C.c_size_t]
F.fake_limit(need + kept // 2)
j = job(residues=300, N=500)
assert F.fake_used() == need
j.close()
cdp.evaluate(aa, tab, pop[:1000])
kept = F.fake_used()
F.fake_limit(4 * kept)
cdp.evaluate(aa, tab, pop[:3200])
""")


def test_tuner_leaves_unused_shapes_alone(fake):
    """(every candidate is timed quicker than the one before, so a shape that
    the launches use ends at its last candidate.)  A pool of 256 with 256 CDS
    uses neither k_fronts nor k_stem_list; one of 5000 with 40000 both."""
    run(fake, """
for N, m, used in ((128, 2, False), (2500, 16, True)):
    j = job(m=m, N=N)
    j.shapes(set=dict(j.shapes(), fronts_threads=256, stem_waves=5))
    got, _ = j.tune(1)
    assert got["niche_threads"] == 1024 and got["assoc_designs"] == 64
    assert (got["fronts_threads"], got["stem_waves"]) == ((1024, 8) if used else (256, 5)), got
""")


@pytest.mark.parametrize("tuned,other", [((1024, 2), (1025, 2)), ((1024, 16), (1025, 16)), ((2048, 2), (2049, 2))])
def test_tuned_shapes_stay_with_their_launches(fake, tuned, other):
    """Sizes of one power of two on the two sides of a rule of the dispatch: the
    fused fronts and the one-workgroup niching (pools of 2048), the list of
    changed CDS (16384), the eight-wave build of k_design (2048 children)."""
    run(fake, f"""
untuned = job(m={other[1]}, N={other[0]}).shapes()
a = job(m={tuned[1]}, N={tuned[0]})
chosen, _ = a.tune(1)
assert chosen != untuned
assert job(m={other[1]}, N={other[0]}).shapes() == untuned
assert job(m={tuned[1]}, N={tuned[0]}, seed=2).shapes() == chosen
""")
