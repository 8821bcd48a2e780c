"""Host side of the library's calls on a double of the HIP runtime (fake_hip.cpp):
what they leave behind when a copy or an allocation fails, what they allocate and
wait for, and how the events of a build add up. No GPU: kernels do nothing, so no
result is looked at."""
import os
import subprocess
import sys

import pytest

from conftest import ROOT

HERE = os.path.dirname(os.path.abspath(__file__))

PRELUDE = """
import ctypes as C, sys
fake = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
fake.fake_extra_memory.restype = C.c_size_t
import numpy as np
import blitzar_amd as B
def cube(n):
    rng = np.random.default_rng(n)
    return rng.random((n, 3)), rng.random((n, 3)), np.full(n, 1.0 / n, np.float32)
"""


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    so = tmp_path_factory.mktemp("fake") / "libfake_hip.so"
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-pthread", "-o", str(so),
                    os.path.join(HERE, "fake_hip.cpp")], check=True)
    return str(so)


def run(fake, body):
    """The body in a process of its own (the library binds to the double there)."""
    p = subprocess.run([sys.executable, "-c", PRELUDE + body, fake], cwd=ROOT, timeout=120,
                       capture_output=True, text=True)
    assert p.returncode == 0, (p.returncode, p.stdout, p.stderr)
    return p.stdout


@pytest.mark.parametrize("copy", [0, 1, 2])
def test_failed_upload_leaves_nothing_in_flight(fake, copy):
    """The caller's arrays are free when bh_hip_upload returns, also where one of
    its three copies failed; a later upload works."""
    run(fake, f"""
state = cube(1000)
with B.OctreeHip(1000) as s:
    fake.fake_fail_copy({copy})
    try:
        s.upload(*state)
    except B.BhHipError as e:
        assert "stage upload" in str(e), e
    else:
        raise SystemExit("the upload did not fail")
    assert fake.fake_uploads() == 0
    fake.fake_fail_copy(-1)
    s.upload(*state)
""")


@pytest.mark.parametrize("started", [0, 1, 3])
def test_download_without_memory_for_its_threads(fake, started):
    """A large copy out whose helper threads cannot all be started (no memory for
    the next one) is emptied by those that were, or by the caller alone."""
    run(fake, f"""
n = 200000
with B.OctreeHip(n) as s:
    s.upload(*cube(n))
    s.download()  # the ring and its events are there
    fake.fake_fail_new({started})
    pos, vel = s.download()
    fake.fake_fail_new(-1)
    assert np.isfinite(pos).all() and np.isfinite(vel).all()
""")


def test_kernels_are_done_before_their_copy_starts_threads(fake):
    """The helper threads of a large copy out spin until its first chunk lands, so
    they start only once the direct sum, or the network, has run."""
    run(fake, """
n = 200000
with B.OctreeHip(n) as s:
    s.upload(*cube(n))
    alone = fake.fake_threads()
    s.direct_forces_fp64(np.arange(n, dtype=np.uint32))  # 4.8 MB of results
    assert fake.fake_waiting_threads() <= alone, (fake.fake_waiting_threads(), alone)
    s.lff_forward(np.zeros((400000, 32), np.float32))
    assert fake.fake_waiting_threads() <= alone, (fake.fake_waiting_threads(), alone)
""")


@pytest.mark.parametrize("n, nt", [(2000000, 2000000), (1000, 2000000), (300000, 300001)])
def test_direct_sum_workspace_is_bounded(fake, n, nt):
    """Many targets are worked through in pieces: nothing above 8 MB is allocated."""
    run(fake, f"""
with B.OctreeHip({n}) as s:
    s.upload(*cube({n}))
    s.direct_forces_fp64([0])
    fake.fake_mark_memory()
    s.direct_forces_fp64(np.arange({nt}, dtype=np.uint32) % {n})
    assert fake.fake_extra_memory() <= 8 << 20, fake.fake_extra_memory()
""")


@pytest.mark.parametrize("n", [1000, 150000])
def test_parts_of_a_one_stream_build_add_up(fake, n):
    """The parts of a build whose kernels run one after the other sum to the whole
    (the double's events count kernels)."""
    run(fake, f"""
with B.OctreeHip({n}) as s:
    s.upload(*cube({n}))
    B.lib().bh_hip_set_timing(s._h, 1)
    s.build_tree()
    t = s.timings()
    parts = [t[k] for k in ("keys_ms", "sort_ms", "permute_ms", "tree_ms", "moments_ms")]
    assert min(parts) > 0 and sum(parts) == t["build_ms"], (parts, t["build_ms"])
    assert t["permute_ms"] == 1, t  # one launch
""")


@pytest.mark.parametrize("n", [1000, 300000])
def test_timed_builds_without_a_walk(fake, n):
    """bh_hip_build_tree with timing on: no walk ends, so none is read (an event never
    recorded left an error that failed the next call; one of an earlier call gave a
    negative time)."""
    run(fake, f"""
with B.OctreeHip({n}) as s:
    s.upload(*cube({n}))
    B.lib().bh_hip_set_timing(s._h, 1)
    for k in range(3):
        s.build_tree()
        assert s.timings()["walk_ms"] == 0 and s.timings()["build_ms"] > 0
    s.compute_accelerations(to_host=False)
    assert s.timings()["walk_ms"] > 0
    s.build_tree()
    assert s.timings()["walk_ms"] == 0
""")
