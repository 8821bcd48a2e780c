"""Caller order <-> store order, and the ring copy that takes results out."""
import numpy as np
import pytest

import blitzar_amd as B

pytestmark = pytest.mark.gpu


# FP64 triples (24 n bytes) around the copy's chunk and thread limits: one
# chunk, one byte past it, one chunk per slot, the start of the threads, a
# ring that wraps, each with a ragged last chunk.
@pytest.mark.parametrize("n", [1, 2, 10922, 10923, 87381, 174762, 174763, 1000003])
def test_download_returns_the_upload_after_the_store_was_permuted(n):
    rng = np.random.default_rng(n)
    with B.OctreeHip(n) as s:
        for _ in range(2):  # the second upload meets a permuted store
            pos, vel = rng.standard_normal((n, 3)), rng.standard_normal((n, 3))
            mass = rng.uniform(0.5, 1.5, n).astype(np.float32)
            s.upload(pos, vel, mass)
            s.build_tree()
            p, v = s.download()
            assert np.array_equal(p, pos) and np.array_equal(v, vel)
        s.upload(pos, None, mass)
        assert np.array_equal(s.download()[1], np.zeros((n, 3)))
        if n == 1:
            return
        # masses follow their particles: two far targets feel the weighted sum
        t = np.array([0, n - 1], np.uint32)
        d = s.direct_forces_fp64(t)
    for k, i in enumerate(t):
        dx = pos - pos[i]
        r2 = (dx * dx).sum(1) + float(np.float32(0.01)) ** 2
        w = mass.astype(np.float64) * r2 ** -1.5
        # two FP64 sums of n terms in different orders
        assert np.allclose(d[k], (w[:, None] * dx).sum(0), rtol=1e-9, atol=1e-9 * w.sum())


@pytest.mark.parametrize("n", [3, 21845, 21846, 349526])
def test_accelerations_come_back_in_caller_order(n):
    rng = np.random.default_rng(n)
    pos = rng.standard_normal((n, 3))
    mass = rng.uniform(0.5, 1.5, n).astype(np.float32)
    order = rng.permutation(n)
    with B.OctreeHip(n) as s:
        s.upload(pos, None, mass)
        a = s.compute_accelerations()
    with B.OctreeHip(n) as s:
        s.upload(pos[order], None, mass[order])
        b = s.compute_accelerations()
    # distinct keys: both stores sort to the same order, so the walks agree bit for bit
    assert np.array_equal(a[order], b)
