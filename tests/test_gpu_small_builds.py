"""Builds of few tiles: the topology's scan inside its emission (up to 256 tiles of
1,024 particles) and the walk groups beside the leaves (up to 200,000 particles)."""
import numpy as np
import pytest

import blitzar_amd as B

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n, bucket", [(1023, 16), (1025, 1), (200000, 16), (200001, 1),
                                       (262144, 16), (262145, 16)])
def test_topology_of_few_tiles_matches_oracle(oracle, n, bucket):
    rng = np.random.default_rng(n)
    pos = rng.standard_normal((n, 3)) ** 3
    with B.OctreeHip(n, leaf_capacity=16, bucket_capacity=bucket) as s:
        s.upload(pos, None, np.full(n, 1.0 / n, np.float32))
        s.build_tree()
        t = s.dump_tree()
    sk, _ = oracle.stable_sort(oracle.keys(pos, 0))
    ref = oracle.hip_tree(sk, oracle.leaf_depth(n, 16), bucket)
    for key in ("level", "prefix", "start", "count", "first_child", "nchild"):
        assert np.array_equal(t[key].astype(np.int64), ref[key].astype(np.int64)), key


# node counts below, around and far past a workgroup of 256 nodes and a look-back
# step of 64 workgroups; bucket 65: the tree built level by level
@pytest.mark.parametrize("n, bucket", [(1, 16), (65, 16), (900, 1), (20000, 1), (20000, 65),
                                       (200000, 2), (200001, 2)])
def test_every_particle_is_in_one_walk_group(n, bucket):
    rng = np.random.default_rng(n + bucket)
    pos = rng.standard_normal((n, 3)) ** 3
    m = rng.uniform(0.5, 1.5, n).astype(np.float32)
    with B.OctreeHip(n, theta=1e-3 if n < 1000 else 0.5, softening=0.05,
                     bucket_capacity=bucket) as s:
        s.upload(pos, None, m)
        for _ in range(3):  # the look-back's workspace is reused
            a = s.compute_accelerations().astype(np.float64)
        t = np.unique(rng.integers(0, n, 1500)).astype(np.uint32)
        ref = s.direct_forces_fp64(t)
    # a particle of no group keeps no acceleration (100 % off); of the walk at
    # theta 0.5 a few 1e-3 is expected, at most 0.05 of the typical force is allowed
    scale = np.linalg.norm(ref, axis=1)
    err = np.linalg.norm(a[t] - ref, axis=1)
    assert np.isfinite(a).all()
    assert (err <= 0.05 * np.maximum(scale, np.median(scale))).all()
    assert n == 1 or (np.linalg.norm(a, axis=1) > 0).all()


# Equal keys leave in particle order whatever order the store had: runs of 2, 3 and
# many, at the array's ends and across workgroups of 256; beyond 200,000 a launch of
# its own does it. The positions come in a second upload, so that the slots of a run
# are not in particle order.
@pytest.mark.parametrize("n, cells", [(2, 1), (3, 1), (300, 1), (5000, 1), (5000, 40),
                                      (200000, 20000), (200001, 20000)])
def test_ties_follow_the_particle_index(oracle, n, cells):
    rng = np.random.default_rng(n + cells)
    first = rng.standard_normal((n, 3))
    pos = rng.standard_normal((cells, 3))[rng.integers(0, cells, n)]
    m = np.full(n, 1.0 / n, np.float32)
    with B.OctreeHip(n, leaf_capacity=16, bucket_capacity=16) as s:
        s.upload(first, None, m)
        s.build_tree()
        s.upload(pos, None, m)
        s.build_tree()
        t = s.dump_tree()
    sk, order = oracle.stable_sort(oracle.keys(pos, 0))
    assert np.array_equal(t["sorted_keys"], sk)
    assert np.array_equal(t["sorted_ids"], order)
