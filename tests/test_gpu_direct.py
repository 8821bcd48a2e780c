"""The FP64 direct sum over target tiles and source ranges against the oracle's."""
import numpy as np
import pytest

import blitzar_amd as B

pytestmark = pytest.mark.gpu


# tiles of 8 targets (one, one short, one over, many, more than n), source
# ranges of at least 1,024 (one range, ragged ones, 8 and more), a workspace
# that fits the staging buffer and one that does not; with softening, and
# without it, where coincident pairs and pairs below min_distance2 are skipped
@pytest.mark.parametrize("eps", [0.01, 0.0])
@pytest.mark.parametrize("n, nt", [(1, 1), (2, 2), (9, 30), (1023, 7), (2049, 8), (8192, 9),
                                   (9001, 3000), (70001, 257)])
def test_direct_sum_matches_oracle(oracle, n, nt, eps):
    rng = np.random.default_rng(n + nt)
    pos = rng.standard_normal((n, 3))
    pos[n // 2] = pos[0]  # a coincident pair (n > 1)
    if n > 4:
        pos[3] = pos[1] + 1e-7  # below min_distance2 when unsoftened
    m = rng.uniform(0.5, 1.5, n).astype(np.float32)
    t = np.concatenate([[0, n - 1], rng.integers(0, n, nt)])[:nt].astype(np.uint32)
    e = float(np.float32(eps))
    with B.OctreeHip(n, softening=eps, min_softening=0.0, min_distance2=1e-12) as s:
        s.upload(pos, None, m)
        if n > 8:
            s.build_tree()  # a permuted store
        a = s.direct_forces_fp64(t)
    ref = oracle.direct_fp64(pos, m.astype(np.float64), t.astype(np.int32), e, float(np.float32(1e-12)))
    for k, i in enumerate(t):
        d = pos - pos[i]
        r2 = (d * d).sum(1) + e * e
        w = np.where(r2 > 1e-12, m * np.maximum(r2, 1e-100) ** -1.5, 0.0)
        S = (w * np.linalg.norm(d, axis=1)).sum()
        # a few FP64 roundings a term and at most n / 256 additions in a row
        assert np.abs(a[k] - ref[k]).max() <= 1e-13 * S, (k, i)


# more targets than the workspace takes at once: two pieces and a ragged last one,
# with ranges of sources below 8 and of 8
@pytest.mark.parametrize("n, nt", [(3000, 200001), (20000, 60003)])
def test_pieces_of_targets_sum_the_same(n, nt):
    rng = np.random.default_rng(n)
    pos = rng.standard_normal((n, 3))
    m = rng.uniform(0.5, 1.5, n).astype(np.float32)
    t = rng.integers(0, n, nt).astype(np.uint32)
    with B.OctreeHip(n, softening=0.01) as s:
        s.upload(pos, None, m)
        s.build_tree()
        # (all n of them in one piece, in as many ranges)
        one = s.direct_forces_fp64(np.arange(n, dtype=np.uint32))
        assert np.array_equal(s.direct_forces_fp64(t), one[t])


# a target's own mass is no part of its force, whatever it is; a pair that is
# neither the target itself nor below min_distance2 counts, at infinity too
@pytest.mark.parametrize("eps", [0.01, 0.0])
@pytest.mark.parametrize("odd", [np.inf, -np.inf, np.nan])
def test_direct_sum_of_values_that_are_not_finite(oracle, eps, odd):
    n, k = 3001, 1234
    rng = np.random.default_rng(5)
    pos = rng.standard_normal((n, 3))
    m = rng.uniform(0.5, 1.5, n).astype(np.float32)
    t = np.array([k - 1, k, k + 1, 7, n - 1], np.uint32)
    far = pos.copy()
    far[k, 0] = odd
    heavy = m.copy()
    heavy[k] = odd
    with B.OctreeHip(n, softening=eps, min_softening=0.0, min_distance2=0.0) as s:
        s.upload(pos, None, heavy)
        a = s.direct_forces_fp64(t)
        s.upload(far, None, m)
        f = s.direct_forces_fp64(t)
    light = m.astype(np.float64)
    light[k] = 0.0
    e = float(np.float32(eps))
    ref = oracle.direct_fp64(pos, light, np.array([k], np.int32), e, 0.0)[0]
    # (the target with the mass that is not finite: FP64 roundings of a sum of |terms|)
    d = pos - pos[k]
    w = light * np.maximum((d * d).sum(1) + e * e, 1e-100) ** -1.5
    assert np.abs(a[1] - ref).max() <= 1e-13 * (w * np.linalg.norm(d, axis=1)).sum()
    assert not np.isfinite(a[[0, 2, 3, 4]]).any()
    assert np.isnan(f[:, 0]).all()
