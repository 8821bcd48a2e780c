"""Walks with 1, 2, 4 and 8 waves per group against the FP64 direct sum.

At theta = 0.05 the walk opens (nearly) everything (not under the extent
criterion, which accepts compact far cells at any theta: left out), so its lists hold every
particle and fill and flush at every size; what is left is FP32 rounding. A
target's error is taken against the sum of the magnitudes it adds up, S: each
term carries a few roundings (about 4 x 6e-8) and a lane adds at most n / 2 of
them, whose roundings grow as the square root, 6e-8 x 160 at n = 50,001:
1e-5 S covers both. One list entry lost or taken twice is of order S / n, which the
smallest sizes resolve (1e-5 S is a hundredth of an entry there).
"""
import numpy as np
import pytest

import blitzar_amd as B

pytestmark = pytest.mark.gpu

EPS = float(np.float32(0.01))


# n on either side of the lines where the waves per group change on a
# 256-CU GPU, and the smallest sizes (groups of one target, one group)
@pytest.mark.parametrize("n, criterion, order", [
    (2, "com", 2), (17, "com", 2), (65, "bounds", 2),          # 4 and 8 waves
    (1009, "com", 2), (1009, "com", 1), (1009, "relative", 2),  # 4
    (1009, "bounds", 2),                                         # 8
    (40001, "relative", 1), (30001, "com", 2), (50001, "relative", 2),  # 2, 4, 2
    (40001, "bounds", 2),                                        # 4
    (50001, "com", 2),                                           # 1
])
def test_near_exact_walk_matches_direct_sum(n, criterion, order):
    pos, _, _ = B.plummer(n, seed=3)
    mass = np.random.default_rng(n).uniform(0.5, 1.5, n).astype(np.float32)
    t = np.unique(np.linspace(0, n - 1, 48).astype(np.uint32))
    with B.OctreeHip(n, theta=0.05, softening=0.01, criterion=criterion,
                     multipole_order=order, relative_alpha=1e-7) as s:
        s.upload(pos, None, mass)
        a = s.compute_accelerations()[t]
        ref = s.direct_forces_fp64(t)
        assert np.array_equal(s.compute_accelerations()[t], a) or criterion == "relative"
    for k, i in enumerate(t):
        d = pos - pos[i]
        S = (mass * np.linalg.norm(d, axis=1) * ((d * d).sum(1) + EPS * EPS) ** -1.5).sum()
        assert np.linalg.norm(a[k] - ref[k]) <= 1e-5 * S, (n, criterion, i)


@pytest.mark.parametrize("n", [1009, 50001])  # 4 and 2 waves
def test_periodic_short_range_walk(oracle, n):
    rng = np.random.default_rng(n)
    pos = rng.random((n, 3))
    m = np.full(n, 1.0 / n, np.float32)
    rs, rc, eps = 1.25 / 64, 4.5 * 1.25 / 64, 0.1 / 64
    with B.OctreeHip(n, theta=0.05, softening=eps, treepm_split_scale=rs, treepm_cutoff=rc,
                     periodic_box=1.0) as s:
        s.upload(pos, None, m)
        a = s.compute_accelerations()
    t = np.arange(0, n, n // 64)
    ref = oracle.direct_tpm_fp64(pos, m.astype(np.float64), t, float(np.float32(eps)),
                                 float(np.float32(rs)), float(np.float32(rc)), box=1.0)
    scale = np.linalg.norm(ref, axis=1).max()
    # the split weight errs by 1.6e-7, separations of neighbours by FP32 rounding
    assert np.abs(a[t] - ref).max() <= 2e-5 * scale



# The extent criterion, on either side of the lines where it takes 8, 4 and 1 waves
# per group on a 256-CU GPU. The particles lie in 216 clumps of radius 1e-3 on a
# lattice of spacing 0.2: a cell of several clumps has bmax >= 0.1 and is opened
# (theta R <= 0.05 x 1.74), a clump is accepted whole from outside, where its
# expansion is exact to (1e-3 / 0.2)^3. So the lists hold one cell or the particles of
# every clump, and what is left is FP32 rounding: of the terms, as above, and of
# positions up to 1, 2.4e-7 times the gradient 1 / R^3 of each term.
@pytest.mark.parametrize("n", [1009, 35001, 36001, 311001, 313001])
def test_extent_walk_of_clumps_matches_direct_sum(n):
    rng = np.random.default_rng(n)
    k = np.arange(n) % 216
    eps = float(np.float32(0.05))
    pos = 0.2 * np.stack([k // 36, k // 6 % 6, k % 6], 1)
    v = rng.standard_normal((n, 3))
    pos += 1e-3 * v / np.maximum(np.linalg.norm(v, axis=1, keepdims=True), 1.0)
    mass = rng.uniform(0.5, 1.5, n).astype(np.float32)
    t = np.unique(np.linspace(0, n - 1, 48).astype(np.uint32))
    with B.OctreeHip(n, theta=0.05, softening=0.05, criterion="extent", multipole_order=2) as s:
        s.upload(pos, None, mass)
        a = s.compute_accelerations()
        assert np.array_equal(s.compute_accelerations(), a)
        ref = s.direct_forces_fp64(t)
    for j, i in enumerate(t):
        d = pos - pos[i]
        r3 = ((d * d).sum(1) + eps * eps) ** -1.5
        S = (mass * np.linalg.norm(d, axis=1) * r3).sum()
        assert np.linalg.norm(a[i] - ref[j]) <= 1e-5 * S + 2.4e-7 * (mass * r3).sum(), (n, i)
