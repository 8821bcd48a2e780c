"""Moments of internal nodes, tile by tile and across tiles, from their children.

Sizes around a tile of 1,024 particles and the 512 tiles that one workgroup of
straddling nodes holds."""
import numpy as np
import pytest

import blitzar_amd as B

pytestmark = pytest.mark.gpu


def _check(t):
    m = t["moments"].astype(np.float64)
    unit = t["geom"][9:12]
    par = np.flatnonzero(t["nchild"] > 0)
    first, nc = t["first_child"][par], t["nchild"][par]
    pos = m[:, :3] + t["lattice"] * unit  # COM from the lattice origin
    mass32 = t["moments"][:, 3]
    M = np.zeros(len(par), np.float32)
    com, M64 = np.zeros((len(par), 3)), np.zeros(len(par))
    for k in range(8):  # children in order, added in FP32: the same bits
        live = k < nc
        c = np.where(live, first + k, first)
        M = (M + np.where(live, mass32[c], np.float32(0.0))).astype(np.float32)
        com += np.where(live, m[c, 3], 0.0)[:, None] * pos[c]
        M64 += np.where(live, m[c, 3], 0.0)
    assert np.array_equal(M, mass32[par])
    com /= M64[:, None]
    width = m[par, 10][:, None]
    # FP32 arithmetic on offsets no larger than the cell: a few roundings of the width
    assert (np.abs(com - pos[par]) <= 1e-5 * width).all()
    trs = np.zeros(len(par))
    bmax = np.zeros(len(par))
    qxx = np.zeros(len(par))
    for k in range(8):
        live = k < nc
        c = np.where(live, first + k, first)
        d = pos[c] - pos[par]
        r2 = (d * d).sum(1)
        w = np.where(live, m[c, 3], 0.0)
        trs += w * r2 + np.where(live, m[c, 11], 0.0)
        qxx += w * (3 * d[:, 0] ** 2 - r2) + np.where(live, m[c, 4], 0.0)
        bmax = np.maximum(bmax, np.where(live & (w > 0), np.sqrt(r2) + m[c, 9], 0.0))
    scale = M * width[:, 0] ** 2
    assert (np.abs(trs - m[par, 11]) <= 1e-5 * scale).all()
    assert (np.abs(qxx - m[par, 4]) <= 1e-5 * scale).all()
    assert (np.abs(bmax - m[par, 9]) <= 1e-5 * width[:, 0]).all()


@pytest.mark.parametrize("bucket", [1, 16])
@pytest.mark.parametrize("n", [2, 9, 1023, 1024, 1025, 5000, 524288, 524289])
def test_internal_moments_follow_from_the_children(n, bucket):
    pos, vel, _ = B.plummer(n, seed=n)
    mass = np.random.default_rng(n).uniform(0.5, 1.5, n).astype(np.float32)
    with B.OctreeHip(n, bucket_capacity=bucket) as s:
        s.upload(pos, vel, mass)
        s.build_tree()
        _check(s.dump_tree())


@pytest.mark.parametrize("bucket", [1, 16, 64])
@pytest.mark.parametrize("n", [2048, 8192, 8193, 40000])
def test_moments_of_units_of_several_tiles_and_full_levels(n, bucket):
    # up to 8 tiles one workgroup takes the whole tree; bucket 1 gives levels of
    # more nodes than its lanes; the coincident particles one deep chain
    pos, vel, _ = B.plummer(n, seed=n + 1)
    pos[: n // 50] = pos[0]
    mass = np.random.default_rng(n).uniform(0.5, 1.5, n).astype(np.float32)
    with B.OctreeHip(n, bucket_capacity=bucket) as s:
        s.upload(pos, vel, mass)
        s.build_tree()
        _check(s.dump_tree())


# With third moments (learned correction) 385 tiles go through two passes of straddling
# nodes, 384 through one.
@pytest.mark.parametrize("n", [393216, 393217])
def test_moments_with_third_order(n):
    pos, vel, m = B.plummer(n, seed=n)
    with B.OctreeHip(n, theta=0.9, softening=0.01) as s:
        s.lff_configure(theta=0.9, band=0.75, min_count=64)
        s.upload(pos, vel, m)
        s.build_tree()
        _check(s.dump_tree())
