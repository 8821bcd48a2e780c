"""The mesh deposit through LDS windows and past them, against the FP64 mesh oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def f32(x):
    return float(np.float32(x))


# 1,024 particles a workgroup; sparse ones overflow the window, a blob across a corner of
# the box wraps it, coincident ones share 8 cells.
@pytest.mark.parametrize("n", [2, 1023, 1024, 1025, 30000])
@pytest.mark.parametrize("kind", ["uniform", "corner", "point"])
@pytest.mark.parametrize("mesh", [16, 96])
def test_deposit(n, kind, mesh):
    import blitzar_amd as B
    from oracle import pm
    print(f"case deposit n={n} {kind} mesh={mesh}", flush=True)
    rng = np.random.default_rng(n + mesh)
    pos = rng.random((n, 3))
    if kind == "corner":
        pos = np.mod(rng.normal(0.0, 0.03, (n, 3)), 1.0)
    if kind == "point":
        pos[: n // 2] = [0.21, 0.43, 0.87]
    m = (rng.uniform(0.5, 1.5, n) / n).astype(np.float32)
    h = 1.0 / mesh
    rs = 1.25 * h
    with B.OctreeHip(n, theta=0.6, softening=0.1 * h, treepm_split_scale=rs,
                     treepm_cutoff=2.5 * rs, periodic_box=1.0, pm_mesh=mesh) as s:
        s.upload(pos, None, m)
        s.compute_accelerations()  # the store is in Morton order from here on
        a = s.pm_accelerations()
    ref = pm.long_range_accel(pos, m.astype(np.float64), 1.0, mesh, f32(rs))
    l2 = np.linalg.norm(a - ref) / np.linalg.norm(ref)
    print(f"  l2={l2:.3e}", flush=True)
    assert l2 < 1e-4
