"""The periodic TreePM walk where pairs take their own nearest image (entries half a box
from some target) and where the group's image serves, against the FP64 direct sum."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def f32(x):
    return float(np.float32(x))


# Few particles: one group spans the box. 20,000: four waves a group; 400,000: one.
@pytest.mark.parametrize("n,theta,rc", [(2, 0.05, 0.24), (17, 0.05, 0.24), (65, 0.05, 0.24),
                                        (300, 0.05, 0.24), (20000, 0.05, 0.05),
                                        (400000, 0.05, 0.05)])
def test_images_of_wide_and_narrow_groups(oracle, n, theta, rc):
    import blitzar_amd as B
    print(f"case images n={n} theta={theta} rc={rc}", flush=True)
    rng = np.random.default_rng(n)
    pos = rng.random((n, 3))
    if n == 2:  # neighbours across a corner of the box
        pos = np.array([[0.02, 0.98, 0.03], [0.97, 0.05, 0.99]])
    m = (rng.uniform(0.5, 1.5, n) / n).astype(np.float32)
    rs, eps = rc / 4.5, 0.05 * rc
    with B.OctreeHip(n, theta=theta, softening=eps, treepm_split_scale=rs, treepm_cutoff=rc,
                     periodic_box=1.0) as s:
        s.upload(pos, None, m)
        a = s.compute_accelerations()
    t = np.unique(np.linspace(0, n - 1, 150).astype(int))
    ref = oracle.direct_tpm_fp64(pos, m.astype(np.float64), t, f32(eps), f32(rs), f32(rc), box=1.0)
    l2 = np.linalg.norm(a[t] - ref) / np.linalg.norm(ref)
    print(f"  l2={l2:.3e}", flush=True)
    # all opened: FP32 sums, and the odd pair in or out at the cutoff
    assert l2 < 1e-4
