"""The sort at the edges of its tiles, merge passes and radix fallback: stable,
bit-exact against numpy."""
import numpy as np
import pytest

import blitzar_amd as B

pytestmark = pytest.mark.gpu


def _keys(kind, n, rng):
    if kind == "random":
        return rng.integers(0, 1 << 64, n, dtype=np.uint64)
    if kind == "equal":
        return np.full(n, 0xfedcba9876543210, np.uint64)
    if kind == "few":  # long runs of ties, the largest key among them
        return rng.choice(np.array([0, 1, 1 << 40, (1 << 64) - 1], np.uint64), n)
    return np.arange(n, dtype=np.uint64)[::-1] << np.uint64(20)  # descending


# one tile of 2,048 / 4,096, two tiles, an odd number of runs with a short last
# one, the switch to tiles of 8,192, and sizes and widths that take the radix sort
@pytest.mark.parametrize("n", [2, 7, 8, 9, 2047, 2048, 2049, 4095, 4096, 4097, 8193, 12289, 40961,
                               1200001])
@pytest.mark.parametrize("bits", [8, 9, 30, 63, 64])
def test_sort_pairs_stable(n, bits):
    rng = np.random.default_rng(n + bits)
    for kind in ("random",) if n > 100000 else ("random", "equal", "few", "descending"):
        k = _keys(kind, n, rng)
        v = rng.integers(0, 1 << 32, n, dtype=np.uint32)
        ko, vo = B.sort_pairs(k, v, bits)
        masked = k & np.uint64((1 << bits) - 1)
        o = np.argsort(masked, kind="stable")
        assert np.array_equal(ko, k[o]) and np.array_equal(vo, v[o]), (kind, n, bits)


@pytest.mark.parametrize("n", [4194304, 4194305])  # the largest merge, the smallest radix sort
def test_sort_pairs_at_the_radix_line(n):
    rng = np.random.default_rng(n)
    k = rng.integers(0, 1 << 63, n, dtype=np.uint64)
    k[: n // 2] = k[n // 2: n // 2 * 2]  # ties far apart
    ko, vo = B.sort_pairs(k, np.arange(n, dtype=np.uint32), 63)
    o = np.argsort(k, kind="stable")
    assert np.array_equal(ko, k[o]) and np.array_equal(vo, o.astype(np.uint32))
