"""The merge sort of the Morton keys at the edges of its tiles (4,096) and merge
chunks (1,024): one tile, a full and an overflowing one, odd and even numbers of
merge passes, runs without a partner, equal keys.  Keys and the stable
permutation against numpy's."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _keys(pos):
    lo = pos.min(0)
    ext = (pos.max(0) - lo).max()
    scale = float(2 ** 21) / (ext * (1.0 + 2.0 ** -30)) if ext > 0 else 0.0
    q = np.clip(np.floor((pos - lo) * scale), 0, 2 ** 21 - 1).astype(np.uint64)
    out = np.zeros(len(pos), np.uint64)
    for b in range(21):
        for a, sh in ((0, 2), (1, 1), (2, 0)):
            out |= ((q[:, a] >> np.uint64(b)) & np.uint64(1)) << np.uint64(3 * b + sh)
    return out


@pytest.mark.parametrize("kind", ["random", "ties", "sorted", "reversed", "one_point"])
@pytest.mark.parametrize("n", [1, 2, 3, 5, 1023, 4095, 4096, 4097, 8192, 8193, 12289, 16385, 40961])
def test_sort(gpu, n, kind):
    from sph_2_amd import libsx

    rng = np.random.default_rng(n)
    pos = rng.random((n, 3))
    if kind == "ties":
        pos = np.floor(pos * 4.0)
    elif kind == "one_point":
        pos[:] = 0.25
    elif kind in ("sorted", "reversed"):
        pos = pos[np.argsort(_keys(pos), kind="stable")]
        if kind == "reversed":
            pos = pos[::-1].copy()
    ref = _keys(pos)
    order = np.argsort(ref, kind="stable")
    keys, perm = libsx.morton_sort(pos)
    assert np.array_equal(perm, order)
    assert np.array_equal(keys, ref[order])
