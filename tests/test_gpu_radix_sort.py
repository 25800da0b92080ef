"""The radix sort against numpy's stable sort, at the edges of its waves (64 and 256 keys), tiles
and groups of tiles (1024 and 4096 keys; 2048 and 8192 above 131,072; 4096 and 16,384 above 1,048,576,
where a launch of its own adds the groups up), and of its digits (9 bits): spread keys, runs of equal keys, one key only."""
import numpy as np
import pytest

import sca2012_amd as sa

from test_zz_no_alloc import _context_sort, _noalloc, _numpy_stable

pytestmark = pytest.mark.gpu


def make_keys(kind, n, seed):
    r = np.random.default_rng(seed)
    if kind == "spread":
        return r.integers(0, 1 << 32, n, dtype=np.uint64).astype(np.uint32)
    if kind == "runs":  # nearly sorted, as a scene's cells are from step to step
        k = (np.arange(n, dtype=np.uint32) // 7) * np.uint32(2654435)
        return k ^ (r.uniform(size=n) < 0.02).astype(np.uint32)
    return np.full(n, 0xfedcba98, dtype=np.uint32)


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 255, 256, 257, 1023, 1024, 1025, 4095, 4096, 4097,
                               100003, 131072, 131073, 139264, 139265, 1048575, 1048576])
@pytest.mark.parametrize("kind", ["spread", "runs", "one"])
def test_against_a_stable_sort(n, kind):
    keys = make_keys(kind, n, n)
    index = np.random.default_rng(n + 1).integers(0, 1 << 32, n, dtype=np.uint64).astype(np.uint32)
    for bits in (1, 2, 9, 10, 18, 27, 0):
        print("n", n, kind, "bits", bits, flush=True)
        rc, k, v = _noalloc(keys, index, bits)
        assert rc == 0
        k0, v0 = _numpy_stable(keys, index, bits)
        assert np.array_equal(k, k0) and np.array_equal(v, v0)


@pytest.mark.parametrize("n", [1048577, 1300001])
def test_context_sort_above_the_group_line(n):
    p = sa.param_defaults(sa.V2D)
    p["world_width"] = p["world_depth"] = 1024.0
    sa.param_derive(sa.V2D, p)
    a = np.zeros(n, dtype=sa.particle_dtype(sa.V2D))
    a["pos"] = np.random.default_rng(n).uniform(0.5, 1023.5, a["pos"].shape)
    a["level"] = 1
    print("n", n, flush=True)
    keys, h, i, _ = _context_sort(sa.V2D, p, a)
    o = np.argsort(keys, kind="stable")
    assert np.array_equal(i, o.astype(np.uint32)) and np.array_equal(h, keys[o])
    c = np.floor(a["pos"]).astype(np.uint32)
    assert np.array_equal(keys, c[:, 1] * p["row_cell"][0] + c[:, 0])
