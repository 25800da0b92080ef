"""Cells of more than 32 particles in the one-thread density and energy kernels, whose walk takes
them in parts of 31 candidates: exact counts around one, two and three parts, spread over the cell
and packed so that every pair interacts (more words than a lane's ring holds), beside sparse
neighbours. Against the oracle, bit for bit, in single scenes and in a batch."""
import numpy as np
import pytest

import sca2012_amd as sa
from oracle import orc

from helpers import assert_particles_equal

pytestmark = pytest.mark.gpu
COUNTS = (30, 31, 32, 33, 34, 61, 62, 63, 64, 65, 92, 93, 94, 125, 300)


def crowded(variant, n, seed):
    """n particles, four to a cell, and clusters of the given counts in cells of their own, every
    third with a second full cell beside it."""
    p = sa.param_defaults(variant)
    r = np.random.default_rng(seed)
    h = float(p["large_kernel"][0])
    dim = 2 if variant == sa.V2D else 3
    made = []
    x = 6
    for k, c in enumerate(COUNTS):
        for packed in (False, True):
            cell = np.array([x, 4 + (k % 3), 5][:dim], dtype=float)
            for side in range(2 if k % 3 == 0 else 1):
                q = r.uniform(0.05, 0.95, (c, dim)) if not packed else 0.5 + r.uniform(-0.2, 0.2, (c, dim))
                q += cell
                q[:, 1] += side
                made.append(q * h)
            x += 4
    pos = np.concatenate(made)
    rest = n - len(pos)
    side = np.ceil((rest / 4.0 / x) ** (1.0 / (dim - 1))) if dim == 3 else np.ceil(rest / 4.0 / x)
    lo = np.array([4.0, 10.0, 10.0][:dim]) * h
    hi = np.array([4.0 + x, 10.0 + side, 10.0 + side][:dim]) * h
    pos = np.concatenate([pos, r.uniform(lo, hi, (rest, dim))])
    names = ("world_width", "world_depth") if dim == 2 else ("world_width", "world_height", "world_length")
    for name, top in zip(names, hi):
        p[name] = top + 4 * h
    if dim == 3:
        p["dens_mul"] = 1
    sa.param_derive(variant, p)
    a = np.zeros(n, dtype=sa.particle_dtype(variant))
    a["pos"] = pos[r.permutation(n)]
    a["vel"] = a["ev"] = r.uniform(-1.0, 1.0, a["vel"].shape)
    a["level"] = 1 + (r.uniform(size=n) < 0.5)
    return p, a


@pytest.mark.parametrize("variant, n", [(sa.V2D, 128001), (sa.V3D2, 180001), (sa.V3D4, 180001)])
def test_context(variant, n):
    p, a = crowded(variant, n, n)
    o = orc.Oracle(variant, p, n)
    o.upload(a)
    print("variant", variant, "n", n, flush=True)
    with sa.SPHContext(variant, p, n, max_triangles=1) as g:
        g.upload(a)
        assert np.array_equal(g.download()["pos"], o.download()["pos"])
        for phase in ("calc_hash", "sort", "cell_ranges", "density", "force", "energy"):
            getattr(g, phase)()
            getattr(o, phase)()
            if phase in ("density", "force", "energy"):
                assert_particles_equal(g.download(), o.download(), what=phase)
        runs = g.get_u32(sa._abi.Q_END).astype(np.int64) - g.get_u32(sa._abi.Q_START)
        assert set(COUNTS) <= set(runs)  # the clusters kept their cells
        g.step(0)
        assert o.step(0) == 0
        assert_particles_equal(g.download(), o.download(), what="step")


@pytest.mark.parametrize("variant", [sa.V3D2, sa.V3D4])
def test_batch(variant):
    made = [crowded(variant, n, k) for k, n in enumerate((60001, 61000, 62003))]
    b = sa.SPHBatch(variant, [p for p, _ in made], [len(a) for _, a in made])
    print("batch", variant, flush=True)
    for s, (_, a) in enumerate(made):
        b.upload(s, a)
    b.step(0)
    for s, (p, a) in enumerate(made):
        o = orc.Oracle(variant, p, len(a))
        o.upload(a)
        assert o.step(0) == 0
        assert_particles_equal(b.download(s), o.download(), what="scene %d" % s)
        o.close()
    b.close()
