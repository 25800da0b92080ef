"""Split and renumbering over bits by slot: scenes around the 32-slot words and the 1024-slot
tiles of the bit arrays, one with more slots than a block counts by itself, and splits at the
capacity limit. Every step against the CPU oracle, bit for bit."""
import numpy as np
import pytest

import sca2012_amd as sa
from oracle import orc
from sca2012_amd import scenes

pytestmark = pytest.mark.gpu
FLAGS = sa.STEP_SPLIT | sa.STEP_MERGE
# split and merge criteria at which particles of these scenes do both within four steps
CRITERIA = {sa.V2D: (0.3, 0.25), sa.V3D2: (0.3, 0.6), sa.V3D4: (0.1, 0.2)}


def same(a, b):
    for f in a.dtype.names:
        x, y = a[f], b[f]
        if x.dtype.kind == "f":
            nan = np.isnan(x)
            assert np.array_equal(nan, np.isnan(y)), f
            x, y = x[~nan].view(np.uint32), y[~nan].view(np.uint32)
        assert np.array_equal(x, y), f


def run(variant, p, a, cap, steps):
    with sa.SPHContext(variant, p, cap) as ctx:
        o = orc.Oracle(variant, p, cap)
        ctx.upload(a)
        o.upload(a)
        changed = False
        for _ in range(steps):
            n = ctx.step(FLAGS)
            assert o.step(FLAGS) == 0
            assert n == o.num_particles()
            changed = changed or n != len(a)
            same(ctx.download(), o.download())
            assert np.array_equal(ctx.get_u32(sa._abi.Q_SPLITFLAG), o.get_u32(orc.SPLITFLAG))
            assert np.array_equal(ctx.get_u32(sa._abi.Q_STATUS), o.get_u32(orc.STATUS))
        return changed


@pytest.mark.parametrize("variant", [sa.V2D, sa.V3D2, sa.V3D4])
@pytest.mark.parametrize("n", [1, 31, 32, 33, 1023, 1024, 1025, 1900])
def test_tile_edges(variant, n):
    p, a = scenes.reference_scene(variant)
    a = a[:n].copy()
    a["vel"] = np.random.default_rng(n).uniform(-1.0, 1.0, a["vel"].shape).astype(np.float32)
    names = ("thresh_split", "thresh_merge") if variant == sa.V2D else ("split_criteria", "merge_criteria")
    for name, v in zip(names, CRITERIA[variant]):
        p[name] = v
    run(variant, p, a, 8 * n, 4)  # from 33 particles on the 2D and 3D-2 scenes split and merge


@pytest.mark.parametrize("variant,extra", [(sa.V3D2, 0), (sa.V3D2, 1), (sa.V3D2, 1000), (sa.V3D4, 2),
                                           (sa.V3D4, 3100)])
def test_split_capacity(variant, extra):
    p, a = scenes.reference_scene(variant)
    a = a[:3000].copy()
    p["split_criteria"] = -1.0  # every large particle splits until the capacity is reached
    run(variant, p, a, len(a) + extra, 3)


def test_counts_from_a_scan():
    """One step of 1.05 million particles: the tiles' offsets come from a scan."""
    p, a = scenes.adaptive_3d2(n_side=102, seed=5, cells=104)
    assert len(a) > 1 << 20
    p["split_criteria"], p["merge_criteria"] = 1.0, 0.5
    assert run(sa.V3D2, p, a, 2 * len(a), 2)
