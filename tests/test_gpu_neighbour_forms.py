"""The neighbour kernels' two forms (one thread per particle, several lanes per particle)
against the oracle, bit for bit, at the sizes where the lanes' split can go wrong: particle
counts around a wave's and a block's share (7, 8, 28, 32), runs longer than a 64-bit mask,
pair lists past their 128 entries, energy lists of more than one window, and counts on both
sides of the rule that picks the form."""
import numpy as np
import pytest

import sca2012_amd as sa
from sca2012_amd import scenes
from oracle import orc

from helpers import assert_particles_equal

pytestmark = pytest.mark.gpu

VARIANTS = [sa.V2D, sa.V3D2, sa.V3D4]


def cloud(variant, n, extent, seed, levels=True):
    """n particles, uniform in a cube (square) of the given extent away from the walls."""
    r = np.random.default_rng(seed)
    p = sa.param_defaults(variant)
    a = np.zeros(n, dtype=sa.particle_dtype(variant))
    a["pos"] = 5.0 + r.uniform(0.0, extent, a["pos"].shape)
    a["vel"] = r.uniform(-1.0, 1.0, a["vel"].shape)
    a["ev"] = r.uniform(-1.0, 1.0, a["ev"].shape)
    a["level"] = 1 + (r.uniform(size=n) < 0.5) if levels else 1
    return p, a


def compare_phases(variant, p, a, cap):
    o = orc.Oracle(variant, p, cap)
    o.upload(a)
    with sa.SPHContext(variant, p, cap, max_triangles=1) as g:
        g.upload(a)
        # the force phase reads density's pair list, then, asked again after integrate, walks
        # the cells; density and energy after integrate see positions outside their cells
        for phase in ("calc_hash", "sort", "cell_ranges", "density", "force", "integrate", "energy",
                      "density", "force", "energy"):
            getattr(g, phase)()
            getattr(o, phase)()
            if phase not in ("calc_hash", "sort", "cell_ranges"):
                assert_particles_equal(g.download(), o.download(), what="after " + phase)


@pytest.mark.parametrize("variant", VARIANTS)
@pytest.mark.parametrize("n", [1, 2, 6, 7, 8, 9, 27, 28, 29, 31, 32, 33, 63, 64, 65, 223, 225, 257])
def test_small_counts(variant, n):
    p, a = cloud(variant, n, 2.0 + 0.5 * n ** (1 / 3), n)
    print("variant", variant, "n", n, flush=True)
    compare_phases(variant, p, a, 2 * n + 8)


@pytest.mark.parametrize("variant", VARIANTS)
@pytest.mark.parametrize("n, extent", [(150, 1.0), (700, 2.5), (1500, 1.5)])
def test_crowded_cells(variant, n, extent):
    """Runs of more than 64 entries, lists of more than 128 pairs, several energy windows."""
    p, a = cloud(variant, n, extent, 100 + n)
    print("variant", variant, "n", n, "extent", extent, flush=True)
    compare_phases(variant, p, a, n)


@pytest.mark.parametrize("variant, n", [(sa.V2D, 31999), (sa.V2D, 32001), (sa.V2D, 100001),
                                        (sa.V2D, 128001), (sa.V3D2, 99999), (sa.V3D2, 100001),
                                        (sa.V3D2, 180001), (sa.V3D4, 100001)])
def test_both_sides_of_the_rule(variant, n):
    """One step at counts next to the rule's lines (Aux::choose_forms)."""
    p = sa.param_defaults(variant)
    r = np.random.default_rng(n)
    if variant == sa.V2D:
        p["world_width"] = p["world_depth"] = 256.0
        lo, hi = (4.0, 4.0), (4.0 + 0.0018 * n, 124.0)
    else:
        p["dens_mul"] = 1
        p["world_width"], p["world_height"], p["world_length"] = 64.0, 32.0, 20.0
        lo, hi = (2.0, 2.0, 2.0), (62.0, 30.0, 2.0 + 7e-5 * n)
    sa.param_derive(variant, p)
    a = np.zeros(n, dtype=sa.particle_dtype(variant))
    a["pos"] = r.uniform(lo, hi, a["pos"].shape)
    a["vel"] = r.uniform(-1.0, 1.0, a["vel"].shape)
    a["level"] = 1 + (r.uniform(size=n) < 0.5)
    print("variant", variant, "n", n, flush=True)
    o = orc.Oracle(variant, p, 2 * n)
    o.upload(a)
    with sa.SPHContext(variant, p, 2 * n, max_triangles=1) as g:
        g.upload(a)
        g.step(0)
        assert o.step(0) == 0
        assert_particles_equal(g.download(), o.download(), what="one step")


def test_batch_of_small_scenes():
    """Scenes of a few particles: a wave holds several scenes' particles."""
    sizes = [1, 3, 7, 8, 30, 64, 129, 500]
    made = [cloud(sa.V3D2, n, 1.0 + n ** (1 / 3), n, levels=False) for n in sizes]
    caps = [2 * n + 2 for n in sizes]
    flags = sa.STEP_SPLIT | sa.STEP_MERGE
    b = sa.SPHBatch(sa.V3D2, [p for p, _ in made], caps)
    for s, (_, a) in enumerate(made):
        b.upload(s, a)
    b.step(flags, steps=4)
    for s, (p, a) in enumerate(made):
        o = orc.Oracle(sa.V3D2, p, caps[s])
        o.upload(a)
        for _ in range(4):
            assert o.step(flags) == 0
        assert_particles_equal(b.download(s), o.download(), what="scene %d" % s)
    b.close()
