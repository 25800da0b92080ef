"""The counts on both sides of the lines at which density, force and energy change from several
lanes per particle to one thread (Aux::choose_forms), and the one-thread force kernel at every
list length: over the density pass's pair list, over cells (after parameters were set again), with
lists that overflow, in 2D and in a batch. Against the oracle, bit for bit; the 3D scene above the force
line, 6,000,000, against its own halves, which lie too far apart to interact and stand below it."""
import numpy as np
import pytest

import sca2012_amd as sa
from oracle import orc

from helpers import assert_particles_equal

pytestmark = pytest.mark.gpu
LISTS = (24, 32, 48)


def cloud(variant, n, seed, dense=0):
    """n particles in about 10 to a cell (2D: 12); the first `dense` of them in a few cells."""
    p = sa.param_defaults(variant)
    r = np.random.default_rng(seed)
    h = float(p["large_kernel"][0])
    if variant == sa.V2D:
        p["world_width"] = p["world_depth"] = 256.0
        side = (n / 12.0) ** 0.5
        lo, hi = (4.0, 4.0), (4.0 + side, 4.0 + side)
    else:
        p["dens_mul"] = 1
        edge = np.ceil((n / 10.0) ** (1 / 3)) * h
        p["world_width"] = p["world_height"] = p["world_length"] = edge + 8.0 * h
        lo, hi = (3.0 * h,) * 3, (3.0 * h + edge,) * 3
    sa.param_derive(variant, p)
    a = np.zeros(n, dtype=sa.particle_dtype(variant))
    a["pos"] = r.uniform(lo, hi, a["pos"].shape)
    if dense:  # lists of more than 128 pairs
        a["pos"][:dense] = np.float32(5.0) * h + r.uniform(0.0, 1.2 * h, a["pos"][:dense].shape)
    a["vel"] = a["ev"] = r.uniform(-1.0, 1.0, a["vel"].shape)
    a["level"] = 1 + (r.uniform(size=n) < 0.5)
    return p, a


@pytest.mark.parametrize("variant, n", [(sa.V3D2, 66000), (sa.V3D2, 66001), (sa.V3D4, 66001),
                                        (sa.V3D2, 180000), (sa.V3D2, 180001), (sa.V3D4, 180001),
                                        (sa.V2D, 32000), (sa.V2D, 32001), (sa.V2D, 100000),
                                        (sa.V2D, 100001), (sa.V2D, 128000), (sa.V2D, 128001)])
def test_lines_of_a_context(variant, n):
    p, a = cloud(variant, n, n)
    print("variant", variant, "n", n, flush=True)
    o = orc.Oracle(variant, p, n)
    o.upload(a)
    with sa.SPHContext(variant, p, n, max_triangles=1) as g:
        g.upload(a)
        for k in range(2):
            g.step(0)
            assert o.step(0) == 0
            assert_particles_equal(g.download(), o.download(), what="step %d" % k)


@pytest.mark.parametrize("length", LISTS)
def test_force_lists_2d(length):
    """A pair list, cells with lists that drain several times, and pair lists that overflowed."""
    n = 100001
    p, a = cloud(sa.V2D, n, 31, dense=1500)
    o = orc.Oracle(sa.V2D, p, n)
    o.upload(a)
    with sa.SPHContext(sa.V2D, p, n) as g:
        g.set_lists(length, 16)
        g.upload(a)
        for phase in ("calc_hash", "sort", "cell_ranges", "density", "force"):
            getattr(g, phase)()
            getattr(o, phase)()
        assert_particles_equal(g.download(), o.download(), what="pair list")
        g.set_params(p)  # pair lists made before are not used
        g.force()
        assert_particles_equal(g.download(), o.download(), what="cells")


@pytest.mark.parametrize("variant", [sa.V3D2, sa.V3D4])
def test_force_lists_of_a_batch(variant):
    """Either side of the batch's line (150,000 particles together), every length above it."""
    for n2, lengths in ((49999, (32,)), (50000, (32,)), (50001, LISTS)):
        sizes = (60000, n2, 40000)
        made = [cloud(variant, n, 40 + k, dense=900 if k == 1 else 0) for k, n in enumerate(sizes)]
        refs = []
        for p, a in made:
            o = orc.Oracle(variant, p, 2 * len(a))
            o.upload(a)
            for _ in range(2):
                assert o.step(0) == 0
            refs.append(o.download())
            o.close()
        for length in lengths:
            print("variant", variant, sum(sizes), "list", length, flush=True)
            b = sa.SPHBatch(variant, [p for p, _ in made], [2 * len(a) for _, a in made])
            b.set_lists(length, 16)
            for s, (_, a) in enumerate(made):
                b.upload(s, a)
            b.step(0, steps=2)
            for s, ref in enumerate(refs):
                assert_particles_equal(b.download(s), ref, what="scene %d" % s)
            b.close()


def test_force_above_the_3d_line():
    """6,000,001 particles in two clouds (one thread per particle), and each cloud by itself."""
    n, first = 6000001, 3000400
    p, a = cloud(sa.V3D2, first, 51, dense=900)
    q, b = cloud(sa.V3D2, n - first, 52)
    edge = float(p["world_width"][0])
    p["world_width"] = 2.0 * edge + 8.0
    sa.param_derive(sa.V3D2, p)
    b["pos"][:, 0] += np.float32(np.ceil(edge))
    both = np.concatenate([a, b])

    def phases(g, part):
        g.upload(part)
        for phase in ("calc_hash", "sort", "cell_ranges", "density", "force"):
            getattr(g, phase)()
        out = [g.download()]
        g.set_params(p)  # pair lists made before are not used
        g.force()
        return out + [g.download()]

    with sa.SPHContext(sa.V3D2, p, n, max_triangles=1) as g:
        halves = [phases(g, both[:first]), phases(g, both[first:])]
        for length in LISTS:
            print("list", length, flush=True)
            g.set_lists(length, 16)
            for k, x in enumerate(phases(g, both)):
                what = "list %d, %s" % (length, ("pair list", "cells")[k])
                assert_particles_equal(x[:first], halves[0][k], what=what)
                assert_particles_equal(x[first:], halves[1][k], what=what)
