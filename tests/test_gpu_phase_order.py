"""Phase calls in orders other than a step's: parameters changed between integrate (or a step)
and energy, above the counts from which the energy kernel reads quantised positions; a split
between merge and compact. Against the CPU oracle, bit for bit."""
import numpy as np
import pytest

import sca2012_amd as sa
from oracle import orc

from helpers import assert_particles_equal

pytestmark = pytest.mark.gpu


def still_cloud(variant, n, seed):
    """n particles that keep their places and velocities through integrate (a time step of 0)."""
    p = sa.param_defaults(variant)
    r = np.random.default_rng(seed)
    if variant == sa.V2D:
        p["world_width"] = p["world_depth"] = 256.0
        lo, hi = (4.0, 4.0), (252.0, 252.0)
    else:
        p["dens_mul"] = 1
        p["world_width"], p["world_height"], p["world_length"] = 64.0, 32.0, 20.0
        lo, hi = (2.0, 2.0, 2.0), (62.0, 30.0, 18.0)
    sa.param_derive(variant, p)
    p["time_step"] = 0.0
    a = np.zeros(n, dtype=sa.particle_dtype(variant))
    a["pos"] = r.uniform(lo, hi, a["pos"].shape)
    a["vel"] = a["ev"] = r.uniform(-1.0, 1.0, a["vel"].shape)
    a["level"] = 1 + (r.uniform(size=n) < 0.5)
    return p, a


def with_radius(variant, p, size, h):
    """p with another kernel radius of one level, on the same grid."""
    q = p.copy()
    sep = "" if variant == sa.V2D else "_"
    q[size + "_kernel"] = h
    q[size + "_kernel" + sep + "2"] = np.float32(h) ** 2
    q[size + "_kernel" + sep + "6"] = np.float32(h) ** 6
    return q


@pytest.mark.parametrize("before", ["integrate", "step"])
@pytest.mark.parametrize("variant, n", [(sa.V3D2, 180001), (sa.V3D2, 180000), (sa.V3D4, 180001),
                                        (sa.V2D, 128001)])
def test_energy_after_other_radii(variant, n, before):
    p, a = still_cloud(variant, n, n)
    radii = [("small", 0.95), ("small", 0.6), ("large", 0.9)] if variant != sa.V2D else \
            [("small", 0.99), ("small", 0.6), ("large", 0.9)]
    with sa.SPHContext(variant, p, n, max_triangles=1) as g:
        g.upload(a)
        for k, (size, h) in enumerate(radii):
            print("variant", variant, "n", n, before, size, h, flush=True)
            g.set_params(p)
            if before == "step":
                g.step(0)
            else:
                for phase in ("calc_hash", "sort", "cell_ranges", "density", "force", "integrate"):
                    getattr(g, phase)()
            q = with_radius(variant, p, size, h * float(p["large_kernel"][0]))
            g.set_params(q)
            o = orc.Oracle(variant, q, n)
            o.upload(g.download())
            g.energy()
            o.calc_hash()
            o.sort()
            o.cell_ranges()
            o.energy()
            assert_particles_equal(g.download(), o.download(), ["pos", "vel", "energy", "level"],
                                   what="radii %d" % k)
            o.close()


def merge_split_scene(variant, n, seed, n_small, large_splits):
    """Small particles that merge in pairs (or fours) and large ones that split or not."""
    p = sa.param_defaults(variant)
    r = np.random.default_rng(seed)
    names = ("thresh_split", "thresh_merge") if variant == sa.V2D else ("split_criteria", "merge_criteria")
    p[names[0]], p[names[1]] = 10.0, 1.0
    p["co_energy"], p["co_surface"] = 1.0, 0.0
    a = np.zeros(n, dtype=sa.particle_dtype(variant))
    a["pos"] = 2.0 + r.uniform(0.0, 12.0 if variant == sa.V2D else 5.0, a["pos"].shape)
    for f in ("vel", "ev", "acc"):
        a[f] = r.uniform(-1.0, 1.0, a[f].shape)
    a["dens"] = 1.0
    a["level"] = 1 + (r.permutation(n) < n_small)
    a["energy"] = np.where(a["level"] == 2, 0.5, 20.0 if large_splits else 5.0)
    return p, a


@pytest.mark.parametrize("variant", [sa.V2D, sa.V3D2, sa.V3D4])
@pytest.mark.parametrize("n", [700, 1024, 1500, 2300])
def test_split_between_merge_and_compact(variant, n):
    """The children's slots lie past those that the merge saw, in words and 1024-slot tiles that an
    earlier, larger merge has used."""
    cap = 12000
    print("variant", variant, "n", n, flush=True)
    with sa.SPHContext(variant, sa.param_defaults(variant), cap, max_triangles=1) as g:
        for count, small, splits in ((8000, 8000, False), (n, n // 3, True)):
            p, a = merge_split_scene(variant, count, count, small, splits)
            o = orc.Oracle(variant, p, cap)
            g.set_params(p)
            for x in (g, o):
                x.upload(a)
                for phase in ("calc_hash", "sort", "cell_ranges"):
                    getattr(x, phase)()
            groups = g.merge()
            assert groups == o.merge() and groups > 0
            assert g.split() == o.split()
            g.compact()
            o.compact()
            assert not splits or g.num_particles() > n  # more children than removed particles
            assert_particles_equal(g.download(), o.download(), what="%d particles" % count)
            assert np.array_equal(g.get_u32(sa._abi.Q_STATUS)[:count], o.get_u32(orc.STATUS)[:count])
            o.close()
