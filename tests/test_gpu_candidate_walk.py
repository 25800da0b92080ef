"""The one-thread density and energy kernels against the oracle, bit for bit, where their quantised
distance test could lose a pair or their walk an order: runs around and above the 32 candidates of a
word, pairs at the kernel radius to the last bit, particles that leave their cells by more than the
16 cells after which quantised coordinates repeat, a small kernel larger than the large one, and a
batch whose scenes have different steps. The counts are above the rule's lines for these kernels
(Aux::choose_forms)."""
import numpy as np
import pytest

import sca2012_amd as sa
from sca2012_amd import scenes
from oracle import orc

from helpers import assert_particles_equal

pytestmark = pytest.mark.gpu

N = {sa.V2D: 130001, sa.V3D2: 180003, sa.V3D4: 180003}


def base(variant, seed, swap=False):
    """N particles, uniform, about seven per cell (2D: four), of both levels."""
    n = N[variant]
    r = np.random.default_rng(seed)
    p = sa.param_defaults(variant)
    if swap:
        p["small_kernel"], p["large_kernel"] = 1.0, 0.9
    if variant == sa.V2D:
        p["world_width"] = p["world_depth"] = 256.0
        lo, hi = np.array([3.0, 3.0]), np.array([253.0, 130.0])
    else:
        p["dens_mul"] = 1
        p["world_width"], p["world_height"], p["world_length"] = 72.0, 24.0, 24.0
        lo, hi = np.array([2.0, 2.0, 2.0]), np.array([70.0, 22.0, 22.0])
    sa.param_derive(variant, p)
    a = np.zeros(n, dtype=sa.particle_dtype(variant))
    a["pos"] = r.uniform(lo, hi, a["pos"].shape)
    a["vel"] = r.uniform(-1.0, 1.0, a["vel"].shape)
    a["ev"] = r.uniform(-1.0, 1.0, a["ev"].shape)
    a["level"] = 1 + (r.uniform(size=n) < 0.5)
    return p, a, r


def crowd(p, a, r):
    """Cells of 24 to 72 particles, one in every few waves."""
    at = 0
    for k in range(400):
        m = 24 + k % 49
        cell = np.floor(a["pos"][at + m] / p["cell_size"][0]) * p["cell_size"][0]
        a["pos"][at:at + m] = cell + r.uniform(0.05, 0.95, a["pos"][at:at + m].shape) * p["cell_size"][0]
        at += m


def edges(p, a, r):
    """Partners at either kernel radius, up to three floats more or less, along an axis."""
    m = 40000
    h = np.where(np.arange(m) % 2, p["small_kernel"][0], p["large_kernel"][0]).astype(np.float32)
    q = a["pos"][:m].copy()
    ax = np.arange(m) % q.shape[1]
    x = q[np.arange(m), ax] + np.where(q[np.arange(m), ax] > 12.0, -h, h)
    for k in range(3):
        x = np.where(np.arange(m) % 7 > k, np.nextafter(x, np.float32(1e9)), x)
        x = np.where(np.arange(m) % 5 > k, np.nextafter(x, np.float32(-1e9)), x)
    q[np.arange(m), ax] = x
    a["pos"][m:2 * m] = q


def brisk(p, a, r):
    """Steps of up to one and a half cells."""
    a["vel"] = r.uniform(-15.0, 15.0, a["vel"].shape)


def fast(p, a, r):
    """Steps of up to 40 cells."""
    a["vel"] = r.uniform(-400.0, 400.0, a["vel"].shape)


@pytest.mark.parametrize("variant", [sa.V2D, sa.V3D2, sa.V3D4])
@pytest.mark.parametrize("kind", ["crowd", "edges", "brisk", "fast", "swap", "nan"])
def test_one_step(variant, kind):
    p, a, r = base(variant, 7, kind == "swap")
    if kind in ("crowd", "edges", "swap"):  # the energy sees small steps, or the same edges again
        p["time_step"] = 0.0 if kind == "edges" else 0.001
    if kind == "nan":  # a few particles whose velocity is not finite
        a["vel"][::9001] = np.nan
        a["vel"][5::9001, -1] = np.inf
    elif kind != "swap":
        {"crowd": crowd, "edges": edges, "brisk": brisk, "fast": fast}[kind](p, a, r)
    print("variant", variant, kind, flush=True)
    o = orc.Oracle(variant, p, len(a))
    o.upload(a)
    with sa.SPHContext(variant, p, len(a), max_triangles=1) as g:
        g.upload(a)
        g.step(0)
        assert o.step(0) == 0
        assert_particles_equal(g.download(), o.download(), what=kind)


def test_batch_with_different_kernels():
    flags = sa.STEP_SPLIT | sa.STEP_MERGE
    made = []
    for k, h in enumerate((1.0, 0.8, 1.25)):
        p, a = scenes.tank_3d2(62000, scenes.SEED_BASE + 77, k)
        p["large_kernel"], p["small_kernel"] = h, 0.9 * h
        sa.param_derive(sa.V3D2, p)
        made.append((p, a))
    b = sa.SPHBatch(sa.V3D2, [p for p, _ in made], [2 * len(a) for _, a in made])
    for s, (_, a) in enumerate(made):
        b.upload(s, a)
    b.step(flags, steps=2)
    for s, (p, a) in enumerate(made):
        o = orc.Oracle(sa.V3D2, p, 2 * len(a))
        o.upload(a)
        for _ in range(2):
            assert o.step(flags) == 0
        assert_particles_equal(b.download(s), o.download(), what="scene %d" % s)
    b.close()
