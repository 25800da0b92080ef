"""Steps launched as one captured graph against the same steps launched one by one (a context that
times its phases launches them so), and batches whose scenes are uploaded again between steps."""
import numpy as np
import pytest

import sca2012_amd as sa
from sca2012_amd import scenes

from helpers import assert_particles_equal

pytestmark = pytest.mark.gpu
S, M, MC = sa.STEP_SPLIT, sa.STEP_MERGE, sa.STEP_MC
ARRAYS = (sa._abi.Q_HASH, sa._abi.Q_INDEX, sa._abi.Q_START, sa._abi.Q_END)


def same_state(a, b, what):
    assert_particles_equal(a.download(), b.download(), what=what)
    for q in ARRAYS:
        assert np.array_equal(a.get_u32(q), b.get_u32(q)), what
    # counters: n, m, n_pre, s_req, s_done, groups, err
    assert np.array_equal(a.get_u32(sa._abi.Q_COUNTERS)[:7], b.get_u32(sa._abi.Q_COUNTERS)[:7]), what


@pytest.mark.parametrize("variant,flags", [(sa.V2D, 0), (sa.V2D, S | M), (sa.V3D2, 0), (sa.V3D2, S),
                                           (sa.V3D2, M), (sa.V3D2, S | M), (sa.V3D4, S | M),
                                           (sa.V3D4, S | M | MC)])
def test_captured_steps_equal_single_launches(variant, flags):
    p, a = scenes.reference_scene(variant)
    a = a[:5000].copy()
    a["vel"] = np.random.default_rng(3).uniform(-0.5, 0.5, a["vel"].shape).astype(np.float32)
    with sa.SPHContext(variant, p, 40000, max_triangles=200000) as g, \
            sa.SPHContext(variant, p, 40000, max_triangles=200000) as r:
        g.autotune(0)
        r.autotune(0)
        r.prof_enable(True)
        for n in (len(a), 900, 1):  # the same context with other scenes: another launch bound
            g.upload(a[:n])
            r.upload(a[:n])
            for k in range(12):
                assert g.step(flags) == r.step(flags)
                same_state(g, r, "n %d step %d" % (n, k))
        if flags & MC:
            assert np.array_equal(g.get_f32(sa._abi.Q_TRI), r.get_f32(sa._abi.Q_TRI))
        # phase calls after captured steps
        for c in (g, r):
            c.upload(a)
            for k in range(10):
                c.step(flags)
            c.calc_hash()
            c.sort()
            c.cell_ranges()
            c.density()
            c.force()
            c.integrate()
            c.energy()
            c.split()
            c.merge()
            c.compact()
        same_state(g, r, "phases")


def test_changed_parameters_reach_captured_steps():
    p, a = scenes.reference_scene(sa.V3D2)
    with sa.SPHContext(sa.V3D2, p, 40000) as g, sa.SPHContext(sa.V3D2, p, 40000) as r:
        r.prof_enable(True)
        for c in (g, r):
            c.autotune(0)
            c.upload(a)
        for k in range(30):
            if k % 10 == 9:  # gravity turns, and a one-step push on the last change
                p["gravity"][0] = (0.5 * k, -5.0, 0.0)
                p["flag0"] = k == 29
                g.set_params(p)
                r.set_params(p)
            assert g.step(S | M) == r.step(S | M)
            assert_particles_equal(g.download(), r.download(), what="step %d" % k)


def test_scenes_of_a_batch_uploaded_again():
    sizes = [700, 2100, 1, 3300, 64]
    made = [scenes.tank_3d2(n, scenes.SEED_BASE + 7, k) for k, n in enumerate(sizes)]
    caps = [3 * n for n in sizes]  # so that uploads run out of entries and removed ones are packed away
    b = sa.SPHBatch(sa.V3D2, [p for p, _ in made], caps)
    alone = [sa.SPHContext(sa.V3D2, p, c) for (p, _), c in zip(made, caps)]
    for k, (_, a) in enumerate(made):
        b.upload(k, a)
        alone[k].upload(a)
    rng = np.random.default_rng(11)
    for turn in range(12):
        steps = int(rng.integers(0, 3))
        if steps:
            b.step(S | M, steps=steps)
            for c in alone:
                for _ in range(steps):
                    c.step(S | M)
        for k in rng.permutation(len(sizes))[:int(rng.integers(1, 4))]:
            a = made[k][1][:int(rng.integers(1, sizes[k] + 1))]
            b.upload(int(k), a)
            alone[k].upload(a)
            assert not b.scene_counts()[:, :3].any()
        for k, c in enumerate(alone):
            assert_particles_equal(b.download(k), c.download(), what="turn %d scene %d" % (turn, k))
    for c in alone:
        c.close()
    b.close()
