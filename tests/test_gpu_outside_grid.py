"""Many particles outside the grid, all of which go to cell 0: the step that finds them counts cells,
the ones after it sort, and the ones after an upload count again. Against the phase calls, which
always sort; a batch's scenes against single scenes."""
import numpy as np
import pytest

import sca2012_amd as sa
from sca2012_amd import scenes

from helpers import assert_particles_equal

pytestmark = pytest.mark.gpu
SM = sa.STEP_SPLIT | sa.STEP_MERGE


def by_phases(g):
    with pytest.raises(sa.SphError) as e:
        g.calc_hash()
    assert e.value.code == sa._abi.EDOMAIN
    for phase in ("sort", "cell_ranges", "density", "force", "integrate", "energy", "split", "merge", "compact"):
        getattr(g, phase)()


def scene(variant, n, seed):
    p, a = scenes.reference_scene(variant)
    a = a[:n].copy()
    r = np.random.default_rng(seed)
    a["vel"] = r.uniform(-0.5, 0.5, a["vel"].shape)
    bad = a.copy()
    bad["pos"][r.permutation(n)[:n // 3]] = np.nan
    return p, a, bad


@pytest.mark.parametrize("variant", [sa.V2D, sa.V3D2, sa.V3D4])
def test_context(variant):
    p, a, bad = scene(variant, 1900, 11)
    with sa.SPHContext(variant, p, 20000, max_triangles=1) as g, \
            sa.SPHContext(variant, p, 20000, max_triangles=1) as r:
        for x in (g, r):
            x.upload(bad)
        for k in range(4):
            assert g.step_raw(SM)[0] == sa._abi.EDOMAIN
            by_phases(r)
            assert_particles_equal(g.download(), r.download(), what="step %d" % k)
        for x in (g, r):  # a scene without them
            x.upload(a)
            x.prof_enable(x is r)  # launched one by one
        for k in range(12):
            assert g.step(SM) == r.step(SM)
        assert_particles_equal(g.download(), r.download(), what="after an upload")


@pytest.mark.parametrize("graph", [False, True])
def test_batch(graph):
    p, a, bad = scene(sa.V3D2, 3000, 12)
    b = sa.SPHBatch(sa.V3D2, [p, p, p], [9000] * 3)
    b.set_graph(graph)
    singles = [sa.SPHContext(sa.V3D2, p, 9000, max_triangles=1) for _ in range(3)]
    for s, x in enumerate((a, bad, a[:500])):
        b.upload(s, x)
        singles[s].upload(x)
    for k in range(3):
        assert b.step_raw(SM)[0] == sa._abi.EDOMAIN
        for s, g in enumerate(singles):
            assert (g.step_raw(SM)[0] == sa._abi.EDOMAIN) == (s == 1)
            assert_particles_equal(b.download(s), g.download(), what="step %d scene %d" % (k, s))
    b.upload(1, a)
    singles[1].upload(a)
    for k in range(3):
        b.step(SM)
        for s, g in enumerate(singles):
            g.step(SM)
            assert_particles_equal(b.download(s), g.download(), what="after an upload, scene %d" % s)
    for g in singles:
        g.close()
    b.close()
