"""More kinds of repeated steps than a context keeps captured graphs of (16): the graph that was
unused for longest gives way, and every step equals the same step launched kernel by kernel."""
import numpy as np
import pytest

import sca2012_amd as sa
from sca2012_amd import scenes

from helpers import assert_particles_equal

pytestmark = pytest.mark.gpu


def test_more_kinds_of_steps_than_kept_graphs():
    p, a = scenes.reference_scene(sa.V3D4)
    a["vel"] = np.random.default_rng(5).uniform(-0.5, 0.5, a["vel"].shape).astype(np.float32)
    flags = (0, sa.STEP_SPLIT, sa.STEP_MERGE, sa.STEP_SPLIT | sa.STEP_MERGE)
    with sa.SPHContext(sa.V3D4, p, 100000, max_triangles=1) as g, \
            sa.SPHContext(sa.V3D4, p, 100000, max_triangles=1) as r:
        g.autotune(0)
        r.autotune(0)
        r.prof_enable(True)  # a context that times its phases launches them one by one
        for n in (700, 5000, 20000, 700, 40000, 5000):  # with both buffers: 4 bounds x 4 flags x 2
            for f in flags:
                g.upload(a[:n])
                r.upload(a[:n])
                for k in range(10):
                    assert g.step(f) == r.step(f)
                assert_particles_equal(g.download(), r.download(), what="n %d flags %d" % (n, f))
