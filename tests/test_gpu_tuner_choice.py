"""What the pair-list tuners do where a length reaches no kernel: one time stands for every
length and the lengths stay; where it does, every length is timed."""
import numpy as np
import pytest

import sca2012_amd as sa
from sca2012_amd import scenes

from test_gpu_phase_order import still_cloud

pytestmark = pytest.mark.gpu
SM = sa.STEP_SPLIT | sa.STEP_MERGE


@pytest.mark.parametrize("variant", [sa.V2D, sa.V3D2, sa.V3D4])
@pytest.mark.parametrize("lengths", [(32, 16), (48, 24)])
def test_context_without_lists(variant, lengths):
    p, a = scenes.reference_scene(variant)
    with sa.SPHContext(variant, p, 8 * len(a), max_triangles=1) as g:
        g.upload(a)
        g.set_lists(*lengths)
        g.autotune(3, after=1, every=12)
        for _ in range(40):
            g.step(SM)
        f, e, best = g.tuned_lists()
        assert (f, e) == lengths
        for k in ("force", "energy"):
            assert min(best[k].values()) > 0 and len(set(best[k].values())) == 1, best


def test_context_with_lists():
    p, a = still_cloud(sa.V2D, 100001, 7)
    with sa.SPHContext(sa.V2D, p, 100001, max_triangles=1) as g:
        g.upload(a)
        g.autotune(2, after=1, every=12)
        for _ in range(30):
            g.step(0)
        _, e, best = g.tuned_lists()
        assert e == 16 and len(set(best["energy"].values())) == 1
        assert min(best["force"].values()) > 0 and len(set(best["force"].values())) == 3


@pytest.mark.parametrize("graph", [False, True])
def test_batch_without_lists(graph):
    sizes = [300, 1200, 77, 2500]
    tanks = [scenes.tank_3d2(int(n), scenes.SEED_BASE + 60, s) for s, n in enumerate(sizes)]
    b = sa.SPHBatch(sa.V3D2, [p for p, _ in tanks], [4 * n + 8 for n in sizes])
    b.set_graph(graph)
    for s, (_, a) in enumerate(tanks):
        b.upload(s, a)
    b.set_lists(24, 32)
    b.autotune(6 if graph else 2, after=1, every=12)
    for _ in range(45):
        b.step(SM)
    f, e, best = b.tuned_lists()
    assert (f, e) == (24, 32)
    for k in ("force", "energy"):
        assert min(best[k].values()) > 0 and len(set(best[k].values())) == 1, best
    b.close()
