"""An error that other code left in the calling thread: the call that finds it says so, and the
calls after it answer as if it had not been there. Steps launched one by one and as a captured
graph, against the CPU oracle."""
import numpy as np
import pytest

import sca2012_amd as sa
from oracle import orc
from sca2012_amd import scenes

from helpers import assert_particles_equal

pytestmark = pytest.mark.gpu
SM = sa.STEP_SPLIT | sa.STEP_MERGE


def leave_error(lib):
    assert lib.hipSetDevice(1 << 20) != 0  # no such device: refused on the host


@pytest.mark.parametrize("variant, flags", [(sa.V2D, SM), (sa.V3D2, SM), (sa.V3D2, 0)])
def test_context_step(variant, flags):
    p, a = scenes.reference_scene(variant)
    cap = 8 * len(a)
    o = orc.Oracle(variant, p, cap)
    o.upload(a)
    with sa.SPHContext(variant, p, cap, max_triangles=1) as g:
        g.autotune(0)  # steps that repeat are captured after three launches of a buffer parity
        g.upload(a)
        for k in range(24):
            fault = k in (1, 12, 17, 18)
            if fault:
                leave_error(g.lib)
                with pytest.raises(sa.SphError) as e:
                    g.step(flags)
                assert e.value.code == sa._abi.EHIP
            else:
                g.step(flags)
            assert o.step(flags) == 0
            assert g.num_particles() == o.num_particles() == g.counters()["n"], k
            if fault or k == 23:
                assert_particles_equal(g.download(), o.download(), what="step %d" % k)


def test_flags_read_in_part():
    """Split flags and statuses, kept as bits, read for any number of slots, also right after a
    refused read."""
    p, a = scenes.reference_scene(sa.V3D2)
    cap = 4 * len(a)
    o = orc.Oracle(sa.V3D2, p, cap)
    o.upload(a)
    with sa.SPHContext(sa.V3D2, p, cap, max_triangles=1) as g:
        g.upload(a)
        for _ in range(3):
            g.step(SM)
            assert o.step(SM) == 0
        for q, r in ((sa._abi.Q_SPLITFLAG, orc.SPLITFLAG), (sa._abi.Q_STATUS, orc.STATUS)):
            ref = o.get_u32(r)
            for n in (1, 2, 31, 32, 33, 63, 64, 65, 1023, 1025, len(ref) - 1, len(ref)):
                leave_error(g.lib)
                with pytest.raises(sa.SphError) as e:
                    g.get_u32(q, n)
                assert e.value.code == sa._abi.EHIP
                assert np.array_equal(g.get_u32(q, n), ref[:n]), (q, n)


@pytest.mark.parametrize("graph", [False, True])
def test_batch_step(graph):
    """Also the places of the scenes' particles, which every step moves: they are read right after
    the refused call."""
    sizes = [300, 1200, 77, 2500]
    tanks = [scenes.tank_3d2(int(n), scenes.SEED_BASE + 50, s) for s, n in enumerate(sizes)]
    caps = [4 * n + 8 for n in sizes]
    b = sa.SPHBatch(sa.V3D2, [p for p, _ in tanks], caps)
    b.set_graph(graph)
    oracles = []
    for s, (p, a) in enumerate(tanks):
        o = orc.Oracle(sa.V3D2, p, caps[s])
        o.upload(a)
        b.upload(s, a)
        oracles.append(o)
    for k in range(8):
        fault = k in (0, 3, 6, 7)
        if fault:
            leave_error(b.lib)
            assert b.step_raw(SM, 2 if graph else 1)[0] == sa._abi.EHIP
        else:
            b.step(SM, 2 if graph else 1)
        for o in oracles:
            for _ in range(2 if graph else 1):
                assert o.step(SM) == 0
        assert list(b.num_particles()) == [o.num_particles() for o in oracles]
        for s, o in enumerate(oracles):
            assert_particles_equal(b.download(s), o.download(), what="call %d scene %d" % (k, s))
        if k == 5:  # an upload that follows refused calls
            leave_error(b.lib)
            with pytest.raises(sa.SphError):
                b.upload(1, tanks[1][1])
            b.upload(2, tanks[2][1])
            for s in (1, 2):
                oracles[s].upload(tanks[s][1])
    b.close()
