"""The work that this framework's users have it do, as cases that a benchmark can time.

A case is a dict of plain values. `prepare` makes what a program holds before the call (the
scene's records in pinned host memory, the context, batch or rollout handle), `run` is one
pass through the public entry points with its whole result, `work` what a pass cannot do
without and `exact` the result in 64 bits where one step or a short smooth rollout has one.

A pass starts every time from the same particle records (an episode: upload, steps, read
back), because a scene that kept moving between passes would be another amount of work in
each of them.

Kinds and the ranges that `draw` spreads over:
  frame    one step of the reference application's start-up scenes (2D, 1->2, 1->4) with the
           full readback that it makes after each step; 200 particles up to the whole scene,
           split, merge and the surface mesh on or off
  dam2d    2D dam breaks, 12^2 to 256^2 particles, 10 to 100 steps between readbacks
  dam      3D 1->2 dam breaks, 6^3 to 64^3 particles before splitting, a mesh every 10 steps
  collide  3D 1->4 collisions, two blocks of 12^3 to 128^3 particles on a sparse grid
  batch    1 to 256 independent tanks of 512 to 65,536 particles stepped together
  rollout  differentiable rollouts, 6^3 to 32^3 particles, forward and backward
  sort     the allocation-free key sort on device arrays, 1,000 to 1,048,576 keys
"""
import ctypes
import math

import numpy as np
import torch

import sca2012_amd as sa
from sca2012_amd import _abi, scenes

SPLIT, MERGE, MESH = sa.STEP_SPLIT, sa.STEP_MERGE, sa.STEP_MC


# ---------------------------------------------------------------------------------------
# cases
# ---------------------------------------------------------------------------------------
def listed():
    return [
        # The application's frame: one step, every particle read back. The smallest calls;
        # launches and host round trips are most of them.
        dict(name="frame_2d", kind="frame", variant=sa.V2D, n=1953, flags=SPLIT | MERGE),
        dict(name="frame_3d2", kind="frame", variant=sa.V3D2, n=7220, flags=0),
        # The same frame in the display mode that draws the fluid's surface.
        dict(name="frame_3d4_mesh", kind="frame", variant=sa.V3D4, n=41850, flags=MESH),
        # Plain 2D dam break of 64 x 64 particles, read back every 50 steps.
        dict(name="dam_2d", kind="dam2d", side=64, steps=50, flags=0),
        # A small 3D scene run as an animation with splitting and merging.
        dict(name="scene_3d2", kind="dam", side=19, cells=24, steps=50, lead=0, flags=SPLIT | MERGE,
             mesh_every=0),
        # The benchmark's scene: a dam break of 64^3 particles, split to about 500,000 when
        # the pass begins, its surface meshed every 10th step.
        dict(name="dam_262k", kind="dam", side=64, cells=64, steps=30, lead=20, flags=SPLIT | MERGE,
             mesh_every=10),
        # The largest scene: two 128^3 blocks collide on 512^3 cells.
        dict(name="collide_4m", kind="collide", side=128, cells=512, steps=10, flags=SPLIT | MERGE,
             mesh_every=10),
        # Many tanks at once, as a program that generates or searches over trajectories steps
        # them: a few uneven ones, and the 256 that a batch holds.
        dict(name="batch_12", kind="batch", tanks=12, n_min=2048, n_max=65536, steps=20,
             flags=SPLIT | MERGE),
        dict(name="batch_256", kind="batch", tanks=256, n_min=2048, n_max=16384, steps=10,
             flags=SPLIT | MERGE),
        # Learning a force field: forward and backward of a short rollout kept on the tape, and
        # of a longer adaptive one replayed from checkpoints.
        dict(name="rollout_4k", kind="rollout", side=16, steps=20, checkpoint=0, flags=0, nodes=8,
             samples=32),
        dict(name="rollout_32k", kind="rollout", side=32, steps=40, checkpoint=20,
             flags=SPLIT | MERGE, nodes=8, samples=64),
        # Sorting by cell key in a program that must not allocate.
        dict(name="sort_700k", kind="sort", n=700001, bits=27),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


_SCENE_N = {sa.V2D: 1953, sa.V3D2: 7220, sa.V3D4: 41850}


def draw(rng):
    kind = rng.choice(["frame", "dam2d", "dam", "collide", "batch", "rollout", "sort"])
    adaptive = rng.choice([0, SPLIT, MERGE, SPLIT | MERGE, SPLIT | MERGE])
    if kind == "frame":
        v = rng.choice([sa.V2D, sa.V3D2, sa.V3D4])
        mesh = MESH if v != sa.V2D and rng.random() < 0.4 else 0
        return dict(kind=kind, variant=v, n=_log(rng, 200, _SCENE_N[v]), flags=adaptive | mesh)
    if kind == "dam2d":
        return dict(kind=kind, side=_log(rng, 12, 256), steps=rng.randint(10, 100), flags=adaptive)
    if kind == "dam":
        side = _log(rng, 6, 64)
        return dict(kind=kind, side=side, cells=side + rng.randint(2, 2 + side // 4),
                    steps=rng.randint(4, 30), lead=rng.choice([0, 20]), flags=adaptive,
                    mesh_every=rng.choice([0, 10]))
    if kind == "collide":
        side = _log(rng, 12, 100)
        return dict(kind=kind, side=side, cells=4 * side + rng.randint(8, 40), steps=rng.randint(3, 10),
                    flags=adaptive, mesh_every=rng.choice([0, 10]))
    if kind == "batch":
        tanks = _log(rng, 1, 256)
        lo = _log(rng, 512, 4096)
        hi = _log(rng, lo, min(65536, max(2 * lo, 2000000 // tanks)))
        return dict(kind=kind, tanks=tanks, n_min=lo, n_max=hi, steps=rng.randint(4, 20),
                    flags=adaptive)
    if kind == "rollout":
        return dict(kind=kind, side=_log(rng, 6, 32), steps=rng.randint(4, 40),
                    checkpoint=rng.choice([0, 7, 20]), flags=adaptive, nodes=rng.randint(2, 11),
                    samples=rng.choice([16, 33, 64]))
    return dict(kind=kind, n=_log(rng, 1000, 1 << 20), bits=rng.randint(10, 32))


# ---------------------------------------------------------------------------------------
# scenes
# ---------------------------------------------------------------------------------------
def _scene(case, seed):
    """(variant, SysParam, records, capacity, most triangles) of a single-scene case."""
    r = np.random.default_rng(seed)
    kind = case["kind"]
    tri = 0
    if kind == "frame":
        variant = case["variant"]
        p, a = scenes.reference_scene(variant)
        a = a[:case["n"]].copy()
        a["vel"] = r.uniform(-0.5, 0.5, a["vel"].shape).astype(np.float32)
        a["ev"] = a["vel"]
        cap = 8 * len(a)
        tri = 400000
    elif kind == "dam2d":
        # the reference's units: h = 1, a block of spacing h/2 in the low corner of a box twice
        # as long and one and a half times as high
        variant, side = sa.V2D, case["side"]
        p = sa.param_defaults(variant)
        p["world_width"], p["world_depth"] = side, 0.75 * side
        sa.param_derive(variant, p)
        a = np.zeros(side * side, dtype=sa.particle_dtype(variant))
        q = 0.5 + 0.5 * np.arange(side)
        X, Y = np.meshgrid(q, q, indexing="ij")
        a["pos"] = np.stack([X.ravel(), Y.ravel()], 1) + r.uniform(0.0, 0.05, (len(a), 2))
        a["level"] = 1
        cap = 4 * len(a)
    elif kind == "dam":
        variant = sa.V3D2
        p, a = scenes.adaptive_3d2(n_side=case["side"], seed=seed, cells=case["cells"])
        cap = 1000000 if len(a) > 125000 else 4 * len(a)
        tri = 1500000 if case["mesh_every"] else 1
    else:
        variant = sa.V3D4
        p, a = scenes.adaptive_3d4_collide(n_side=case["side"], seed=seed, cells=case["cells"])
        cap = 2 * len(a)
        tri = 4000000 if case["mesh_every"] else 1
    return variant, p, a, cap, tri


def _pinned(nbytes):
    return torch.zeros(max(int(nbytes), 16), dtype=torch.uint8, pin_memory=True).numpy()


def _records(a):
    """The records in pinned host memory, as a program that uploads often keeps them."""
    buf = _pinned(a.nbytes)[:a.nbytes].view(a.dtype)
    buf[:] = a
    return buf


def _fields(variant, buf, n):
    """The fields of all n records of the buffer as plain arrays (views)."""
    if variant == sa.V2D:
        w, cols = 14, [("pos", 0, 2), ("vel", 2, 4), ("ev", 4, 6), ("acc", 6, 8), ("dens", 8, 9),
                       ("pres", 9, 10), ("energy", 10, 11), ("surface", 12, 13)]
        lev = 11
    else:
        w, cols = 18, [("pos", 0, 3), ("vel", 3, 6), ("ev", 6, 9), ("acc", 9, 12), ("dens", 12, 13),
                       ("press", 13, 14), ("energy", 14, 15), ("surface", 15, 16), ("tension", 16, 17)]
        lev = 17
    f = buf[:4 * w * n].view(np.float32).reshape(n, w)
    out = {name: f[:, lo:hi] for name, lo, hi in cols}
    out["level"] = buf[:4 * w * n].view(np.int32).reshape(n, w)[:, lev]
    return out


def _most(variant, a):
    """Records that a pass can end with: a level-1 particle splits once, in two (2D, 1->2) or
    four; merging only undoes that."""
    return len(a) + int((a["level"] == 1).sum()) * (3 if variant == sa.V3D4 else 1)


def _ok(code):
    if code != 0:
        raise sa.SphError(code, "pass")


# ---------------------------------------------------------------------------------------
# prepare and run
# ---------------------------------------------------------------------------------------
def _step_flags(case, k):
    every = case.get("mesh_every", 0)
    return case["flags"] | (MESH if every and (k + 1) % every == 0 else 0)


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case, "kind": kind}
    if kind in ("frame", "dam2d", "dam", "collide"):
        variant, p, a, cap, tri = _scene(case, seed)
        ctx = sa.SPHContext(variant, p, cap, max_triangles=tri)
        if case.get("lead"):
            ctx.upload(a)
            for k in range(case["lead"]):
                ctx.step(case["flags"])
            a = ctx.download()
        most = _most(variant, a)
        s.update(variant=variant, ctx=ctx, start=_records(a), most=most,
                 out=_pinned(most * a.dtype.itemsize))
        if variant != sa.V2D and tri > 1:
            s["mesh"] = _pinned(tri * 72).view(np.float32)
    elif kind == "batch":
        sizes = _tank_sizes(case)
        made = [scenes.tank_3d2(n, seed, k) for k, n in enumerate(sizes)]
        s.update(batch=sa.SPHBatch(sa.V3D2, [p for p, _ in made], [3 * n for n in sizes]),
                 start=[_records(a) for _, a in made], most=2 * sum(sizes),
                 out=_pinned(72 * 2 * sum(sizes)))
    elif kind == "rollout":
        p, a, theta, target = _rollout_inputs(case, seed)
        adj = sa.SPHAdjoint(p, len(a), case["nodes"], case["samples"], case["checkpoint"],
                            case["flags"])
        adj.set_target(torch.from_numpy(target).cuda())
        s.update(adj=adj, start=_records(a), theta=torch.from_numpy(theta).cuda(),
                 most=2 * len(a), out=_pinned(2 * a.nbytes), sample=torch.empty(case["samples"] ** 3, device="cuda"),
                 dtheta=torch.empty(theta.size, device="cuda"))
    else:
        r = np.random.default_rng(seed)
        keys = r.integers(0, 1 << case["bits"], case["n"], dtype=np.uint64).astype(np.uint32)
        s.update(keys=torch.from_numpy(keys.view(np.int32)).cuda(),
                 index=torch.arange(case["n"], dtype=torch.int32, device="cuda"),
                 k=torch.empty(case["n"], dtype=torch.int32, device="cuda"),
                 v=torch.empty(case["n"], dtype=torch.int32, device="cuda"))
    return s


def run(s):
    return {"frame": _run_scene, "dam2d": _run_scene, "dam": _run_scene, "collide": _run_scene,
            "batch": _run_batch, "rollout": _run_rollout, "sort": _run_sort}[s["kind"]](s)


def _run_scene(s):
    case, ctx = s["case"], s["ctx"]
    ctx.upload(s["start"])
    n, meshed = 0, False
    for k in range(case.get("steps", 1)):
        flags = _step_flags(case, k)
        n = ctx.step(flags)
        meshed = meshed or bool(flags & MESH)
    assert n <= s["most"]
    _ok(ctx.lib.sph_download_particles(ctx.h, s["out"].ctypes.data, n))
    got = dict(_fields(s["variant"], s["out"], s["most"]), n=n)  # zeros past the n records
    if meshed:  # the last mesh made
        m = ctx.count(_abi.Q_TRI)
        _ok(ctx.lib.sph_get_f32(ctx.h, _abi.Q_TRI, s["mesh"].ctypes.data, m))
        got.update(mesh=s["mesh"], triangles=m // 18)
    return got


def _run_batch(s):
    case, b = s["case"], s["batch"]
    for k, a in enumerate(s["start"]):
        b.upload(k, a)
    b.step(case["flags"], steps=case["steps"])
    at, base = 0, s["out"].ctypes.data
    sizes = b.num_particles()
    assert int(sizes.sum()) <= s["most"]
    for k, n in enumerate(sizes):
        _ok(b.lib.sph_batch_download(b.h, k, base + 72 * at, int(n)))
        at += int(n)
    return dict(_fields(sa.V3D2, s["out"], s["most"]), sizes=sizes.astype(np.int64),
                counts=b.scene_counts())


def _run_rollout(s):
    case, adj = s["case"], s["adj"]
    adj.upload(s["start"])
    loss = adj.forward(s["theta"], case["steps"], s["sample"])
    adj.backward(s["dtheta"])
    g = adj.state_grad()
    n = adj.num_particles()
    assert n <= s["most"]
    _ok(adj.lib.sph_adj_download(adj.h, s["out"].ctypes.data, n))
    return dict(_fields(sa.V3D2, s["out"], s["most"]), n=n, loss=np.float32(loss), sample=s["sample"],
                dtheta=s["dtheta"], dpos=g[0], dvel=g[1], dev=g[2])


def _run_sort(s):
    case = s["case"]
    s["k"].copy_(s["keys"])
    s["v"].copy_(s["index"])
    _ok(sa.load_library().sph_sort_noalloc(
        ctypes.c_void_p(s["k"].data_ptr()), ctypes.c_void_p(s["v"].data_ptr()), case["n"],
        case["bits"], ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
    return {"keys": s["k"], "index": s["v"]}


def _tank_sizes(case):
    """Log-uniform sizes, unevenly ordered, the same for every seed (so is the result's size)."""
    lo, hi, k = math.log(case["n_min"]), math.log(case["n_max"]), case["tanks"]
    sizes = [int(round(math.exp(lo + (hi - lo) * (i + 0.5) / k))) for i in range(k)]
    return [sizes[i] for i in np.random.default_rng(k).permutation(k)]


def _rollout_inputs(case, seed):
    n = case["side"]
    p, a = scenes.rollout_block(n_side=n, seed=seed, box=(n + max(4, n // 2), max(8, n), max(8, n)),
                                time_step=0.01)
    r = np.random.default_rng(seed)
    theta = r.uniform(-1.0, 1.0, case["nodes"] ** 3 * 3).astype(np.float32)
    # the density to reach: the fluid gathered in the box's far half
    m = case["samples"]
    t = np.zeros((m, m, m), dtype=np.float32)  # z, y, x
    t[:, :m // 2, m // 2:] = r.uniform(0.8, 1.2, (m, m // 2, m - m // 2)).astype(np.float32)
    return p, a, theta, t.reshape(-1)


# ---------------------------------------------------------------------------------------
# work
# ---------------------------------------------------------------------------------------
# A step reads and writes each particle's position, velocity, ev and slot (52 bytes) and
# writes acceleration, density, pressure and energy (28). Interacting pairs per particle: about
# 30 in 3D and 14 in 2D, and each costs a density term (15 operations), a force term (60) and
# an energy term (50).
def work(case):
    kind = case["kind"]
    if kind == "sort":
        return {"bytes": 2 * 8 * case["n"] + 2 * 8 * case["n"], "flops": 0}
    if kind == "rollout":
        n, t = case["side"] ** 3, case["steps"]
        grown = 1.5 if case["flags"] & SPLIT else 1.0
        # forward, and a backward that reads each step's state and pairs once more
        steps = t * (3 if case["checkpoint"] else 2)
        return {"bytes": 132 * n * grown * steps + 8 * case["samples"] ** 3,
                "flops": 30 * 125 * n * grown * steps}
    if kind == "batch":
        lo, hi = case["n_min"], case["n_max"]
        mean = (hi - lo) / math.log(hi / lo) if hi > lo else lo
        n, grown, steps, pairs = mean * case["tanks"], 1.8 if case["flags"] & SPLIT else 1.0, case["steps"], 30
        rec = 72
    else:
        pairs = 30
        rec = 72
        steps = case.get("steps", 1)
        grown = 1.0
        if kind == "frame":
            n = case["n"]
        elif kind == "dam2d":
            n, pairs, rec = case["side"] ** 2, 14, 56
        elif kind == "dam":
            n, grown = case["side"] ** 3, 1.9 if case["flags"] & SPLIT else 1.0
        else:
            n = 2 * case["side"] ** 3
        if kind == "frame" and case["variant"] == sa.V2D:
            pairs, rec = 14, 56
    return {"bytes": n * grown * (132 * steps + rec) + rec * n, "flops": n * grown * steps * pairs * 125}


# ---------------------------------------------------------------------------------------
# exact: one step of a frame, and short rollouts without splitting, in 64 bits. Many steps
# of a splashing scene have no such value: nearby trajectories part within ten steps.
# ---------------------------------------------------------------------------------------
def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _pairs(xi, xj, lim2, extra=None):
    """(i, j) with |xi - xj|^2 < lim2, by chunks; extra(i0, i1) may narrow them."""
    ii, jj = [], []
    step = max(1, 20000000 // max(1, len(xj)))
    for i0 in range(0, len(xi), step):
        i1 = min(len(xi), i0 + step)
        d2 = torch.zeros(i1 - i0, len(xj), dtype=torch.float64, device=xi.device)
        for c in range(xi.shape[1]):
            d2 += (xi[i0:i1, c:c + 1] - xj[None, :, c]) ** 2
        ok = d2 < lim2
        if extra is not None:
            ok &= extra(i0, i1)
        i, j = ok.nonzero(as_tuple=True)
        ii.append(i + i0)
        jj.append(j)
    return torch.cat(ii), torch.cat(jj)


class _Exact3D:
    """The 3D step without splitting and merging, from its formulas, in float64."""

    def __init__(self, p, variant, level):
        g = {k: p[k][0] for k in p.dtype.names}
        d = _device()
        L = (level != 1).long()

        def per(a, b):
            return torch.tensor([float(g[a]), float(g[b])], dtype=torch.float64, device=d)
        h = per("large_kernel", "small_kernel")
        pi = 3.141592
        self.L, self.h, self.m, self.rad = L, h, per("large_mass", "small_mass"), per("large_radius", "small_radius")
        self.poly6 = 315 / (64 * pi * h ** 9)
        self.spiky, self.visco = -45 / (pi * h ** 6), 45 / (pi * h ** 6)
        self.grad, self.lap = -945 / (32 * pi * h ** 9), -945 / (8 * pi * h ** 9)
        self.p6r = 315 / (64 * pi * self.rad ** 9)
        self.dt, self.mu = float(g["time_step"]), float(g["viscosity"])
        self.rho0, self.k = float(g["rest_density"]), float(g["gas_constant"])
        self.sigma, self.damp = float(g["surface_tension"]), float(g["wall_damping"])
        self.cs = 0.02 if variant == sa.V3D4 else 0.1
        self.variant = variant
        self.cell = float(g["cell_size"])
        self.gravity = torch.tensor([float(v) for v in g["gravity"]], dtype=torch.float64, device=d)
        self.world = torch.tensor([float(g[k]) for k in ("world_width", "world_height", "world_length")],
                                  dtype=torch.float64, device=d)
        self.h2max = float(torch.max(h[L]) ** 2)

    def forces(self, x, ev):
        h, L, m = self.h, self.L, self.m
        with torch.no_grad():
            i, j = _pairs(x, x, self.h2max)
            far = ((x[i] - x[j]) ** 2).sum(1) >= 1e-4
            i, j = i[far], j[far]
        n = len(x)
        hi, hj, mi, mj = h[L[i]], h[L[j]], m[L[i]], m[L[j]]
        u = x[i] - x[j]
        r2 = (u * u).sum(1)
        r = r2.sqrt()
        zero = torch.zeros_like(r2)
        rho = self.m[L] * self.poly6[L] * h[L] ** 6
        rho = rho.index_add(0, i, torch.where(r2 < hi * hi, mj * self.poly6[L[i]] * (hi * hi - r2) ** 3, zero))
        press = ((rho / self.rho0) ** 3 - 1) * self.k
        oni, onj = hi - r > 0, hj - r > 0
        wp = torch.where(oni, self.spiky[L[i]] * (hi - r) ** 2 / hi ** 6, zero) + \
            torch.where(onj, self.spiky[L[j]] * (hj - r) ** 2 / hj ** 6, zero)
        wv = torch.where(oni, self.visco[L[i]] / hi ** 6 * (hi - r), zero) + \
            torch.where(onj, self.visco[L[j]] / hj ** 6 * (hj - r), zero)
        tp = mi * mj * (press[i] / rho[i] ** 2 + press[j] / rho[j] ** 2) * wp / 2
        tv = (mi / rho[i]) * (mj / rho[j]) * self.mu * wv / 2
        f = torch.zeros_like(x).index_add(0, i, -u * (tp / r)[:, None] + (ev[j] - ev[i]) * tv[:, None])
        d = hi * hi - r2
        cg = torch.where(oni, -self.grad[L[i]] * mj / rho[j] * d * d, zero)
        g = torch.zeros_like(x).index_add(0, i, cg[:, None] * u)
        lap = torch.zeros(n, dtype=x.dtype, device=x.device).index_add(
            0, i, torch.where(oni, self.lap[L[i]] * mj / rho[j] * d * r2, zero))
        g2 = (g * g).sum(1)
        on = (g2 > self.sigma ** 2)
        nrm = torch.where(on, g2, torch.ones_like(g2)).sqrt()
        f = f + torch.where(on, self.cs * lap / nrm, torch.zeros_like(lap))[:, None] * g
        return rho, press, f, g2.detach().sqrt()

    def integrate(self, x, v, ev, rho, f):
        v = v + (f + self.gravity) * self.dt / rho[:, None]
        x = x + v * self.dt
        rad = self.rad[self.L][:, None]
        top = self.world - rad
        hit = x.detach() >= top
        v = torch.where(hit, v * self.damp, v)
        x = torch.where(hit, top.expand_as(x), x)
        hit = x.detach() < rad
        v = torch.where(hit, v * self.damp, v)
        x = torch.where(hit, rad.expand_as(x), x)
        return x, v, (ev + v) / 2

    def energy(self, x0, x, v):
        """Neighbours: the cells around the new position in the step's first cell lists."""
        c0, c1 = (x0 / self.cell).floor(), (x / self.cell).floor()
        k = float(self.h[0])

        def near(i0, i1):
            ok = torch.ones(i1 - i0, len(x), dtype=torch.bool, device=x.device)
            for c in range(3):
                ok &= (c1[i0:i1, c:c + 1] - c0[None, :, c]).abs() <= 1
            return ok
        i, j = _pairs(x, x, k * k, near)
        far = ((x[i] - x[j]) ** 2).sum(1) >= 1e-4
        i, j = i[far], j[far]
        a = 2 / (3.141592 ** 0.25 * 6 ** 0.5)
        out = torch.zeros(len(x), dtype=x.dtype, device=x.device)
        for c in range(2):
            q = ((x[i, c] - x[j, c]) / k) ** 2
            w = a * (q / 4 - 1) * torch.pow(torch.tensor(2.718281, dtype=x.dtype, device=x.device), -q / 8)
            num = torch.zeros_like(out).index_add(0, i, v[j, c] * w / k ** 0.5)
            den = torch.zeros_like(out).index_add(0, i, w)
            out = out + (num / den) ** 2
        return 0.5 * out * (self.m[self.L] if self.variant == sa.V3D4 else 1.0)


def exact(case, seed):
    if case["kind"] == "frame" and case["variant"] != sa.V2D and not case["flags"] & (SPLIT | MERGE):
        return _exact_frame(case, seed)
    if case["kind"] == "rollout" and not case["flags"] and case["side"] ** 3 * case["steps"] <= 100000:
        return _exact_rollout(case, seed)
    return None


def _exact_frame(case, seed):
    variant, p, a, _, _ = _scene(case, seed)
    d = _device()
    x0, v0, e0 = (torch.from_numpy(a[k].astype(np.float64)).to(d) for k in ("pos", "vel", "ev"))
    E = _Exact3D(p, variant, torch.from_numpy(a["level"].astype(np.int64)).to(d))
    rho, press, f, surface = E.forces(x0, e0)
    x, v, ev = E.integrate(x0, v0, e0, rho, f)
    one = {"pos": x, "vel": v, "ev": ev, "acc": f, "dens": rho[:, None], "press": press[:, None],
           "energy": E.energy(x0, x, v)[:, None], "surface": surface[:, None],
           "tension": torch.zeros_like(rho)[:, None], "level": None, "n": None}
    if case["flags"] & MESH:
        one["mesh"] = one["triangles"] = None
    most = _most(variant, a)
    return {k: t if t is None else torch.cat([t, t.new_zeros(most - len(t), t.shape[1])])
            for k, t in one.items()}


def _exact_rollout(case, seed):
    p, a, theta, target = _rollout_inputs(case, seed)
    d = _device()
    x0, v0, e0 = (torch.from_numpy(a[k].astype(np.float64)).to(d).requires_grad_()
                  for k in ("pos", "vel", "ev"))
    E = _Exact3D(p, sa.V3D2, torch.from_numpy(a["level"].astype(np.int64)).to(d))
    nf, ns = case["nodes"], case["samples"]
    th = torch.from_numpy(theta.astype(np.float64)).to(d).requires_grad_()
    field = th.view(nf, nf, nf, 3)  # z, y, x
    x, v, ev = x0, v0, e0
    for _ in range(case["steps"]):
        rho, _, f, _ = E.forces(x, ev)
        g = (x / E.world * (nf - 1)).clamp(0.0, float(nf - 1))
        i0 = g.detach().floor().clamp(max=nf - 2).long()
        t = g - i0
        for k in range(8):
            b = [(k >> c) & 1 for c in range(3)]
            w = 1.0
            for c in range(3):
                w = w * (t[:, c] if b[c] else 1 - t[:, c])
            f = f + w[:, None] * field[i0[:, 2] + b[2], i0[:, 1] + b[1], i0[:, 0] + b[0]]
        x, v, ev = E.integrate(x, v, ev, rho, f)
    q = (torch.arange(ns, dtype=torch.float64, device=d) + 0.5) / ns
    Z, Y, X = torch.meshgrid(q * E.world[2], q * E.world[1], q * E.world[0], indexing="ij")
    pts = torch.stack([X.reshape(-1), Y.reshape(-1), Z.reshape(-1)], 1)
    rad = E.rad[E.L]
    with torch.no_grad():
        # a sample point sums the particles of the 27 cells around its own
        cp, cx = (pts / E.cell).floor(), (x / E.cell).floor()

        def near(i0, i1):
            ok = torch.ones(i1 - i0, len(x), dtype=torch.bool, device=d)
            for c in range(3):
                ok &= (cp[i0:i1, c:c + 1] - cx[None, :, c]).abs() <= 1
            return ok
        i, j = _pairs(pts, x, float(rad.max()) ** 2, near)
    r2 = ((pts[i] - x[j]) ** 2).sum(1)
    inside = r2 < rad[j] ** 2
    w = torch.where(inside, E.m[E.L[j]] * E.p6r[E.L[j]] * (rad[j] ** 2 - r2) ** 3, torch.zeros_like(r2))
    rho_s = torch.zeros(len(pts), dtype=torch.float64, device=d).index_add(0, i, w)
    loss = ((rho_s - torch.from_numpy(target.astype(np.float64)).to(d)) ** 2).sum()
    loss.backward()
    def padded(t):
        return torch.cat([t.detach(), t.new_zeros(t.shape)])
    return {"pos": padded(x), "vel": padded(v), "ev": padded(ev), "n": None, "acc": None, "dens": None,
            "press": None, "energy": None, "surface": None, "tension": None, "level": None,
            "loss": np.float64(loss.item()), "sample": rho_s.detach(), "dtheta": th.grad,
            "dpos": x0.grad, "dvel": v0.grad, "dev": e0.grad}
