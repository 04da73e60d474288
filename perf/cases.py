"""The work this framework is used for, as cases that can be timed and checked.

Kinds of case:
  forward  time stepping of one mesh with n right-hand sides on one GPU, from a
           wavefield that fills the mesh, driven by point forces: the solver's
           main path (element forces, assembly, C-PML, Newmark update, strain
           recording).  What a program reads back is the strain of the
           recording cells at every snapshot, one array per force ("records"),
           or, when x, y and z forces run together, the strain Green's tensors
           of those cells ("tiles", three fields per station).
  batch    independent meshes of uneven size advanced together.
  trace    tile interpolation: every time sample at one place (a synthetic).
  interp   tile interpolation at many places and times.
  query    the learned surrogate in front of a tile: network, tile
           interpolation or zero by region.
  train    training of the surrogate's network on a tile.
  plugin   the element force of the reference's backend interface on host
           arrays (FP64).

Sizes: the halfspace and layered boxes of pygfx.workloads (1 km and 0.6 km
hexes, order 4, C-PML on the sides and the bottom) from 1,000 to 131,072
elements, 1 to 24 fields, and the surrogate's own shapes (64 frequencies,
6 layers of 256, batches of 8,192).  exact() restates each path in FP64 with
plain torch and numpy.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gf-only-sem_amd"))

import pygfx  # noqa: E402
from pygfx import workloads  # noqa: E402


# --------------------------------------------------------------------------- cases

def listed():
    def fwd(name, nx, ny, nz, fields, steps, **kw):
        c = dict(name=name, kind="forward", nx=nx, ny=ny, nz=nz, pml=2, fields=fields, steps=steps, stride=10,
                 layered=True, jitter=0.0, sls=0, complete=False, receivers=96, tiles=False)
        c.update(kw)
        return c

    return [
        # one force on the small homogeneous box: the reference's own CPU-sized run,
        # a few microseconds per kernel, so launches and latency count
        fwd("small_halfspace_1", 20, 20, 10, 1, 40, pml=3, layered=False),
        # one force on a large mesh: the plain single-direction run
        fwd("plain_large_1", 64, 64, 32, 1, 40),
        # x, y and z forces of one station on an odd-sized mesh, straight into a
        # tile of Green's tensors: what a Green's function database is built from
        fwd("station_xyz_3", 45, 39, 21, 3, 20, tiles=True),
        # x, y and z forces at 8 stations: the batched run
        fwd("stations_xyz_24", 36, 36, 18, 24, 20, tiles=True),
        # hexahedra that are not axis-aligned (full 3 x 3 geometry)
        fwd("deformed_hexes_3", 34, 31, 17, 3, 20, jitter=0.15),
        # shear attenuation by three standard linear solids
        fwd("attenuation_3", 28, 26, 15, 3, 20, sls=3),
        # complete C-PML (stretched stresses inside the PML elements)
        fwd("complete_cpml_3", 30, 28, 15, 3, 20, complete=True),
        # many small meshes of uneven size in one batch
        dict(name="batch_small_meshes", kind="batch", meshes=20, lo=500, hi=4000, mesh_seed=6, fields=3, steps=20,
             stride=10, groups=4),
        # one synthetic: all samples of a 30 s tile at one place
        dict(name="trace_600", kind="trace", nx=8, ny=8, nz=3, n_time=600),
        # the surrogate in front of a tile, 150,000 queries (three chunks, the last one ragged)
        dict(name="query_150k", kind="query", nx=20, ny=18, nz=4, n_time=40, n=150001, windows=10, judge=0.2, zero=0.2),
        # training at the network's default shape and batch, late in the cosine schedule
        dict(name="train_8192", kind="train", nx=12, ny=12, nz=4, n_time=40, batch=8192, iters=8, depth=6, width=256),
        # the backend plugin: one call on host arrays
        dict(name="plugin_800", kind="plugin", n_elem=800, ngll=5),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["forward"] * 7 + ["batch", "trace", "interp", "query", "train", "plugin"])
    if kind == "forward":
        fields = rng.choice([1, 1, 2, 3, 3, 6, 12, 24])
        n = _logint(rng, 1000, min(125000, 500000 // fields))
        nx = max(6, int(round((2 * n) ** (1 / 3) * rng.uniform(0.85, 1.15))))
        ny = max(6, int(round((2 * n) ** (1 / 3) * rng.uniform(0.85, 1.15))))
        nz = max(4, min(n // (nx * ny), 32))
        form = rng.choice(["box"] * 4 + ["jitter", "sls", "complete"])
        if form in ("sls", "complete"):  # their memories make a step several times as dear
            while nx * ny * nz * fields > 60000:
                fields = max(1, fields // 2)
                nx, ny = max(6, int(nx * 0.9)), max(6, int(ny * 0.9))
        return dict(kind="forward", nx=nx, ny=ny, nz=nz, pml=rng.choice([1, 2, 3]) if min(nx, ny) >= 9 and nz >= 6 else 1,
                    fields=fields, steps=rng.choice([10, 20]), stride=10, layered=rng.random() < 0.8,
                    jitter=0.15 if form == "jitter" else 0.0, sls=rng.choice([1, 2, 3]) if form == "sls" else 0,
                    complete=form == "complete", receivers=_logint(rng, 8, 150),
                    tiles=fields % 3 == 0 and rng.random() < 0.6)
    if kind == "batch":
        return dict(kind="batch", meshes=rng.randint(4, 20), lo=500, hi=4000, mesh_seed=rng.randint(0, 10 ** 6), fields=3,
                    steps=10, stride=10, groups=rng.choice([0, 2, 4]))
    tile = dict(nx=rng.randint(5, 18), ny=rng.randint(5, 18), nz=rng.randint(2, 4))
    if kind == "trace":
        return dict(kind=kind, **tile, n_time=rng.randint(100, 400))
    if kind == "interp":
        return dict(kind=kind, **tile, n_time=rng.randint(10, 40), n=_logint(rng, 500, 150000))
    if kind == "query":
        return dict(kind=kind, **tile, n_time=rng.randint(10, 40), n=_logint(rng, 500, 140000), windows=rng.choice([1, 5, 10]),
                    judge=rng.choice([0.1, 0.4, 0.8]), zero=rng.choice([0.0, 0.2]))
    if kind == "train":
        return dict(kind=kind, **tile, n_time=rng.randint(10, 40), batch=_logint(rng, 1000, 8192), iters=rng.randint(2, 8),
                    depth=rng.choice([4, 6]), width=rng.choice([128, 256]))
    return dict(kind=kind, n_elem=_logint(rng, 8, 1000), ngll=rng.choice([4, 5, 5, 5, 6]))


# --------------------------------------------------------------------------- inputs

F0 = 1.5      # Hz, the Ricker wavelets and the C-PML
FORCE = 2e10  # N; with the metre-scale wavefields below both parts matter


def _mesh(case, seed):
    h = 600.0 if case["layered"] else 1000.0
    nx, ny, nz, p = case["nx"], case["ny"], case["nz"], case["pml"]
    kw = dict(nx=nx, ny=ny, nz=nz, lx=h * nx, ly=h * ny, lz=h * nz, pml_xmin=p, pml_xmax=p, pml_ymin=p, pml_ymax=p,
              pml_zmax=p, f0_pml=F0, cfl_safety=0.5, output_dt=0.05, duration=5.0, record_depth_max=600.0,
              want_coords=0, want_beta=0, jitter=case["jitter"], jitter_seed=seed + 1)
    if case["layered"]:
        kw.update(layers=workloads.LAYERED, rf_amp=0.05, rf_corr_len=2000.0, rf_modes=64, rf_seed=seed + 2)
    else:
        f = 1.0 + 0.01 * (seed % 7)
        kw.update(layers=[(zb, vp * f, vs * f, rho) for zb, vp, vs, rho in workloads.HALFSPACE])
    if case["sls"]:
        kw.update(n_sls=case["sls"], q_mu=[60.0, 120.0, 250.0], att_fmin=0.05, att_fmax=2.0)
    if case["complete"]:
        kw.update(want_profiles=1, pml_profile=1)
    return pygfx.build_box(pygfx.make_spec(**kw), copy=False)


def _receivers(mesh, n):
    """Recording cells scattered outside the C-PML, next to it included; they belong to the mesh, not to the seed."""
    rng = np.random.default_rng(mesh.n_elem)
    inner = np.flatnonzero(mesh.pml_region == 0)
    return np.sort(rng.choice(inner, min(n, inner.size), replace=False)).astype(np.int32)


def _sources(mesh, fields, rng):
    """Fields 3k, 3k+1, 3k+2: x, y and z forces at one seeded place; one field: a z force."""
    x0, x1, y0, y1, z0, z1 = mesh.bounds
    out = []
    for f in range(fields):
        if f % 3 == 0:
            at = (x0 + (x1 - x0) * rng.uniform(0.35, 0.65), y0 + (y1 - y0) * rng.uniform(0.35, 0.65),
                  z0 + (z1 - z0) * rng.uniform(0.3, 0.5))
            cells, w = mesh.locate_source(*at)
            stf = pygfx.ricker(F0, 0.05, FORCE * rng.uniform(0.5, 2.0), mesh.dt, 4000)
        out.append((2 if fields == 1 else f % 3, cells, w, stf))
    return out


def _waves(mesh, fields, rng):
    """u, v [n_node, 3] of each field: two plane waves through the whole mesh."""
    xyz = mesh.node_xyz.reshape(-1, 3)
    k = rng.normal(size=(2, 3))
    k *= (2 * math.pi / rng.uniform(4000.0, 9000.0, (2, 1))) / np.linalg.norm(k, axis=1, keepdims=True)
    ph = rng.uniform(0, 2 * math.pi, 2)
    a, b = np.sin(xyz @ k[0] + ph[0]), np.cos(xyz @ k[1] + ph[1])
    for _ in range(fields):
        c = rng.normal(size=(4, 3)) * np.array([[1e-2], [1e-2], [5e-2], [5e-2]])
        yield a[:, None] * c[0] + b[:, None] * c[1], a[:, None] * c[2] + b[:, None] * c[3]


def _tile_nodes(mesh, cells):
    ib = mesh.ibool.reshape(-1, 125)[cells]
    nodes, inv = np.unique(ib.ravel(), return_inverse=True)
    return nodes, mesh.node_xyz.reshape(-1, 3)[nodes], inv.reshape(-1, 125).astype(np.int32)


def _solver(case, mesh, rng):
    """A solver with its sources and its wavefield, as gather assembly runs it."""
    rec = _receivers(mesh, case.get("receivers", 24))
    n_snap = case["steps"] // case["stride"]
    s = pygfx.Solver(mesh, n_fields=case["fields"], assembly=pygfx.GFX_ASSEMBLY_GATHER, record_capacity=n_snap,
                     snapshot_stride=case["stride"], rec_cell=rec, cpml_complete=bool(case.get("complete")))
    for f, (d, cells, w, stf) in enumerate(_sources(mesh, case["fields"], rng)):
        s.set_source(f, d, cells, w, stf)
    zero = np.zeros(mesh.n_node * 3)
    for f, (u, v) in enumerate(_waves(mesh, case["fields"], rng)):
        s.set_state(f, u.ravel(), v.ravel(), zero)
    return s, rec


def _box(nx, ny, nz, pml, h, layers, duration=5.0):
    return pygfx.make_spec(nx=nx, ny=ny, nz=nz, lx=h * nx, ly=h * ny, lz=h * nz, layers=layers, pml_xmin=pml,
                           pml_xmax=pml, pml_ymin=pml, pml_ymax=pml, pml_zmax=pml, f0_pml=F0, cfl_safety=0.5,
                           output_dt=0.05, duration=duration, record_depth_max=600.0, want_coords=0, want_beta=0)


def _batch_sizes(case):
    """(nx, ny, nz, pml) of each mesh: sizes belong to the case, what is in them to the seed."""
    rng = np.random.default_rng(case["mesh_seed"])
    out = []
    for _ in range(case["meshes"]):
        n = math.exp(rng.uniform(math.log(case["lo"]), math.log(case["hi"])))
        nx = max(6, int(round((2 * n) ** (1 / 3))))
        out.append((nx, nx, max(4, int(round(nx / 2))), int(rng.integers(1, 3))))
    return out


def _batch_meshes(case, rng):
    for nx, ny, nz, pml in _batch_sizes(case):
        vs = np.sort(rng.uniform(1500.0, 4500.0, 3))
        layers = [(600.0 * nz * f, 1.73 * v, v, rng.uniform(2300.0, 3300.0)) for f, v in zip((0.3, 0.6, 0.0), vs)]
        yield pygfx.build_box(_box(nx, ny, nz, pml, 600.0, layers), copy=False)


def _tile_inputs(case, seed):
    """A tile over the cells of a box near the surface, and its values [n_node, 18] per time sample."""
    rng = np.random.default_rng(seed)
    mesh = pygfx.build_box(_box(case["nx"], case["ny"], case["nz"], 1, 600.0, workloads.HALFSPACE), copy=False)
    nodes, xyz, cidx = _tile_nodes(mesh, np.arange(mesh.n_elem))
    r = np.linalg.norm(xyz - xyz.mean(axis=0), axis=1)[:, None]
    amp, decay = rng.normal(size=(2, 18)) * 1e-9, 1500.0 / (r + 1500.0)
    ph = r / rng.uniform(1500.0, 2500.0) + rng.uniform(0, 6.28, 18)
    a = (decay * amp[0] * np.sin(ph)).astype(np.float32)
    b = (decay * amp[1] * np.cos(ph * 1.3)).astype(np.float32)
    w = float(rng.uniform(0.2, 0.5))

    def values(t):
        return a * np.float32(math.cos(w * t)) + b * np.float32(math.sin(1.7 * w * t))

    return rng, xyz, cidx, values


def _tile(case, seed):
    rng, xyz, cidx, values = _tile_inputs(case, seed)
    tile = pygfx.GreenTile(case["n_time"], xyz, cidx)
    for t in range(case["n_time"]):
        tile.set_values(t, values(t))
    return rng, tile


def _places(xyz, n, rng):
    lo, hi = xyz.min(axis=0), xyz.max(axis=0)
    return lo + (0.002 + 0.996 * rng.random((n, 3))) * (hi - lo)


DT_SNAP = 0.05


def _net(case, rng, xyz, **cfg):
    """The surrogate's network with its input box, output scales, moveout and radial envelope."""
    lo, hi = xyz.min(axis=0), xyz.max(axis=0)
    c = 0.5 * (lo + hi)
    slow = 1.0 / 3000.0
    r_max = float(np.hypot(xyz[:, 0] - c[0], xyz[:, 1] - c[1]).max())
    t_hi = case["n_time"] * DT_SNAP
    half = np.r_[hi - lo, t_hi + slow * r_max] * 0.5 + 1.0
    mid = np.r_[c, 0.5 * (t_hi - slow * r_max)]
    scale = rng.uniform(0.5e-9, 2e-9, 18)
    net = pygfx.MLP(mid - half, mid + half, scale, sigma=1.0, seed=int(rng.integers(1, 1 << 30)), **cfg)
    env = (1.0 / (1.0 + 4.0 * (np.arange(32) + 0.5) / 32)).astype(np.float32)
    net.set_envelope(c[0], c[1], r_max, env, slowness=slow)
    return net, dict(lo=mid - half, hi=mid + half, scale=scale, c=c, slow=slow, r_max=r_max, env=env)


def _query_inputs(case, rng, xyz, n_cell):
    pts = _places(xyz, case["n"], rng)
    tix = rng.integers(0, case["n_time"], case["n"]).astype(np.int32)
    u = rng.random((n_cell, case["windows"]))
    policy = np.where(u < case["judge"], 1, np.where(u < case["judge"] + case["zero"], 2, 0)).astype(np.uint8)
    return pts, tix, policy


def _gll(n):
    """Gauss-Lobatto-Legendre points, weights and derivative matrix D[i][j] = l_j'(x_i)."""
    p = np.polynomial.legendre.Legendre.basis(n - 1)
    x = np.r_[-1.0, np.sort(p.deriv().roots().real), 1.0]
    w = 2.0 / (n * (n - 1) * p(x) ** 2)
    D = np.array([[p(x[i]) / (p(x[j]) * (x[i] - x[j])) if i != j else 0.0 for j in range(n)] for i in range(n)])
    D[0, 0], D[-1, -1] = -n * (n - 1) / 4.0, n * (n - 1) / 4.0
    return x, w, D


def _plugin_inputs(case, seed):
    rng = np.random.default_rng(seed)
    n, q = case["n_elem"], case["ngll"]
    _, w, D = _gll(q)
    P = n * q ** 3
    dxi = np.eye(3)[None] / 300.0 + rng.normal(size=(P, 3, 3)) * 2e-4
    jac = 1.0 / np.linalg.det(dxi)
    mu = rng.uniform(2e10, 4e10, P)
    return dict(dxi=dxi.reshape(-1), jac=jac, lam=rng.uniform(2e10, 5e10, P), mu=mu, D=np.ascontiguousarray(D), w=w,
                ngll=q, u=rng.normal(size=P * 3) * 1e-3, r=rng.normal(size=P * 3) * 1e9)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "forward":
        rng = np.random.default_rng(seed)
        mesh = _mesh(case, seed)
        s, rec = _solver(case, mesh, rng)
        st = dict(kind=kind, case=case, solver=s, tiles=[], mesh=mesh)
        if case["tiles"]:  # one tile per station (three fields)
            nodes, xyz, cidx = _tile_nodes(mesh, rec)
            cmap = pygfx.green_capture_map(mesh, rec, nodes)
            for _ in range(case["fields"] // 3):
                t = pygfx.GreenTile(case["steps"] // case["stride"], xyz, cidx)
                t.set_capture_map(*cmap)
                st["tiles"].append(t)
        return st
    if kind == "batch":
        rng = np.random.default_rng(seed)
        meshes = list(_batch_meshes(case, rng))
        solvers = [_solver(case, m, rng)[0] for m in meshes]
        return dict(kind=kind, case=case, solvers=solvers, batch=pygfx.Batch(solvers, groups=case["groups"]))
    if kind in ("trace", "interp"):
        rng, tile = _tile(case, seed)
        if kind == "trace":
            pts = np.repeat(_places(tile.xyz, 1, rng), case["n_time"], axis=0)
            tix = np.arange(case["n_time"], dtype=np.int32)
        else:
            pts = _places(tile.xyz, case["n"], rng)
            tix = rng.integers(0, case["n_time"], case["n"]).astype(np.int32)
        return dict(kind=kind, tile=tile, pts=pts, tix=tix)
    if kind == "query":
        rng, tile = _tile(case, seed)
        net, _ = _net(case, rng, tile.xyz)
        pts, tix, policy = _query_inputs(case, rng, tile.xyz, tile.n_cell)
        return dict(kind=kind, tile=tile, net=net, pts=pts, tix=tix, policy=policy)
    if kind == "train":
        rng, tile = _tile(case, seed)
        net, _ = _net(case, rng, tile.xyz, lr=1e-4, lr_final=5e-5, batch=case["batch"], depth=case["depth"],
                      width=case["width"])
        return dict(kind=kind, tile=tile, net=net, iters=case["iters"], seed=seed % 1000003)
    return dict(kind=kind, **_plugin_inputs(case, seed))


def _records(s, fields, n_snap):
    """Strain of the last n_snap snapshots [n_snap][fields][n_rec*125*6], in the single precision record files hold."""
    done = s.n_snapshots
    return np.stack([np.stack([s.get_record(f, k).astype(np.float32) for f in range(fields)])
                     for k in range(done - n_snap, done)])


def run(st):
    kind = st["kind"]
    if kind == "forward":
        c, s = st["case"], st["solver"]
        n_snap = c["steps"] // c["stride"]
        s.run(c["steps"])
        if not st["tiles"]:
            return _records(s, c["fields"], n_snap)
        done = s.n_snapshots
        for k in range(n_snap):
            for i, t in enumerate(st["tiles"]):
                t.capture(s, done - n_snap + k, [3 * i, 3 * i + 1, 3 * i + 2], k)
        return np.stack([np.stack([t.get_values(k) for k in range(n_snap)]) for t in st["tiles"]])
    if kind == "batch":
        c = st["case"]
        st["batch"].run(c["steps"])
        return [_records(s, c["fields"], c["steps"] // c["stride"]) for s in st["solvers"]]
    if kind in ("trace", "interp"):
        out, cell = st["tile"].interpolate(st["pts"], st["tix"])
        return {"greens": out, "cell": cell}
    if kind == "query":
        out, n_judge = st["net"].query(st["tile"], st["policy"], 0.0, DT_SNAP, st["pts"], st["tix"])
        return {"greens": out, "n_judge": n_judge}
    if kind == "train":
        loss = st["net"].train(st["tile"], 0.0, DT_SNAP, st["iters"], seed=st["seed"])
        return {"loss": loss, "params": st["net"].params()[0]}
    r = st["r"].copy()
    pygfx.element_residual(st["dxi"], st["jac"], st["lam"], st["mu"], st["D"], st["w"], st["ngll"], st["u"], r)
    return r


# --------------------------------------------------------------------------- what a pass cannot do without

def _step_work(nx, ny, nz, pml, fields, general=False, sls=0, complete=False):
    """Bytes and flops of one step: geometry, moduli and node ids once, displacement and velocity of every field
    read and written once, the C-PML's and the solids' memories read and written once."""
    E = nx * ny * nz
    P, G = E * 125, (4 * nx + 1) * (4 * ny + 1) * (4 * nz + 1)
    b = P * ((36 if general else 12) + 8 + 4) + G * (4 + 48 * fields)
    # PML elements by the number of damped axes (x and y on both sides, z at the bottom)
    axes = [[(n - k * pml) if d == 0 else k * pml for d in (0, 1)] for n, k in ((nx, 2), (ny, 2), (nz, 1))]
    for m in range(1, 8):
        cnt = 1
        for q in range(3):
            cnt *= max(0, axes[q][m >> q & 1])
        on = bin(m).count("1")
        if complete:
            b += cnt * 125 * (28 * 4 + 8 * fields * (12, 27, 45)[on - 1])
        else:
            b += cnt * 64 * (56 + 8 * fields * (3 + 3 * on + 3))
    if sls:
        b += P * (12 * sls + 8 * fields * (5 * sls + 5))
    return b, P * fields * (180 + (60 if not general else 96))


def work(case):
    kind = case["kind"]
    if kind == "forward":
        b, f = _step_work(case["nx"], case["ny"], case["nz"], case["pml"], case["fields"], case["jitter"] > 0, case["sls"],
                          case["complete"])
        return {"bytes": b * case["steps"], "flops": f * case["steps"]}
    if kind == "batch":
        w = [_step_work(*size, case["fields"]) for size in _batch_sizes(case)]
        return {"bytes": case["steps"] * sum(x[0] for x in w), "flops": case["steps"] * sum(x[1] for x in w)}
    if kind in ("trace", "interp"):
        n = case["n_time"] if kind == "trace" else case["n"]
        return {"bytes": n * (28 + 76 + 125 * 72), "flops": n * 125 * 18 * 2}
    shape = [128] + [case.get("width", 256)] * case.get("depth", 6) + [18]
    macs = sum(a * b for a, b in zip(shape, shape[1:]))
    if kind == "query":
        return {"bytes": case["n"] * (28 + 72 + case["judge"] * 125 * 72) + 2 * macs, "flops": case["n"] * 2 * macs}
    if kind == "train":
        return {"bytes": case["iters"] * (case["batch"] * 72 + 28 * macs), "flops": case["iters"] * case["batch"] * 6 * macs}
    n, q = case["n_elem"], case["ngll"]
    return {"bytes": n * q ** 3 * 8 * (12 + 9), "flops": n * q ** 3 * (36 * q + 120)}


# --------------------------------------------------------------------------- the same in 64 bits

def _t(a, *shape):
    t = torch.from_numpy(np.ascontiguousarray(a)).to("cuda")
    return t.reshape(*shape) if shape else t


class _Ref:
    """The time step in FP64: displacement form of the solver's scheme (beta = 0, gamma = 1/2)."""

    def __init__(self, mesh, sls=0, complete=False):
        E, G = mesh.n_elem, mesh.n_node
        self.E, self.G, self.dt = E, G, mesh.dt
        _, w, D = _gll(5)
        self.D = _t(D)
        w3 = np.einsum("i,j,k->ijk", w, w, w).ravel()
        self.ib = _t(mesh.ibool).long()
        self.g = _t(mesh.dxi_dx, E, 125, 3, 3)  # [m][a] = d xi_a / d x_m
        self.jw = _t(mesh.jacobian, E, 125) * _t(w3)
        self.lam, self.mu = _t(mesh.lambda_, E, 125).clone(), _t(mesh.mu_, E, 125).clone()
        mass = _t(mesh.mass, E, 125).clone()
        pml = mesh.pml_region != 0
        self.sls, self.complete = sls, complete
        if complete:
            self.pe = _t(np.flatnonzero(pml))
            K, d, al = (_t(a, E, 125, 3)[self.pe].clone() for a in (mesh.pml_K, mesh.pml_d, mesh.pml_alpha))
            self.K, self.d, self.al = K, d, al
            self.rjw = mass[self.pe].clone()
            cv = K[..., 2] * (K[..., 1] * d[..., 0] + K[..., 0] * d[..., 1]) + K[..., 0] * K[..., 1] * d[..., 2]
            mass[self.pe] *= K.prod(-1) + 0.5 * self.dt * cv
            self.abc_a = self._recursion(al, d)
            self.abc_b = self._recursion(al + d / K, d)
        self.m = torch.zeros(G, dtype=torch.float64, device="cuda").index_add_(0, self.ib, mass.reshape(-1))
        if complete:  # the outer faces of the C-PML are held rigid
            x = _t(mesh.node_xyz, G, 3)
            lo, hi = x.amin(0), x.amax(0)
            t = 1e-6 * (hi - lo)
            out = (x < lo + t) | (x > hi - t)
            rigid = out[:, 0] | out[:, 1] | (x[:, 2] > hi[2] - t[2])
            self.m[rigid] = 0.0
        self.minv = torch.where(self.m > 0, 1.0 / self.m.clamp(min=1e-300), torch.zeros_like(self.m))
        if not complete:
            pe = np.flatnonzero(pml)
            self.pe = _t(pe)
            self.pnode = self.ib.reshape(E, 125)[self.pe].reshape(-1)
            rho = _t(mesh.density, E, 125)[self.pe]
            self.S = (self.jw[self.pe] / rho).reshape(-1, 1) * _t(mesh.coef_abar, E, 125, 5)[self.pe].reshape(-1, 5)
            self.pal = _t(mesh.coef_alpha, E, 125, 9)[self.pe].reshape(-1, 3, 3)
        if sls:
            ts, te = _t(mesh.tau_sigma, E, 125, sls), _t(mesh.tau_epsilon, E, 125, sls)
            a = torch.exp(-self.dt / ts)
            q = ts * (1 - a) / self.dt
            Y = 2 * self.mu[..., None] * (te / ts - 1)
            self.za, self.zb, self.zc = a, Y * (q - a), Y * (1 - q)
            mu_u = self.mu * (1 + (te / ts - 1).sum(-1))
            self.lam = self.lam + 2 * (self.mu - mu_u) / 3
            self.mu = mu_u

    def _recursion(self, p, d):
        """(a, b, c) of one exact step of a first-order filter; zero on axes that are not damped."""
        x = p * self.dt
        small = x.abs() < 1e-4
        xs = torch.where(small, torch.ones_like(x), x)
        em = torch.expm1(-xs)
        i0 = torch.where(small, 1 - x / 2 + x * x / 6 - x ** 3 / 24, -em / xs)
        c = torch.where(small, 0.5 - x / 6 + x * x / 24 - x ** 3 / 120, (xs + em) / (xs * xs))
        on = (d != 0).double()
        return torch.exp(-x) * on, self.dt * (i0 - c) * on, self.dt * c * on

    def _along(self, u, a, M):
        """sum_s M[i][s] u(.., s, ..) along reference axis a of u [E, 125, c]."""
        v = u.reshape(-1, 5, 5, 5, u.shape[-1]).movedim(1 + a, -1)
        return (v @ M.T).movedim(-1, 1 + a).reshape(u.shape)

    def gradient(self, u, g):
        du = torch.stack([self._along(u, a, self.D) for a in range(3)], -1)  # [E, p, c, a]
        return du @ g.transpose(-1, -2)                                     # [E, p, c, m]

    def start(self, u, v):
        z = lambda *s: torch.zeros(*s, dtype=torch.float64, device="cuda")  # noqa: E731
        f = dict(u=u, v=v, a=torch.zeros_like(u))
        n = self.pe.numel()
        if self.complete:
            f["q"] = [[[z(n, 125) for _ in range(4)] for _ in range(9)], [[z(n, 125) for _ in range(3)] for _ in range(3)]]
        else:
            f["pm"], f["pn"] = z(n * 125, 3, 3), z(n * 125, 3)  # [component][direction]
        if self.sls:
            f["zeta"], f["dev"] = z(self.E, 125, self.sls, 5), z(self.E, 125, 5)
        return f

    def _conv(self, abc, store, k, g):
        m = store[k] + abc[2] * g
        store[k] = abc[0] * m + abc[1] * g
        return m

    def _complete_terms(self, f, gr, U, w):
        """Stretched stresses S[a][b] and the inertia term of the PML elements."""
        ax = lambda t, q: t[..., q]  # noqa: E731
        A = [[t[..., q] for t in self.abc_a] for q in range(3)]
        B = [[t[..., q] for t in self.abc_b] for q in range(3)]
        G = [[None] * 9 for _ in range(3)]
        for k in range(3):
            for l in range(3):
                m, n = (1 if l == 0 else 0), (1 if l == 2 else 2)
                Q = f["q"][0][k * 3 + l]
                gv = gr[..., k, l]
                Km, Kn, dm, dn = ax(self.K, m), ax(self.K, n), ax(self.d, m), ax(self.d, n)
                Mm, Mn = self._conv(A[m], Q, 0, gv), self._conv(A[n], Q, 1, gv)
                Mmn = self._conv(A[n], Q, 2, Mm)
                y2 = Km * Kn * gv + Kn * dm * Mm + dn * (Km * Mn + dm * Mmn)
                Mb = self._conv(B[l], Q, 3, y2)
                G[l][k * 3 + l] = (y2 - ax(self.d, l) / ax(self.K, l) * Mb) / ax(self.K, l)
                G[n][k * 3 + l] = Km * gv + dm * Mm
                G[m][k * 3 + l] = Kn * gv + dn * Mn
        lam, mu = self.lam[self.pe], self.mu[self.pe]
        S = torch.empty_like(gr)
        for a in range(3):
            for b in range(3):
                S[..., a, b] = mu * (G[b][a * 3 + b] + G[b][b * 3 + a])
                if a == b:
                    S[..., a, b] += lam * (G[b][0] + G[b][4] + G[b][8])
        K, d, al = self.K, self.d, self.al
        L = torch.empty_like(U)
        for c in range(3):
            Q, u, v = f["q"][1][c], U[..., c], w[..., c]
            C1 = self._conv(A[0], Q, 0, u)
            z1 = K[..., 0] * u + d[..., 0] * C1
            C2 = self._conv(A[1], Q, 1, z1)
            z2 = K[..., 1] * z1 + d[..., 1] * C2
            C3 = self._conv(A[2], Q, 2, z2)
            L1 = d[..., 0] * (v - al[..., 0] * u + al[..., 0] ** 2 * C1)
            D1 = K[..., 0] * v + d[..., 0] * (u - al[..., 0] * C1)
            L2 = K[..., 1] * L1 + d[..., 1] * (D1 - al[..., 1] * z1 + al[..., 1] ** 2 * C2)
            D2 = K[..., 1] * D1 + d[..., 1] * (z1 - al[..., 1] * C2)
            L[..., c] = K[..., 2] * L2 + d[..., 2] * (D2 - al[..., 2] * z2 + al[..., 2] ** 2 * C3)
        return S, L * self.rjw[..., None]

    def step(self, f, src, n):
        dt = self.dt
        u, v, a = f["u"], f["v"], f["a"]
        U = u + dt * v + 0.5 * dt * dt * a
        Ue = U[self.ib].reshape(self.E, 125, 3)
        gr = self.gradient(Ue, self.g)
        tr = gr.diagonal(dim1=-2, dim2=-1).sum(-1)
        sig = self.mu[..., None, None] * (gr + gr.transpose(-1, -2))
        if self.sls:
            i, j = [0, 1, 0, 0, 1], [0, 1, 1, 2, 2]
            dev = 0.5 * (gr + gr.transpose(-1, -2))[..., i, j]
            dev[..., :2] -= tr[..., None] / 3
            f["zeta"] = self.za[..., None] * f["zeta"] + self.zb[..., None] * f["dev"][..., None, :] + \
                self.zc[..., None] * dev[..., None, :]
            f["dev"] = dev
            z = f["zeta"].sum(-2)
            for q, (x, y) in enumerate(zip(i, j)):
                sig[..., x, y] -= z[..., q]
                if x != y:
                    sig[..., y, x] -= z[..., q]
            sig[..., 2, 2] += z[..., 0] + z[..., 1]
        for q in range(3):
            sig[..., q, q] += self.lam * tr
        extra = None
        if self.complete:
            w = (v + 0.5 * dt * a)[self.ib].reshape(self.E, 125, 3)[self.pe]
            sig[self.pe], extra = self._complete_terms(f, gr[self.pe], Ue[self.pe], w)
        del gr
        F = (sig @ self.g) * self.jw[..., None, None]  # [E, p, c, a]
        re = -sum(self._along(F[..., q], q, self.D.T) for q in range(3))
        if extra is not None:
            re[self.pe] -= extra
        direction, cells, w, stf = src
        if n < stf.size:
            for k, e in enumerate(cells):
                re[int(e), :, direction] += float(stf[n]) * _t(w.reshape(-1, 125)[k])
        r = torch.zeros_like(u).index_add_(0, self.ib, re.reshape(-1, 3))
        if not self.complete and self.pe.numel():
            th = 1.0 / 8.0
            c1, c2 = (1 - 2 * th) * 0.5 * dt, (1 - th) * 0.5 * dt * dt
            pn = self.pnode
            old, new = f["pn"] + c2 * a[pn], u[pn] + c1 * v[pn]
            S, m = self.S, f["pm"]
            r.index_add_(0, pn, S[:, 0:1] * v[pn] + S[:, 1:2] * u[pn] + (m * S[:, None, 2:5]).sum(-1))
            al = self.pal
            f["pm"] = al[:, None, :, 0] * m + al[:, None, :, 1] * new[..., None] + al[:, None, :, 2] * old[..., None]
            f["pn"] = new
        a1 = r * self.minv[:, None]
        f["u"] = torch.where((self.m > 0)[:, None], U, u)
        f["v"] = v + 0.5 * dt * (a + a1)
        f["a"] = a1

    def strain(self, f, rec):
        ib = self.ib.reshape(self.E, 125)[rec]
        gr = self.gradient(f["u"][ib], self.g[rec])
        e = 0.5 * (gr + gr.transpose(-1, -2))
        return torch.stack([e[..., 0, 0], e[..., 1, 1], e[..., 2, 2], e[..., 0, 1], e[..., 0, 2], e[..., 1, 2]], -1)


def _march(case, mesh, rng):
    """Strain [n_snap][field][n_rec][125][6] of one pass, and the recording cells."""
    rec = _receivers(mesh, case.get("receivers", 24))
    src = _sources(mesh, case["fields"], rng)
    ref = _Ref(mesh, case.get("sls", 0), bool(case.get("complete")))
    rc = _t(rec).long()
    out = []
    for f, (u, v) in enumerate(_waves(mesh, case["fields"], rng)):
        s = ref.start(_t(u), _t(v))
        got = []
        for n in range(case["steps"]):
            ref.step(s, src[f], n)
            if n % case["stride"] == 0:
                got.append(ref.strain(s, rc))
        out.append(torch.stack(got))
    return torch.stack(out, 1), rec


def _exact_tiles(strain, mesh, rec):
    nodes, _, cidx = _tile_nodes(mesh, rec)
    ix = _t(cidx.reshape(-1)).long()
    w = _t(mesh.mass.reshape(-1, 125)[rec].reshape(-1))
    sw = torch.zeros(len(nodes), dtype=torch.float64, device="cuda").index_add_(0, ix, w)
    S, F = strain.shape[:2]
    tiles = []
    for k in range(F // 3):
        x = strain[:, 3 * k:3 * k + 3].reshape(S, 3, -1, 6).permute(2, 0, 3, 1).contiguous()  # [point][snap][comp][dir]
        m = torch.zeros(len(nodes), S, 6, 3, dtype=torch.float64, device="cuda").index_add_(0, ix, x * w[:, None, None, None])
        tiles.append((m / sw[:, None, None, None]).permute(1, 0, 2, 3).reshape(S, len(nodes), 18))
    return torch.stack(tiles).cpu().numpy()


def _exact_interp(case, xyz, cidx, values, pts, tix):
    """Tensor-product Lagrange interpolation in the box cell that holds each place."""
    box = xyz[cidx]
    lo, hi = box.min(axis=1), box.max(axis=1)
    x0, h = lo.min(axis=0), (hi - lo).mean(axis=0)
    ncell = np.round((hi.max(axis=0) - x0) / h).astype(int)
    key = lambda q: (q[:, 0] * ncell[1] + q[:, 1]) * ncell[2] + q[:, 2]  # noqa: E731
    where = np.empty(len(cidx), int)
    where[key(np.round((lo - x0) / h).astype(int))] = np.arange(len(cidx))
    cell = where[key(np.floor((pts - x0) / h).astype(int))]
    xi = 2 * (pts - lo[cell]) / (hi[cell] - lo[cell]) - 1
    g, _, _ = _gll(5)
    L = np.ones((3, len(pts), 5))
    for i in range(5):
        for j in range(5):
            if i != j:
                L[:, :, i] *= ((xi - g[j]) / (g[i] - g[j])).T
    w = np.einsum("na,nb,nc->nabc", *L).reshape(-1, 125)
    w /= w.sum(axis=1, keepdims=True)
    out = np.zeros((len(pts), 18))
    W, ci = _t(w), _t(cidx[cell]).long()
    for t in range(case["n_time"]):
        sel = np.flatnonzero(tix == t)
        if sel.size:
            v = _t(values(t)).double()
            k = _t(sel)
            out[sel] = (W[k, :, None] * v[ci[k]]).sum(1).cpu().numpy()
    return out, cell.astype(np.int32)


def _exact_net(case, net, info, x, params, fourier):
    """Scaled network outputs for raw (x, y, z, t) rows, in the given FP64 parameters."""
    r = torch.hypot(x[:, 0] - info["c"][0], x[:, 1] - info["c"][1])
    xt = torch.cat([x[:, :3], (x[:, 3] - info["slow"] * r)[:, None]], 1)
    lo, hi = _t(info["lo"]), _t(info["hi"])
    ph = (2 * (xt - lo) / (hi - lo) - 1) @ fourier.T * (2 * math.pi)
    h = torch.cat([torch.sin(ph), torch.cos(ph)], 1)
    depth, width, at = int(net.cfg.depth), int(net.cfg.width), 0
    for l in range(depth + 1):
        i, o = h.shape[1], 18 if l == depth else width
        W, b = params[at:at + i * o].reshape(i, o), params[at + i * o:at + i * o + o]
        at += i * o + o
        h = h @ W + b
        if l < depth:
            h = torch.nn.functional.gelu(h)
    return h, _envelope(info, r)


def _envelope(info, r):
    n = len(info["env"])
    return _t(np.interp((r * n / info["r_max"] - 0.5).cpu().numpy(), np.arange(n), info["env"].astype(np.float64)))


def _exact_query(case, seed):
    rng, xyz, cidx, values = _tile_inputs(case, seed)
    net, info = _net(case, rng, xyz)
    pts, tix, policy = _query_inputs(case, rng, xyz, len(cidx))
    out, cell = _exact_interp(case, xyz, cidx, values, pts, tix)
    how = policy[cell, tix.astype(np.int64) * case["windows"] // case["n_time"]]
    w, b = net.params()
    sel = np.flatnonzero(how == 0)
    x = _t(np.c_[pts, tix * DT_SNAP][sel])
    y, e = _exact_net(case, net, info, x, _t(w).double(), _t(b).double())
    out[sel] = (y * _t(info["scale"]) * e[:, None]).cpu().numpy()
    out[how == 2] = 0.0
    return {"greens": out, "n_judge": None}


def _mix64(z):
    with np.errstate(over="ignore"):
        z = z + np.uint64(0x9E3779B97F4A7C15)
        z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
        z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
        return z ^ (z >> np.uint64(31))


def _exact_train(case, seed):
    rng, xyz, cidx, values = _tile_inputs(case, seed)
    net, info = _net(case, rng, xyz, lr=1e-4, lr_final=5e-5, batch=case["batch"], depth=case["depth"], width=case["width"])
    w, b = net.params()
    w, b = _t(w).double().requires_grad_(True), _t(b).double()
    vals = np.stack([values(t) for t in range(case["n_time"])])
    m, v = torch.zeros_like(w), torch.zeros_like(w)
    rows, iters, losses = np.arange(case["batch"], dtype=np.uint64), case["iters"], []
    b1, b2 = float(np.float32(0.9)), float(np.float32(0.999))
    lr0, lr1 = float(np.float32(1e-4)), float(np.float32(5e-5))
    for it in range(iters):
        with np.errstate(over="ignore"):
            sd = np.uint64(seed % 1000003) * np.uint64(0x9E3779B97F4A7C15) + np.uint64(it)
            h = _mix64(sd ^ (rows * np.uint64(0xD1B54A32D192ED03)))
        node = (h % np.uint64(len(xyz))).astype(np.int64)
        t = ((h >> np.uint64(32)) % np.uint64(case["n_time"])).astype(np.int64)
        y, e = _exact_net(case, net, info, _t(np.c_[xyz[node], t * DT_SNAP]), w, b)
        target = _t(vals[t, node].astype(np.float64)) / _t(info["scale"]) / e[:, None]
        loss = ((y - target) ** 2).mean()
        (g,) = torch.autograd.grad(loss, w)
        m, v = b1 * m + (1 - b1) * g, b2 * v + (1 - b2) * g * g
        ph = it / (iters - 1) if iters > 1 else 1.0
        lr = lr1 + 0.5 * (lr0 - lr1) * (1 + math.cos(math.pi * ph))
        with torch.no_grad():
            w -= lr * (m / (1 - b1 ** (it + 1))) / (torch.sqrt(v / (1 - b2 ** (it + 1))) + 1e-8)
        losses.append(float(loss))
    return {"loss": float(np.mean(losses[-max(1, iters // 10):])), "params": w.detach().cpu().numpy()}


def _exact_plugin(case, seed):
    x = _plugin_inputs(case, seed)
    n, q = case["n_elem"], case["ngll"]
    D = x["D"]
    u = x["u"].reshape(n, q, q, q, 3)
    g = x["dxi"].reshape(n, q, q, q, 3, 3)
    du = np.stack([np.einsum("is,nsjkc->nijkc", D, u), np.einsum("js,niskc->nijkc", D, u),
                   np.einsum("ks,nijsc->nijkc", D, u)], -1)
    gr = np.einsum("nijkca,nijkma->nijkcm", du, g)
    mu, lam = x["mu"].reshape(n, q, q, q, 1, 1), x["lam"].reshape(n, q, q, q, 1, 1)
    sig = mu * (gr + np.swapaxes(gr, -1, -2)) + lam * np.trace(gr, axis1=-2, axis2=-1)[..., None, None] * np.eye(3)
    w = x["w"]
    f = x["jac"].reshape(n, q, q, q) * np.einsum("i,j,k->ijk", w, w, w)
    F = np.einsum("nijkcm,nijkma->nijkca", sig, g) * f[..., None, None]
    r = np.einsum("si,nsjkc->nijkc", D, F[..., 0]) + np.einsum("sj,niskc->nijkc", D, F[..., 1]) + \
        np.einsum("sk,nijsc->nijkc", D, F[..., 2])
    return x["r"] - r.reshape(-1)


def exact(case, seed):
    kind = case["kind"]
    if kind == "forward":
        rng = np.random.default_rng(seed)
        mesh = _mesh(case, seed)
        strain, rec = _march(case, mesh, rng)
        if case["tiles"]:
            return _exact_tiles(strain, mesh, rec)
        return strain.reshape(strain.shape[0], strain.shape[1], -1).cpu().numpy()
    if kind == "batch":
        rng = np.random.default_rng(seed)
        out = []
        for mesh in list(_batch_meshes(case, rng)):
            s, _ = _march(case, mesh, rng)
            out.append(s.reshape(s.shape[0], s.shape[1], -1).cpu().numpy())
        return out
    if kind in ("trace", "interp"):
        rng, xyz, cidx, values = _tile_inputs(case, seed)
        n = 1 if kind == "trace" else case["n"]
        pts = _places(xyz, n, rng)
        if kind == "trace":
            pts, tix = np.repeat(pts, case["n_time"], axis=0), np.arange(case["n_time"])
        else:
            tix = rng.integers(0, case["n_time"], n)
        return {"greens": _exact_interp(case, xyz, cidx, values, pts, tix)[0], "cell": None}
    if kind == "query":
        return _exact_query(case, seed)
    if kind == "train":
        return _exact_train(case, seed)
    return _exact_plugin(case, seed)
