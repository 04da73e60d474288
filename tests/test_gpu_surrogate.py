"""Surrogate on the GPU: the device GLL judge against the FP64 host judge,
the MFMA forward / backward of the MLP against the CPU model (oracle/mlp.py,
BF16 operands emulated), Adam training on a tile, Green's tensor capture from
solver records against the mass-weighted merge computed from the records on
the host, and the fallback rule of the surrogate query."""
import os
import sys

import numpy as np
import pytest

import meshcases as mc
import pygfx

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "oracle"))
import mlp as mlp_oracle  # noqa: E402
from test_surrogate import tile_from_mesh  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if pygfx.device_count() < 1:
        pytest.fail("no HIP device visible; GPU tests must run on an MI355X box")


@pytest.fixture(scope="module")
def box():
    m = pygfx.build_box(nx=6, ny=5, nz=3, lx=3600.0, ly=3000.0, lz=1800.0, pml_xmin=0, pml_xmax=0, pml_ymin=0,
                        pml_ymax=0, pml_zmax=0, output_dt=0.05, duration=0.2, record_depth_max=0.0)
    nodes, xyz, cidx = tile_from_mesh(m, np.arange(m.n_elem))
    return m, xyz, cidx


def smooth_field(xyz, t):
    x, y, z = xyz[:, 0] / 3600.0, xyz[:, 1] / 3000.0, xyz[:, 2] / 1800.0
    base = np.stack([np.sin(2.1 * x + 0.7 * k) * np.cos(1.3 * y - 0.2 * k) * (1 + 0.5 * z) * np.cos(0.8 * t + 0.1 * k)
                     for k in range(18)], axis=1)
    return base.astype(np.float32)


def test_device_judge_matches_host_judge(box):
    m, xyz, cidx = box
    g = pygfx.GreenTile(3, xyz, cidx)
    for t in range(3):
        g.set_values(t, smooth_field(xyz, t) + 0.01 * t)
    rng = np.random.default_rng(11)
    lo, hi = xyz.min(axis=0), xyz.max(axis=0)
    pts = lo + rng.random((300, 3)) * (hi - lo)
    pts[:20] = xyz[rng.integers(0, len(xyz), 20)]  # exact nodes
    tix = rng.integers(0, 3, 300).astype(np.int32)
    out, cell = g.interpolate(pts, tix)
    assert (cell >= 0).all()
    for i in range(300):
        ref = pygfx.gll_interpolate_host(xyz, cidx, g.get_values(tix[i]).astype(np.float64), pts[i])
        assert np.allclose(out[i], ref, rtol=1e-5, atol=1e-6 * np.abs(ref).max())
    out2, cell2 = g.interpolate(hi + np.array([[10.0, 0, 0]]), np.array([0], np.int32))
    assert cell2[0] == -1 and np.isnan(out2).all()


def _model_pair(width=64, depth=3, n_freq=16, seed=3):
    lo, hi = np.array([0.0, 0.0, 0.0, 0.0]), np.array([3600.0, 3000.0, 1800.0, 2.0])
    scale = np.linspace(0.5, 2.0, 18)
    net = pygfx.MLP(lo, hi, scale, n_freq=n_freq, width=width, depth=depth, seed=seed, batch=1024, sigma=1.0)
    w, B = net.params()
    ref = mlp_oracle.Model(w, B, n_freq, width, depth, lo, hi, scale)
    return net, ref, lo, hi


def test_mlp_forward_and_gradient_match_cpu_model():
    net, ref, lo, hi = _model_pair()
    rng = np.random.default_rng(5)
    x = lo + rng.random((200, 4)) * (hi - lo)
    y = rng.standard_normal((200, 18)).astype(np.float32)
    out = net.forward(x)
    want = ref.predict(x)
    err = np.linalg.norm(out - want) / np.linalg.norm(want)
    print(f"MLP forward rel L2 vs CPU model = {err:.3e}")
    assert err < 1e-3
    g, loss = net.gradient(x, y)
    lref, gref = ref.loss_grad(x, y)
    gerr = np.linalg.norm(g - gref) / np.linalg.norm(gref)
    print(f"MLP gradient rel L2 vs CPU model = {gerr:.3e}; loss {loss:.6g} vs {lref:.6g}")
    assert abs(loss - lref) <= 1e-4 * abs(lref)
    assert gerr < 2e-3
    # per layer block, so that no layer's gradient hides behind another's
    for off, iw, ow in ref.shapes:
        blk = slice(off, off + iw * ow + ow)
        assert np.linalg.norm(g[blk] - gref[blk]) <= 5e-3 * np.linalg.norm(gref[blk]) + 1e-12


def _envelope_np(x, y, cx, cy, r_max, env):
    """e(r): piecewise linear through env[i] at (i + 0.5) r_max / n, constant outside."""
    n = len(env)
    r = np.hypot(x - cx, y - cy)
    return np.interp(r, (np.arange(n) + 0.5) * r_max / n, env)


def test_envelope_scales_outputs_and_gradient_targets():
    net, ref, lo, hi = _model_pair()
    rng = np.random.default_rng(8)
    x = lo + rng.random((300, 4)) * (hi - lo)
    y = rng.standard_normal((300, 18)).astype(np.float32)
    plain = net.forward(x)
    g0, l0 = net.gradient(x, y)
    env = np.exp(-np.linspace(0.0, 3.0, 17)).astype(np.float32)
    cx, cy, r_max = 1200.0, 900.0, 4000.0
    net.set_envelope(cx, cy, r_max, env)
    e = _envelope_np(x[:, 0], x[:, 1], cx, cy, r_max, env.astype(np.float64))
    out = net.forward(x)
    assert np.allclose(out, plain * e[:, None], rtol=1e-5, atol=1e-6 * np.abs(plain).max())
    # the loss is taken on targets divided by the envelope: y * e gives the plain loss
    g1, l1 = net.gradient(x, (y * e[:, None]).astype(np.float32))
    assert abs(l1 - l0) <= 1e-4 * abs(l0)
    assert np.linalg.norm(g1 - g0) <= 1e-4 * np.linalg.norm(g0)
    # moveout: the time input becomes t - slowness * r
    s = 2e-4
    net.set_envelope(cx, cy, r_max, env, slowness=s)
    moved = net.forward(x)
    xs = x.copy()
    xs[:, 3] -= s * np.hypot(x[:, 0] - cx, x[:, 1] - cy)
    net.set_envelope(cx, cy, r_max, env)
    assert np.allclose(moved, net.forward(xs), rtol=1e-5, atol=1e-6 * np.abs(moved).max())
    assert not np.allclose(moved, out, rtol=1e-3)
    net.set_envelope(0, 0, 1, [])
    assert np.array_equal(net.forward(x), plain)
    with pytest.raises(pygfx.GfxError, match="> 0"):
        net.set_envelope(cx, cy, r_max, np.r_[env[:-1], 0.0])


def test_training_fits_a_smooth_tile(box):
    m, xyz, cidx = box
    nt = 8
    g = pygfx.GreenTile(nt, xyz, cidx)
    for t in range(nt):
        g.set_values(t, smooth_field(xyz, t * 0.25))
    lo = np.r_[xyz.min(axis=0), 0.0]
    hi = np.r_[xyz.max(axis=0), (nt - 1) * 0.25]
    net = pygfx.MLP(lo, hi, np.ones(18), n_freq=32, width=128, depth=3, batch=4096, lr=2e-3, sigma=1.0)
    l0 = net.train(g, 0.0, 0.25, 5)
    l1 = net.train(g, 0.0, 0.25, 3000)
    print(f"training loss {l0:.4g} -> {l1:.4g}")
    assert l1 < 0.1 * l0
    # the fit generalises between nodes: judge vs network at random points
    rng = np.random.default_rng(2)
    pts = xyz.min(axis=0) + rng.random((2000, 3)) * (xyz.max(axis=0) - xyz.min(axis=0))
    tix = rng.integers(0, nt, 2000).astype(np.int32)
    jv, _ = g.interpolate(pts, tix)
    mv = net.forward(np.c_[pts, tix * 0.25])
    rel = np.linalg.norm(mv - jv) / np.linalg.norm(jv)
    print(f"network vs judge rel L2 at random points = {rel:.3e}")
    assert rel < 0.2


def test_surrogate_query_falls_back_per_cell(box):
    m, xyz, cidx = box
    g = pygfx.GreenTile(2, xyz, cidx)
    for t in range(2):
        g.set_values(t, smooth_field(xyz, t))
    lo = np.r_[xyz.min(axis=0), 0.0]
    hi = np.r_[xyz.max(axis=0), 1.0]
    net = pygfx.MLP(lo, hi, np.ones(18), n_freq=8, width=32, depth=2, batch=256)
    rng = np.random.default_rng(4)
    pts = lo[:3] + rng.random((500, 3)) * (hi[:3] - lo[:3])
    tix = rng.integers(0, 2, 500).astype(np.int32)
    jv, cell = g.interpolate(pts, tix)
    mv = net.forward(np.c_[pts, tix * 1.0])
    allfb, n_all = net.query(g, np.ones(g.n_cell, np.uint8), 0.0, 1.0, pts, tix)
    assert n_all == 500 and np.array_equal(allfb, jv)
    nofb, n_none = net.query(g, np.zeros(g.n_cell, np.uint8), 0.0, 1.0, pts, tix)
    assert n_none == 0 and np.array_equal(nofb, mv)
    flags = (np.arange(g.n_cell) % 2).astype(np.uint8)
    mixed, n_mixed = net.query(g, flags, 0.0, 1.0, pts, tix)
    use = flags[cell].astype(bool)
    assert n_mixed == use.sum()
    assert np.array_equal(mixed[use], jv[use]) and np.array_equal(mixed[~use], mv[~use])


def test_surrogate_query_falls_back_per_cell_and_time_window(box):
    m, xyz, cidx = box
    nt, nw = 6, 3  # windows {0, 1}, {2, 3}, {4, 5}
    g = pygfx.GreenTile(nt, xyz, cidx)
    for t in range(nt):
        g.set_values(t, smooth_field(xyz, 0.5 * t))
    lo = np.r_[xyz.min(axis=0), 0.0]
    hi = np.r_[xyz.max(axis=0), 2.5]
    net = pygfx.MLP(lo, hi, np.ones(18), n_freq=8, width=32, depth=2, batch=256)
    rng = np.random.default_rng(9)
    pts = lo[:3] + rng.random((800, 3)) * (hi[:3] - lo[:3])
    tix = rng.integers(0, nt, 800).astype(np.int32)
    jv, cell = g.interpolate(pts, tix)
    mv = net.forward(np.c_[pts, tix * 0.5])
    flags = ((np.arange(g.n_cell)[:, None] + np.arange(nw)[None, :]) % 2).astype(np.uint8)
    out, n_fb = net.query(g, flags, 0.0, 0.5, pts, tix)
    use = flags[cell, tix * nw // nt].astype(bool)
    assert 0 < use.sum() < len(use) and n_fb == use.sum()
    assert np.array_equal(out[use], jv[use]) and np.array_equal(out[~use], mv[~use])


def test_green_capture_is_the_mass_weighted_merge_of_records():
    mesh = mc.small_halfspace(nx=6, ny=6, nz=4, pml=1, duration=0.5)
    cells, w, stf = mc.surface_centre_source(mesh)
    s = pygfx.Solver(mesh, n_fields=3, record_uva=False)
    for d in range(3):
        s.set_source(d, d, cells, w, stf)
    s.run(mesh.nsteps)
    nodes, xyz, cidx = tile_from_mesh(mesh, mesh.rec_cell)
    g = pygfx.GreenTile(s.n_snapshots, xyz, cidx)
    off, rp, wt = pygfx.green_capture_map(mesh, mesh.rec_cell, nodes)
    g.set_capture_map(off, rp, wt)
    ib = mesh.ibool.reshape(-1, 125)[mesh.rec_cell].ravel()
    mass = mesh.mass.reshape(-1, 125)[mesh.rec_cell].ravel()
    pos = np.searchsorted(nodes, ib)
    den = np.bincount(pos, weights=mass, minlength=len(nodes))
    for k in range(s.n_snapshots):
        g.capture(s, k, [0, 1, 2], k)
        got = g.get_values(k).reshape(len(nodes), 6, 3)
        for d in range(3):
            st = s.get_record(d, k).reshape(-1, 6)
            want = np.stack([np.bincount(pos, weights=mass * st[:, c], minlength=len(nodes)) for c in range(6)],
                            axis=1) / den[:, None]
            scale = np.abs(want).max() + 1e-30
            assert np.abs(got[:, :, d] - want).max() <= 1e-5 * scale
    # a direction left out stays zero
    g.capture(s, 0, [0, -1, 2], 0)
    assert np.abs(g.get_values(0).reshape(-1, 6, 3)[:, :, 1]).max() == 0.0


def test_tile_and_surrogate_pipeline_small():
    """Solver -> device tile -> trained network (envelope on) -> scored
    queries with the (cell, time window) fallback: the combined answer meets
    the bound the gate enforces on the validation queries (checked on an
    independent test set, with a factor 2 for validation noise), and the
    network is far smaller than the tile it replaces."""
    from pygfx import greens
    mesh = mc.small_halfspace(nx=8, ny=8, nz=5, pml=2, duration=1.5)
    stf = pygfx.ricker(1.0, 0.6, 1e20, mesh.dt, mesh.nsteps)
    xyz = (0.5 * (mesh.bounds[0] + mesh.bounds[1]), 0.5 * (mesh.bounds[2] + mesh.bounds[3]), 0.0)
    tile, info = greens.build_tile(mesh, xyz, stf, depth_max=1000.0, ring=4)
    assert info["samples"] == (mesh.nsteps + mesh.snapshot_stride - 1) // mesh.snapshot_stride
    res = greens.experiment(tile, info["dt_snap"], xyz[:2], iters=800, n_query=20000, n_valid=400000, n_window=4,
                            bound=0.01, n_freq=32, width=128, depth=3, batch=4096)
    print(res)
    assert 0.0 <= res["fallback_fraction"] <= 1.0
    assert res["rel_l2_with_fallback"] <= 0.02
    assert res["rel_l2_with_fallback"] <= res["rel_l2_mlp"]
    assert res["fallback_tile_bytes"] <= res["tile_bytes"]
    assert res["mlp_bytes_bf16"] < res["tile_bytes"]


def test_network_serves_regions_the_zero_predictor_cannot():
    """What the trained network adds over the method without it.  Without the
    network, a query gate can answer a (cell, time window) region with 0 where
    the region's values are within the error bound of 0, and must send every
    other region to the judge (stored tile + GLL interpolation).  With it, the
    gate also serves the regions where the network's validation error is
    within the bound.  On a small halfspace tile (0.5 Hz source, the network
    of the benchmark configuration: 64 frequencies, 6 x 256 GELU layers, 3000
    Adam iterations) the network serves regions the zero predictor cannot, the
    judge needs fewer tile bytes, and the combined answer stays within the
    bound (x 2 for validation-set noise) on an independent test set."""
    from pygfx import greens
    mesh = mc.small_halfspace(nx=8, ny=8, nz=5, pml=2, duration=2.5)
    stf = pygfx.ricker(0.5, 2.4, 1e20, mesh.dt, mesh.nsteps)
    xyz = (0.5 * (mesh.bounds[0] + mesh.bounds[1]), 0.5 * (mesh.bounds[2] + mesh.bounds[3]), 0.0)
    tile, info = greens.build_tile(mesh, xyz, stf, depth_max=1000.0, ring=4)
    res = greens.experiment(tile, info["dt_snap"], xyz[:2], iters=3000, n_query=20000, n_valid=400000, n_window=4,
                            bound=0.01, n_freq=64, width=256, depth=6, batch=4096)
    print({k: res[k] for k in ("rel_l2_mlp", "regions", "regions_served", "regions_served_by_zero",
                               "network_only_regions", "combined_network_fraction", "combined_zero_fraction",
                               "combined_judge_fraction", "combined_rel_l2", "combined_tile_bytes",
                               "zero_gate_tile_bytes", "tile_bytes")})
    assert res["network_only_regions"] > 0 and res["combined_network_fraction"] > 0.0
    assert res["combined_tile_bytes"] < res["zero_gate_tile_bytes"] <= res["tile_bytes"]
    assert res["combined_judge_fraction"] < 1.0 - res["combined_zero_fraction"]
    assert res["combined_rel_l2"] <= 0.02


@pytest.mark.parametrize("width,depth,n_freq,rows", [(16, 1, 1, 1), (48, 2, 10, 63), (100, 3, 13, 65), (64, 2, 32, 257),
                                                     (200, 2, 8, 1000), (320, 1, 70, 130), (50, 2, 5, 70)])
def test_mlp_products_at_tile_edges(width, depth, n_freq, rows):
    """Widths, feature counts and rows off the products' tiles (64, 128) and
    padding (64): forward and every gradient block against the CPU model, with
    the bars of the default shape (BF16 operands on both sides; only the order
    of the FP32 sums differs)."""
    net, ref, lo, hi = _model_pair(width=width, depth=depth, n_freq=n_freq)
    rng = np.random.default_rng(rows)
    x = lo + rng.random((rows, 4)) * (hi - lo)
    y = rng.standard_normal((rows, 18)).astype(np.float32)
    want = ref.predict(x)
    for _ in range(2):  # the second call finds the first one's activations in the buffers
        assert np.linalg.norm(net.forward(x) - want) < 1e-3 * np.linalg.norm(want)
    lref, gref = ref.loss_grad(x, y)
    for _ in range(2):
        g, loss = net.gradient(x, y)
        assert abs(loss - lref) <= 1e-4 * abs(lref)
        for off, iw, ow in ref.shapes:
            for b in (slice(off, off + iw * ow), slice(off + iw * ow, off + iw * ow + ow)):
                assert np.linalg.norm(g[b] - gref[b]) <= 5e-3 * np.linalg.norm(gref[b]) + 1e-12


def test_mlp_large_tiles_equal_small_tiles():
    """Enough rows for the 128 x 128 tiles: each output equals, bit for bit, the
    one a small call computes on 64 x 64 tiles (one output, the same products in
    the same order)."""
    net, _, lo, hi = _model_pair(width=256, depth=2, n_freq=16)
    rng = np.random.default_rng(2)
    x = lo + rng.random((33000, 4)) * (hi - lo)
    big = net.forward(x)
    for b in (0, 16384, 32900):
        assert np.array_equal(net.forward(x[b:b + 100]), big[b:b + 100])


def test_judge_groups_of_queries_equal_single_queries():
    """More than 8,192 queries run several to a wavefront; each answer is the one
    a small call gives, inside the tile, at its nodes and outside."""
    rng = np.random.default_rng(4)
    mesh = mc.small_halfspace(nx=4, ny=4, nz=3, pml=1)
    ib = mesh.ibool.reshape(-1, 125)
    nodes, inv = np.unique(ib.ravel(), return_inverse=True)
    xyz = mesh.node_xyz.reshape(-1, 3)[nodes]
    tile = pygfx.GreenTile(3, xyz, inv.reshape(-1, 125).astype(np.int32))
    for t in range(3):
        tile.set_values(t, rng.normal(size=(len(nodes), 18)).astype(np.float32))
    lo, hi = xyz.min(axis=0), xyz.max(axis=0)
    q = lo - 50.0 + rng.random((20001, 3)) * (hi - lo + 100.0)
    q[::37] = xyz[rng.integers(0, len(nodes), len(q[::37]))]
    tix = rng.integers(-1, 4, len(q)).astype(np.int32)
    out, cell = tile.interpolate(q, tix)
    assert (cell < 0).any() and (cell >= 0).any()
    for b in (0, 7777, 19990):
        o, c = tile.interpolate(q[b:b + 300], tix[b:b + 300])
        assert np.array_equal(c, cell[b:b + 300])
        assert np.array_equal(o, out[b:b + 300], equal_nan=True)
