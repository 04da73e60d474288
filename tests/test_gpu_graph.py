"""Graph-captured steps and batches of uneven meshes, on the GPU.

A captured step is replayed many times with the program's own eager work
(state reads, record reads, synchronisations) between the replays; every
replay must equal the kernel-by-kernel run bit for bit.  A batch of meshes of
different size, material, C-PML thickness, time step and run length, advanced
as one graph (one branch per mesh, or launches shared by all meshes), must
reproduce each mesh's single run bit for bit, and one of them is checked
against the FP64 oracle."""
import numpy as np
import pytest

import meshcases as mc
import pygfx
import pyoracle

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if pygfx.device_count() < 1:
        pytest.fail("no HIP device visible; GPU tests must run on an MI355X box")


def _solver(mesh, sources, assembly, graph=False, **kw):
    s = pygfx.Solver(mesh, n_fields=len(sources), assembly=assembly, record_uva=True, **kw)
    for f, (cells, w, stf, d) in enumerate(sources):
        s.set_source(f, d, cells, w, stf)
    if graph:
        s.set_graph(True)
    return s


def _all_records(s, n_snap):
    return [s.get_record(f, k, uva=True) for f in range(s.n_fields) for k in range(n_snap)]


@pytest.mark.parametrize("assembly", [pygfx.GFX_ASSEMBLY_COLORED, pygfx.GFX_ASSEMBLY_GATHER])
def test_graph_replays_equal_eager_steps(assembly):
    mesh = mc.small_layered(duration=1.0)
    cells, w, stf = mc.buried_source(mesh)
    c2, w2, stf2 = mc.buried_source(mesh, frac=(0.4, 0.6, 0.0), depth=900.0)
    src = [(cells, w, stf, 2), (c2, w2, stf2, 0)]
    eager = _solver(mesh, src, assembly)
    graph = _solver(mesh, src, assembly, graph=True)
    done = 0
    for chunk in (1, 5, 3, 17, mesh.nsteps):
        chunk = min(chunk, mesh.nsteps - done)
        if chunk <= 0:
            break
        eager.run(chunk)
        graph.run(chunk)
        done += chunk
        assert graph.step == eager.step == done
        for f in range(2):  # eager reads between replays
            for x, y in zip(graph.get_state(f), eager.get_state(f)):
                assert np.array_equal(x, y)
    assert graph.n_snapshots == eager.n_snapshots
    for a, b in zip(_all_records(graph, graph.n_snapshots), _all_records(eager, eager.n_snapshots)):
        for x, y in zip(a, b):
            assert np.array_equal(x, y)


def test_graph_is_recaptured_after_launch_and_source_changes():
    mesh = mc.small_halfspace(duration=0.6)
    cells, w, stf = mc.surface_centre_source(mesh)
    eager = _solver(mesh, [(cells, w, stf, 2)], pygfx.GFX_ASSEMBLY_GATHER)
    graph = _solver(mesh, [(cells, w, stf, 2)], pygfx.GFX_ASSEMBLY_GATHER, graph=True)
    for s in (eager, graph):
        s.run(10)
        s.set_launch(pygfx.GFX_ELEMENT_BLOCK, 4, node_field_groups=2)
        s.run(10)
        s.set_source(0, 1, cells, w, 0.5 * stf)  # new source arrays on the device
        s.run(mesh.nsteps - 20)
    for x, y in zip(graph.get_state(0), eager.get_state(0)):
        assert np.array_equal(x, y)


def _uneven_meshes():
    """Three boxes of different size, layering, C-PML thickness, dt and length."""
    m0 = mc.small_halfspace(nx=6, ny=6, nz=4, pml=1, duration=0.8)
    m1 = mc.small_layered(nx=9, ny=7, nz=5, pml=2, duration=1.2)
    m2 = pygfx.build_box(nx=7, ny=5, nz=5, lx=4200.0, ly=3000.0, lz=3000.0,
                         layers=[(1200.0, 3000.0, 1700.0, 2300.0), (0.0, 5200.0, 3000.0, 2900.0)],
                         pml_xmin=3, pml_xmax=1, pml_ymin=1, pml_ymax=1, pml_zmax=2, f0_pml=1.5,
                         duration=0.5, record_depth_max=1200.0)
    return [m0, m1, m2]


@pytest.mark.parametrize("assembly,groups", [(pygfx.GFX_ASSEMBLY_COLORED, 2), (pygfx.GFX_ASSEMBLY_GATHER, 0),
                                             (pygfx.GFX_ASSEMBLY_GATHER, 1), (pygfx.GFX_ASSEMBLY_GATHER, 2)])
def test_batch_of_uneven_meshes_equals_single_runs(assembly, groups):
    """GATHER batches share one launch per stage among the meshes of a launch
    group; COLORED ones, and GATHER with groups=0, keep one branch per mesh."""
    meshes = _uneven_meshes()
    assert len({m.dt for m in meshes}) > 1 and len({m.nsteps for m in meshes}) == 3
    srcs = []
    for m in meshes:
        cells, w, stf = mc.surface_centre_source(m, f0=1.5, t0=0.3)
        srcs.append([(cells, w, stf, 2), (cells, w, stf, 0)])
    batched = [_solver(m, s, assembly) for m, s in zip(meshes, srcs)]
    single = [_solver(m, s, assembly) for m, s in zip(meshes, srcs)]
    batch = pygfx.Batch(batched, groups=groups)
    until = [m.nsteps for m in meshes]
    # in pieces, with eager reads in between
    batch.run(7, until)
    assert batch.last_groups == (groups if assembly == pygfx.GFX_ASSEMBLY_GATHER else 0)
    for s in batched:
        s.get_state(0)
    batch.run(10 ** 6, until)
    for s, m in zip(batched, meshes):
        assert s.step == m.nsteps
    for s, m in zip(single, meshes):
        s.run(m.nsteps)
    for b, s in zip(batched, single):
        assert b.n_snapshots == s.n_snapshots
        for f in range(2):
            for x, y in zip(b.get_state(f), s.get_state(f)):
                assert np.array_equal(x, y)
        for x, y in zip(_all_records(b, b.n_snapshots), _all_records(s, s.n_snapshots)):
            for p, q in zip(x, y):
                assert np.array_equal(p, q)
    # one instance against the FP64 oracle
    m = meshes[1]
    cells, w, stf, d = srcs[1][0]
    ref = pyoracle.Run(m.arrays, m.n_elem, 5, m.n_node, m.dt, m.nsteps, m.snapshot_stride, d, cells, w, stf,
                       m.rec_cell).run()["strain"]
    got = np.stack([batched[1].get_record(0, k) for k in range(batched[1].n_snapshots)])
    err = mc.rel_l2(got, ref)
    print(f"batched instance strain rel L2 vs oracle = {err:.3e}")
    assert err <= 1e-4
    batch.close()


@pytest.mark.parametrize("pieces", [(4,), (3, 5, 4), (9, 1, 8)])
def test_group_steps_chained_in_one_graph_equal_single_runs(pieces):
    """A group's graph holds four steps: runs shorter, equal and longer than
    that, one mesh ending between, give every run's state (residuals of the last
    step included) and records bit for bit."""
    meshes = _uneven_meshes()
    srcs = [[mc.surface_centre_source(m, f0=1.5, t0=0.02) + (2,)] for m in meshes]
    batched = [_solver(m, s, pygfx.GFX_ASSEMBLY_GATHER) for m, s in zip(meshes, srcs)]
    single = [_solver(m, s, pygfx.GFX_ASSEMBLY_GATHER) for m, s in zip(meshes, srcs)]
    until = [10 ** 6, 6, 10 ** 6]
    batch = pygfx.Batch(batched, groups=2)
    for n in pieces:
        batch.run(n, until)
        for b, s, u in zip(batched, single, until):
            s.run(max(0, min(n, u - s.step)))
            assert b.step == s.step and b.n_snapshots == s.n_snapshots
            for x, y in zip(b.get_state(0), s.get_state(0)):
                assert np.array_equal(x, y)
            for x, y in zip(_all_records(b, b.n_snapshots), _all_records(s, s.n_snapshots)):
                for p, q in zip(x, y):
                    assert np.array_equal(p, q)
    batch.close()


@pytest.mark.parametrize("kernel", [pygfx.GFX_ELEMENT_BLOCK, pygfx.GFX_ELEMENT_WAVE])
@pytest.mark.parametrize("n_fields", [(3, 6), (6, 3), (1, 5, 4)])
def test_launch_group_of_different_field_counts_equals_single_runs(kernel, n_fields):
    """One launch group of solvers with few and with many fields: each gives
    its single run's state and records bit for bit, whichever comes first."""
    meshes = _uneven_meshes()[:len(n_fields)]
    batched, single = [], []
    for m, nf in zip(meshes, n_fields):
        cells, w, stf = mc.surface_centre_source(m, f0=1.5, t0=0.02)
        src = [(cells, w, stf * (1.0 + f), f % 3) for f in range(nf)]
        for to in (batched, single):
            to.append(_solver(m, src, pygfx.GFX_ASSEMBLY_GATHER, element_kernel=kernel))
    batch = pygfx.Batch(batched, groups=1)
    for n in (1, 6):
        batch.run(n)
        assert batch.last_groups == 1
        for b, s in zip(batched, single):
            s.run(n)
            assert b.step == s.step and b.n_snapshots == s.n_snapshots
            for f in range(s.n_fields):
                for x, y in zip(b.get_state(f), s.get_state(f)):
                    assert np.any(y) or s.step == 1  # u after the first step is zero
                    assert np.array_equal(x, y)
            for x, y in zip(_all_records(b, b.n_snapshots), _all_records(s, s.n_snapshots)):
                for p, q in zip(x, y):
                    assert np.array_equal(p, q)
    batch.close()


def _with_a_repeated_node(mesh):
    """The mesh with one element that has a node twice (a corner it shared with
    other elements replaced by the next point): no clusters then."""
    ib = mesh.ibool.reshape(-1, 125).copy()
    e = mesh.n_elem // 2
    corner = next(p for p in (0, 20, 100, 120) if np.count_nonzero(ib == ib[e, p]) > 1)
    ib[e, corner] = ib[e, corner + 1]
    return mesh.derive(ibool=ib)


@pytest.mark.parametrize("repeated", [(True, True), (True, False)])
def test_wave_solvers_without_clusters_share_launch_groups(repeated):
    """Solvers in the wave form whose mesh allows no clusters share launches, with
    each other and with cluster solvers, and equal their single runs."""
    meshes = [_with_a_repeated_node(m) if r else m for m, r in zip(_uneven_meshes(), repeated)]
    batched, single = [], []
    for m in meshes:
        cells, w, stf = mc.surface_centre_source(m, f0=1.5, t0=0.02)
        for to in (batched, single):
            to.append(_solver(m, [(cells, w, stf, 2), (cells, w, stf, 0)], pygfx.GFX_ASSEMBLY_GATHER,
                              element_kernel=pygfx.GFX_ELEMENT_WAVE))
    batch = pygfx.Batch(batched, groups=1)
    for n in (1, 6):
        batch.run(n)
        assert batch.last_groups == 1
        for b, s in zip(batched, single):
            s.run(n)
            for f in range(2):
                for x, y in zip(b.get_state(f), s.get_state(f)):
                    assert np.isfinite(y).all() and np.array_equal(x, y)
    batch.close()


@pytest.mark.parametrize("groups", [0, 1])
def test_batch_recaptures_after_a_member_was_driven_by_stages(groups):
    """A member driven stage by stage between batch runs has a larger buffer of
    residual entries afterwards; the batch's captured steps follow it."""
    meshes = _uneven_meshes()[:2]
    srcs = [[mc.surface_centre_source(m, f0=1.5, t0=0.02) + (2,)] for m in meshes]
    batched = [_solver(m, s, pygfx.GFX_ASSEMBLY_GATHER) for m, s in zip(meshes, srcs)]
    single = [_solver(m, s, pygfx.GFX_ASSEMBLY_GATHER) for m, s in zip(meshes, srcs)]
    batch = pygfx.Batch(batched, groups=groups)
    for n in (5, 6, 1):
        batch.run(n)
        m, (cells, w, stf, d), s = meshes[0], srcs[0][0], batched[0]
        step = s.step
        s.stage("newmark_predict", m.dt, 0.0)
        s.stage("element_residual", 5, m.n_elem)
        s.stage("source_injection", 0, d, float(stf[step]), np.asarray(w, np.float64), len(cells))
        s.stage("scatter_to_rank")
        s.stage("newmark_correct", m.dt, 0.0, 0.5)
        single[0].run(n + 1)
        single[1].run(n)
        for b, t in zip(batched, single):
            assert b.step == t.step
            for x, y in zip(b.get_state(0), t.get_state(0)):
                assert np.any(y) and np.array_equal(x, y)
    batch.close()


@pytest.mark.parametrize("groups", [0, 1])
def test_batch_after_a_switch_of_the_element_kernel(groups):
    """The entries of another element form are made by the batch's first run: many
    fields, so that clearing them takes as long as the first launches."""
    meshes = _uneven_meshes()[:2]
    batched, single = [], []
    for m in meshes:
        cells, w, stf = mc.surface_centre_source(m, f0=1.5, t0=0.02)
        for to in (batched, single):
            s = pygfx.Solver(m, n_fields=256, assembly=pygfx.GFX_ASSEMBLY_GATHER, record_capacity=0)
            for f in (0, 255):
                s.set_source(f, f % 3, cells, w, stf)
            s.run(3)
            to.append(s)
    batch = pygfx.Batch(batched, groups=groups)
    for s in batched + single:
        s.set_launch(pygfx.GFX_ELEMENT_BLOCK, 1)
    batch.run(4)
    for b, s in zip(batched, single):
        s.run(4)
        for f in (0, 255):
            for x, y in zip(b.get_state(f), s.get_state(f)):
                assert np.any(y) and np.array_equal(x, y)
    batch.close()


def test_launch_groups_fall_back_to_branches_when_a_mesh_cannot_share():
    """An attenuating mesh runs its own element kernel form, so a batch holding
    one keeps one branch per mesh even with launch groups requested; dropping it
    from the active set (its run is over) lets the rest share launches."""
    m0 = mc.small_halfspace(nx=6, ny=6, nz=4, pml=1, duration=0.3)
    m1 = mc.small_layered(duration=0.8, n_sls=2, q_mu=[30.0, 30.0, 30.0], att_fmin=0.1, att_fmax=4.0)
    m2 = mc.small_halfspace(nx=7, ny=6, nz=4, pml=1, duration=0.6)
    meshes = [m0, m1, m2]
    srcs = [[mc.surface_centre_source(m) + (2,)] for m in meshes]
    batched = [_solver(m, s, pygfx.GFX_ASSEMBLY_GATHER) for m, s in zip(meshes, srcs)]
    single = [_solver(m, s, pygfx.GFX_ASSEMBLY_GATHER) for m, s in zip(meshes, srcs)]
    assert int(batched[1].query("n_sls")) == 2
    until = [40, 20, 40]
    batch = pygfx.Batch(batched, groups=1)
    batch.run(10, until)
    assert batch.last_groups == 0  # the attenuating mesh is active
    batch.run(10 ** 6, until)
    assert batch.last_groups == 1  # meshes 0 and 2 alone
    for b, s, n in zip(batched, single, until):
        s.run(n)
        for x, y in zip(b.get_state(0), s.get_state(0)):
            assert np.array_equal(x, y)
    batch.close()
