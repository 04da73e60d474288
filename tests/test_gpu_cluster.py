"""The cluster kernel (GATHER assembly, wavefront element form) at the sizes
where its tables have edges: clusters of one element, of fewer than eight, odd
element counts per axis, elements in caller order (no centroids, runs of eight),
axis-aligned and general geometry, one and several fields, with and without
C-PML, forces whose cells share nodes across clusters.

Against the lane-per-point block kernel on the same mesh, which sums each
node's points in another order: both round in FP32, so after a few dozen steps
the states agree to some 1e-6 relative; the bars are 1e-5 for u and v and 1e-4
for the acceleration, which is a difference of much larger element forces."""
import ctypes as C
import os

import numpy as np
import pytest

import meshcases as mc
import pygfx

pytestmark = pytest.mark.gpu

GOLDEN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "images_without_clusters.npz")


def _run(mesh, nf, kernel, has_cpml, morton, steps=30):
    cells, w, stf = mc.buried_source(mesh, frac=(0.5, 0.5, 0.0), depth=0.4 * (mesh.bounds[5] - mesh.bounds[4]))
    s = pygfx.Solver(mesh, n_fields=nf, assembly=pygfx.GFX_ASSEMBLY_GATHER, element_kernel=kernel, has_cpml=has_cpml,
                     morton=morton, record_capacity=1, rec_cell=np.zeros(0, np.int32))
    rng = np.random.default_rng(3)
    for f in range(nf):
        s.set_source(f, f % 3, cells, w, stf)
        u, v = (rng.normal(size=mesh.n_node * 3) * k for k in (1e-3, 1e-2))
        s.set_state(f, u, v, np.zeros_like(u))
    s.run(steps)
    return [s.get_state(f) for f in range(nf)]


@pytest.mark.parametrize("nx,ny,nz,nf,jitter,has_cpml,morton", [
    (1, 1, 1, 1, 0.0, False, True),    # one element, every node interior
    (3, 1, 1, 2, 0.0, False, True),
    (3, 3, 2, 1, 0.2, False, True),
    (2, 2, 2, 3, 0.0, False, True),    # exactly one full cluster
    (5, 7, 3, 3, 0.0, True, True),
    (5, 4, 5, 1, 0.15, True, True),
    (4, 5, 3, 25, 0.0, True, False),   # runs of eight in caller order
    (9, 6, 7, 4, 0.1, True, False)])
def test_cluster_kernel_matches_block_kernel(nx, ny, nz, nf, jitter, has_cpml, morton):
    pml = 1 if has_cpml else 0
    mesh = pygfx.build_box(nx=nx, ny=ny, nz=nz, lx=600.0 * nx, ly=600.0 * ny, lz=600.0 * nz,
                           layers=[(900.0, 5000.0, 2900.0, 2500.0), (0.0, 6200.0, 3600.0, 2800.0)],
                           pml_xmin=pml, pml_xmax=pml, pml_ymin=pml, pml_ymax=pml, pml_zmax=pml, f0_pml=1.5,
                           jitter=jitter, jitter_seed=5, duration=1.0, record_depth_max=0.0)
    print(f"case: {nx}x{ny}x{nz}, {nf} fields, jitter {jitter}, cpml {has_cpml}, centroids {morton}", flush=True)
    a = _run(mesh, nf, pygfx.GFX_ELEMENT_AUTO, has_cpml, morton)
    b = _run(mesh, nf, pygfx.GFX_ELEMENT_BLOCK, has_cpml, morton)
    for x, y in zip(a, b):
        for p, q, bar in zip(x, y, (1e-5, 1e-5, 1e-4)):
            assert np.isfinite(p).all()
            assert mc.rel_l2(p, q) <= bar


@pytest.mark.parametrize("nf,has_cpml,n_sls", [(1, True, 0), (4, False, 0), (3, True, 2)])
def test_one_node_launch_equals_staged_launches(nf, has_cpml, n_sls):
    """Entries per element point: small meshes of few fields take all nodes in one
    launch; two field groups per workgroup keep the two staged launches.  The
    same sums in the same order: bit for bit."""
    mesh = mc.small_layered(duration=0.8, n_sls=n_sls, q_mu=[60.0, 90.0, 120.0], att_fmin=0.1, att_fmax=4.0)
    cells, w, stf = mc.buried_source(mesh)
    states = []
    for groups in (1, 2):
        s = pygfx.Solver(mesh, n_fields=nf, assembly=pygfx.GFX_ASSEMBLY_GATHER, element_kernel=pygfx.GFX_ELEMENT_BLOCK,
                         has_cpml=has_cpml, node_field_groups=groups)
        for f in range(nf):
            s.set_source(f, f % 3, cells, w, stf)
        s.run(25)
        states.append([s.get_state(f) for f in range(nf)])
    for a, b in zip(*states):
        for x, y in zip(a, b):
            assert np.any(y) and np.array_equal(x, y)


def test_switching_the_element_kernel_keeps_the_state():
    """A solver moved between the cluster and the block form mid-run (each has
    its own residual entries) continues from the same state, and the
    acceleration read after a switch is the last step's."""
    mesh = mc.small_layered(duration=0.8)
    cells, w, stf = mc.buried_source(mesh)
    s = pygfx.Solver(mesh, assembly=pygfx.GFX_ASSEMBLY_GATHER, record_capacity=1)
    s.set_source(0, 2, cells, w, stf)
    s.run(12)
    before = s.get_state(0)
    s.set_launch(pygfx.GFX_ELEMENT_BLOCK, 1)
    for x, y in zip(s.get_state(0), before):
        assert np.array_equal(x, y)
    image = s.checkpoint()
    s.run(5)
    s.set_launch(pygfx.GFX_ELEMENT_WAVE, 4)
    after = s.get_state(0)
    s.restore(image)
    for x, y in zip(s.get_state(0), before):
        assert np.array_equal(x, y)
    s.set_launch(pygfx.GFX_ELEMENT_BLOCK, 1)
    s.run(5)
    for x, y in zip(s.get_state(0), after):
        assert np.array_equal(x, y)


def _free_memory():
    free, total = C.c_size_t(0), C.c_size_t(0)
    assert pygfx.lib.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


class _DeviceMemory:
    """Holds all of the device's free memory but 256 to 320 MB."""

    def __init__(self):
        self.hip = pygfx.lib  # its own HIP runtime
        self.hip.hipMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t]
        self.hip.hipFree.argtypes = [C.c_void_p]
        self.held = []
        assert self._take(_free_memory() - (1 << 30))
        while self._take(64 << 20):  # what is reported as free may be less than there is
            assert len(self.held) < 500
        self.hip.hipGetLastError()
        for _ in range(4):
            self.hip.hipFree(self.held.pop())

    def _take(self, n):
        p = C.c_void_p()
        ok = self.hip.hipMalloc(C.byref(p), n) == 0
        if ok:
            self.held.append(p)
        return ok

    def close(self):
        while self.held:
            self.hip.hipFree(self.held.pop())


def test_a_switch_that_finds_no_memory_leaves_the_state():
    """The entries per point of a solver switched away from the cluster form do
    not fit beside what the device holds: the run is refused, the state and the
    acceleration stay readable, and the solver goes on in its earlier form."""
    mesh = pygfx.build_box(nx=10, ny=10, nz=10, lx=6000.0, ly=6000.0, lz=6000.0,
                           layers=[(0.0, 6200.0, 3600.0, 2800.0)], pml_xmin=0, pml_xmax=0, pml_ymin=0, pml_ymax=0,
                           pml_zmax=0, duration=0.2, record_depth_max=0.0)
    cells, w, stf = mc.buried_source(mesh, t0=0.02)
    nf, last = 2048, 2047  # 3.1 GB of entries per point, 2.2 GB per cluster
    solvers = [pygfx.Solver(mesh, n_fields=n, assembly=pygfx.GFX_ASSEMBLY_GATHER, has_cpml=False, record_capacity=0)
               for n in (nf, 1)]
    for s, f in zip(solvers, (last, 0)):
        s.set_source(f, 2, cells, w, stf)
        s.run(4)
    s, one = solvers
    hog = _DeviceMemory()
    try:
        s.set_launch(pygfx.GFX_ELEMENT_BLOCK, 1)
        with pytest.raises(pygfx.GfxError) as ei:
            s.run(1)
        assert ei.value.status == 4 and s.step == 4
        for x, y in zip(s.get_state(last), one.get_state(0)):
            assert np.any(y) and np.array_equal(x, y)
        s.set_launch(pygfx.GFX_ELEMENT_WAVE)
        s.run(1)
    finally:
        hog.close()
    one.run(1)
    for x, y in zip(s.get_state(last), one.get_state(0)):
        assert np.array_equal(x, y)
    for t in (s, one):
        t.set_launch(pygfx.GFX_ELEMENT_BLOCK, 1)
        t.run(1)
    for x, y in zip(s.get_state(last), one.get_state(0)):
        assert np.array_equal(x, y)


def test_both_forms_share_one_buffer_of_entries():
    """A solver that runs whole steps in the cluster form, stages and the block
    form by turns holds no more than the entries per point (what a solver in the
    block form holds), under graphs too, and gives the states of solvers that
    never switch between the two kinds of entries."""
    mesh = pygfx.build_box(nx=10, ny=10, nz=10, lx=6000.0, ly=6000.0, lz=6000.0,
                           layers=[(0.0, 6200.0, 3600.0, 2800.0)], pml_xmin=0, pml_xmax=0, pml_ymin=0, pml_ymax=0,
                           pml_zmax=0, duration=0.2, record_depth_max=0.0)
    cells, w, stf = mc.buried_source(mesh, t0=0.02)
    nf = 512
    point_bytes = mesh.n_elem * 125 * 12 * nf  # 768 MB

    def solver(graph):
        s = pygfx.Solver(mesh, n_fields=nf, assembly=pygfx.GFX_ASSEMBLY_GATHER, has_cpml=False, record_capacity=0)
        s.set_source(nf - 1, 2, cells, w, stf)
        s.set_graph(graph)
        return s

    def stages(s):
        step = s.step
        s.stage("newmark_predict", mesh.dt, 0.0)
        s.stage("zero_residual")
        s.stage("element_residual", 5, mesh.n_elem)
        s.stage("source_injection", nf - 1, 2, float(stf[step]), np.asarray(w, np.float64), len(cells))
        s.stage("scatter_to_rank")
        s.stage("newmark_correct", mesh.dt, 0.0, 0.5)

    for graph in (False, True):
        s, ref = solver(graph), solver(False)
        s.run(3)
        before = _free_memory()
        stages(s)
        s.run(2)
        stages(s)
        # entries per cluster are some three quarters of those per point; the plan's
        # tables are a few MB
        assert before - _free_memory() < 0.45 * point_bytes
        s.run(1)
        ref.run(8)  # one step is the same bits in stages and whole
        for x, y in zip(s.get_state(nf - 1), ref.get_state(nf - 1)):
            assert np.any(y) and np.array_equal(x, y)
        for t in (s, ref):
            t.set_launch(pygfx.GFX_ELEMENT_BLOCK, 1)
            t.run(2)
            t.set_launch(pygfx.GFX_ELEMENT_WAVE)
            t.run(2)
        assert before - _free_memory() < point_bytes  # of two solvers now
        for x, y in zip(s.get_state(nf - 1), ref.get_state(nf - 1)):
            assert np.array_equal(x, y)
        del s, ref


def image_case(form):
    """The solver of the stored images (tests/golden/README.md): axis-aligned and
    general elements, C-PML nodes of several direction sets, one recorded cell, a
    number of special nodes that is no multiple of four; memory per node or, with
    one element's coefficient changed, per element."""
    nx = 4 if form == "nodal" else 3
    mesh = pygfx.build_box(nx=nx, ny=2, nz=2, lx=700.0 * nx, ly=1500.0, lz=1300.0,
                           layers=[(700.0, 5000.0, 2900.0, 2500.0), (0.0, 6200.0, 3600.0, 2800.0)], pml_xmin=1,
                           pml_xmax=0, pml_ymin=0, pml_ymax=0, pml_zmax=1, f0_pml=1.5, duration=1.0,
                           record_depth_max=0.0)
    dd = mesh.dxi_dx.reshape(-1, 125, 9).copy()
    dd[::3, :, 1] = 1e-9 * dd[::3, :, 0]  # every third element takes the general form
    mesh = mesh.derive(dxi_dx=dd.reshape(-1))
    if form == "element":
        al = mesh.coef_alpha.reshape(-1, 125, 9).copy()
        use = (mesh.pml_region[:, None] != 0) & (mesh.coef_abar.reshape(-1, 125, 5)[:, :, 2] != 0)
        ids, n = np.unique(mesh.ibool.reshape(-1, 125)[use], return_counts=True)
        e, q = (int(x[0]) for x in np.nonzero(use & (mesh.ibool.reshape(-1, 125) == ids[n >= 2][0])))
        al[e, q, 0] *= 0.999
        mesh = mesh.derive(coef_alpha=al.reshape(-1))
    cells, w, stf = mc.buried_source(mesh, depth=500.0, t0=0.05)
    s = pygfx.Solver(mesh, n_fields=1, assembly=pygfx.GFX_ASSEMBLY_GATHER, record_capacity=1,
                     rec_cell=np.array([mesh.n_elem - 1], np.int32))
    s.set_source(0, 2, cells, w, stf)
    return mesh, s


@pytest.mark.parametrize("form", ["nodal", "element"])
def test_images_in_the_order_without_clusters_load(form):
    """An image taken before elements and nodes were ordered by clusters loads
    into the solver of the same inputs: the state it was taken at bit for bit,
    and five steps on from there the displacement reached then, to the
    rounding of another order of sums (1e-5)."""
    mesh, s = image_case(form)
    assert s.query("pml_nodal") == (form == "nodal")
    assert form == "element" or 0 < s.query("diag_elements") < mesh.n_elem
    with np.load(GOLDEN) as z:
        image, at, later = (z[f"{form}_{k}"] for k in ("image", "at", "later"))
    s.restore(image.tobytes())
    assert s.step == 6
    for x, y in zip(s.get_state(0), at):
        assert np.any(y) and np.array_equal(x, y.astype(np.float64))
    own = s.checkpoint()  # from here on in this solver's own order
    s.run(5)
    after = s.get_state(0)
    assert mc.rel_l2(after[0], later) <= 1e-5
    s.restore(own)
    s.run(5)
    for x, y in zip(s.get_state(0), after):
        assert np.array_equal(x, y)
    bad = image.copy()
    bad[56] ^= 1  # another numbering is refused
    with pytest.raises(pygfx.GfxError):
        s.restore(bad.tobytes())
