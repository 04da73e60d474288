"""Host-side solver set-up without a device.

gfx_solver_create builds its whole host plan (element order, node numbering
with the C-PML direction-mask grouping, nodal C-PML coefficients, gather
slots, recording tables) and checks its invariants before the first device
call, so on a machine with no HIP device the call must end in
GFX_ERR_DEVICE ("no HIP device available"), never in an internal check or a
crash.  A numbering that is not a permutation of the nodes (a node queued
once per element that touches it) fails the plan's own check instead."""
import os
import shutil
import subprocess

import numpy as np
import pytest

import meshcases as mc
import pygfx

GFX_ERR_DEVICE = 2


@pytest.fixture(scope="module", autouse=True)
def _no_device():
    if pygfx.device_count() > 0:
        pytest.skip("a HIP device is visible: the device-free path is not reached")


@pytest.mark.parametrize("assembly", [pygfx.GFX_ASSEMBLY_COLORED, pygfx.GFX_ASSEMBLY_ATOMIC,
                                      pygfx.GFX_ASSEMBLY_GATHER])
@pytest.mark.parametrize("has_cpml", [True, False])
def test_create_plans_fully_before_the_device_check(assembly, has_cpml):
    mesh = mc.small_layered(nx=5, ny=4, nz=4, pml=1)
    with pytest.raises(pygfx.GfxError) as ei:
        pygfx.Solver(mesh, n_fields=3, assembly=assembly, has_cpml=has_cpml, record_capacity=2)
    assert ei.value.status == GFX_ERR_DEVICE, str(ei.value)
    assert "no HIP device" in str(ei.value)


def test_create_still_rejects_bad_arguments_first():
    mesh = mc.small_halfspace(nx=4, ny=4, nz=3, pml=1)
    with pytest.raises(pygfx.GfxError, match="elems_per_block"):
        pygfx.Solver(mesh, elems_per_block=3)
    with pytest.raises(pygfx.GfxError, match="pair element kernel"):
        pygfx.Solver(mesh, n_fields=2, element_kernel=pygfx.GFX_ELEMENT_PAIR, elems_per_block=8)
    with pytest.raises(pygfx.GfxError, match="elems_per_block must be 0"):
        pygfx.Solver(mesh, element_kernel=pygfx.GFX_ELEMENT_PENCIL, elems_per_block=2)
    with pytest.raises(pygfx.GfxError, match="unknown element kernel"):
        pygfx.Solver(mesh, element_kernel=5)
    good = mesh.arrays["ibool"]
    bad = np.array(good, copy=True)
    bad.reshape(-1)[7] = mesh.n_node
    mesh.arrays["ibool"] = bad
    try:
        with pytest.raises(pygfx.GfxError, match="ibool"):
            pygfx.Solver(mesh)
    finally:
        mesh.arrays["ibool"] = good


@pytest.mark.parametrize("assembly", [pygfx.GFX_ASSEMBLY_COLORED, pygfx.GFX_ASSEMBLY_GATHER])
def test_complete_cpml_plans_and_rejects_bad_inputs(assembly):
    mesh = mc.small_layered(nx=5, ny=4, nz=4, pml=1, want_profiles=1, pml_profile=1)
    with pytest.raises(pygfx.GfxError) as ei:
        pygfx.Solver(mesh, n_fields=2, assembly=assembly, cpml_complete=True, record_capacity=2)
    assert ei.value.status == GFX_ERR_DEVICE, str(ei.value)
    with pytest.raises(pygfx.GfxError, match="needs has_cpml"):
        pygfx.Solver(mesh, cpml_complete=True, has_cpml=False)
    bad = mesh.derive(pml_K=np.where(np.arange(mesh.pml_K.size) == 3 * 125 * 2 + 1, 0.0, mesh.pml_K))
    with pytest.raises(pygfx.GfxError, match="pml_K must be > 0"):
        pygfx.Solver(bad, cpml_complete=True)
    bad = mesh.derive(pml_alpha=-mesh.pml_alpha)
    with pytest.raises(pygfx.GfxError, match="pml_alpha >= 0"):
        pygfx.Solver(bad, cpml_complete=True)
    no_profiles = mc.small_layered(nx=5, ny=4, nz=4, pml=1)
    with pytest.raises(ValueError, match="want_profiles"):
        pygfx.Solver(no_profiles, cpml_complete=True)


@pytest.mark.parametrize("nx,ny,nz,morton", [(1, 1, 1, True), (3, 1, 2, True), (2, 2, 2, False), (5, 7, 3, True),
                                             (9, 6, 7, False)])
def test_cluster_tables_plan_at_every_size(nx, ny, nz, morton):
    """The cluster form's tables (partial clusters, odd counts, caller order)
    pass the plan's own checks: every point listed once, the interior nodes one
    run of ids per cluster."""
    mesh = pygfx.build_box(nx=nx, ny=ny, nz=nz, lx=600.0 * nx, ly=600.0 * ny, lz=600.0 * nz,
                           layers=[(0.0, 6200.0, 3600.0, 2800.0)], pml_xmin=0, pml_xmax=0, pml_ymin=0, pml_ymax=0,
                           pml_zmax=0, duration=1.0, record_depth_max=0.0)
    with pytest.raises(pygfx.GfxError) as ei:
        pygfx.Solver(mesh, assembly=pygfx.GFX_ASSEMBLY_GATHER, has_cpml=False, morton=morton, record_capacity=0)
    assert ei.value.status == GFX_ERR_DEVICE, str(ei.value)


_LOOP = """
#include <atomic>
#include "common.hpp"
int main() {
    using gfx::parallel_for;
    std::atomic<int> done{0};
    bool caught = false;
    try {  // two workers fail, the others finish
        parallel_for(8192, [&](int64_t i) {
            if (i == 5 || i == 8000) throw gfx::Error(GFX_ERR_NOMEM, "no memory");
            ++done;
        }, 8);
    } catch (const gfx::Error& e) {
        caught = e.code == GFX_ERR_NOMEM;
    }
    if (!caught || done < 6 * 1024) return 1;
    done = 0;
    parallel_for(8191, [&](int64_t) { ++done; }, 5);
    if (done != 8191) return 2;
    done = 0;  // few items of much work each: workers by the grain
    parallel_for(70, [&](int64_t) { ++done; }, 4, 16);
    return done == 70 ? 0 : 3;
}
"""


def test_an_exception_in_a_worker_reaches_the_caller(tmp_path):
    """The host plan's loops allocate inside their workers: a failure there is an
    error of the call, not the end of the process."""
    if shutil.which("g++") is None:
        pytest.skip("no g++")
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    src, exe = tmp_path / "loop.cpp", tmp_path / "loop"
    src.write_text(_LOOP)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-pthread", "-I", os.path.join(root, "include"), "-I",
                    os.path.join(root, "gf-only-sem_amd", "csrc"), str(src), "-o", str(exe)], check=True)
    assert subprocess.run([str(exe)]).returncode == 0
