"""The library's host side on a stand-in HIP runtime (host_runtime.cpp):
which kernels it launches on which buffers, and what it does when an
allocation fails.  No GPU; each test runs in a process of its own, since the
stand-in takes the place of the HIP runtime there."""
import os
import subprocess
import sys

import pytest

from conftest import ROOT

PRELUDE = """
import ctypes as C
import sys
sys.path.insert(0, {root!r})
rt = C.CDLL({rt!r}, mode=C.RTLD_GLOBAL)
rt.rt_used.restype = C.c_size_t
rt.rt_limit.argtypes = [C.c_size_t]
rt.rt_host_limit.argtypes = [C.c_size_t]
rt.rt_log.restype = C.c_char_p
rt.rt_watch.argtypes = [C.c_char_p, C.c_int]
import numpy as np
from specfem3d_geotech_amd import _lib as L
from specfem3d_geotech_amd.batch import BatchEngine
from specfem3d_geotech_amd.mesh import slope_mesh
from specfem3d_geotech_amd.slope import DeviceSlope
from specfem3d_geotech_amd.solver import (K_F32, K_F64, KFMT_FULL, KFMT_PACKED, Context,
                                          DeviceMesh)
from specfem3d_geotech_amd.spec import hex2spec

def log():
    s = rt.rt_log().decode().splitlines()
    rt.rt_clear()
    return s

ctx = Context(0)
mesh = slope_mesh(3, 2, 2)
spec = hex2spec(mesh)
gam, ym, nu, phi, coh, psi = mesh.material_arrays()
"""
# leaves without the exit handlers of the HIP runtime that was loaded, but
# not used
EPILOGUE = """
import os
print("done", flush=True)
os._exit(0)
"""


@pytest.fixture(scope="module")
def runtime(tmp_path_factory):
    lib = str(tmp_path_factory.mktemp("runtime") / "libhostruntime.so")
    src = os.path.join(ROOT, "tests", "host_runtime.cpp")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__",
                    "-I/opt/rocm/include", src, "-o", lib], check=True)

    def run(body):
        code = PRELUDE.format(root=ROOT, rt=lib) + body + EPILOGUE
        r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True,
                           timeout=120)
        assert r.returncode == 0 and r.stdout.endswith("done\n"), r.stdout + r.stderr
    return run


# k_bmv_mfma's KP is its argument 3, k_bmf_lane's and k_bmf_point's geo their 2
@pytest.mark.parametrize("build_first", [True, False])
@pytest.mark.parametrize("ncol", [1, 64])
def test_autotune_after_the_stiffness_changed_hands(runtime, build_first, ncol):
    """An engine whose mesh got uploaded matrices after it was made on built
    ones, or the other way round, tunes the product that its mesh has now, on
    operands that exist."""
    runtime(f"""
dm = DeviceMesh(ctx, spec, len(gam))
n = spec.nelmt
def build():
    return dm.build_stiffness(gam, ym, nu)
def upload():
    dm.upload_stiffness(np.zeros((81, 81, n), order='F'), np.ones(spec.neq + 1))
ext, _ = build()
if not {build_first}:
    upload()
eng = BatchEngine(dm, ext, {ncol})
eng.set_graphs(False)
eng.begin(0, ym, nu, phi, coh, psi, 0.1)
eng.advance(1e-8, 100, 1e-4, 5e-4, 10, max_steps=8)
(upload if {build_first} else build)()
name, arg = ("k_bmv_mfma", 3) if {build_first} else ("k_bmf_", 2)
rt.rt_watch(name.encode(), arg)
log()
eng.autotune(2)
products = [s for s in log() if s.startswith("launch") and ("k_bmv_mfma" in s or "k_bmf_" in s)]
assert products
for s in products:
    assert name in s and s.split()[-1] != "0", s
""")


def test_failed_allocation_takes_the_kept_matrices_buffer(runtime):
    """Where device memory runs out while the matrices buffer of a closed
    mesh lies idle, the buffer goes and the call succeeds; where there is
    none, the call fails as out of memory and leaves nothing behind for the
    calls after it."""
    runtime("""
big = 8 * 6561 * spec.nelmt
dm = DeviceMesh(ctx, spec, len(gam))
dm.build_stiffness(gam, ym, nu)
dm.close()
rt.rt_limit(rt.rt_used() + 1000)
log()
dm = DeviceMesh(ctx, spec, len(gam))  # larger than what is left beside the buffer
s = log()
assert any(x.startswith("fail") for x in s) and "free %d" % big in s, s
rt.rt_limit(rt.rt_used() + 1000)
for call in (lambda: dm.build_stiffness(gam, ym, nu), lambda: DeviceMesh(ctx, spec, len(gam))):
    try:
        call()
        assert False, "no room for it"
    except RuntimeError as e:
        assert "failed: out of memory" in str(e), e
rt.rt_limit(1 << 40)
dm.build_stiffness(gam, ym, nu)
DeviceMesh(ctx, spec, len(gam)).close()
""")


def test_numbering_takes_the_kept_matrices_buffer(runtime):
    """The device numbering of the next mesh, too, gets memory that only the
    buffer of a closed mesh holds, whichever of its allocations fails first;
    where there is no buffer it fails and keeps nothing."""
    runtime("""
from specfem3d_geotech_amd.spec import hex2spec_device
mesh = slope_mesh(3, 2, 2)
big = 8 * 6561 * spec.nelmt
log()
hex2spec_device(ctx, mesh)
sizes = [int(x.split()[1]) for x in log() if x.startswith("malloc")]
assert len(sizes) > 15
for left in np.cumsum([0] + sizes[:-1]):
    dm = DeviceMesh(ctx, spec, len(gam))
    dm.build_stiffness(gam, ym, nu)
    dm.close()
    rt.rt_limit(rt.rt_used() + int(left))
    log()
    hex2spec_device(ctx, mesh)
    s = log()
    assert sum(x.startswith("fail") for x in s) == 1 and "free %d" % big in s, (left, s)
    rt.rt_limit(1 << 40)
    used = rt.rt_used()
    rt.rt_limit(used + int(left))
    try:
        hex2spec_device(ctx, mesh)
        assert False, "no room for it"
    except RuntimeError as e:
        assert "out of memory" in str(e), e
    assert rt.rt_used() == used
    rt.rt_limit(1 << 40)
    hex2spec_device(ctx, mesh)
""")


def test_failed_larger_mesh_leaves_the_others_their_partials(runtime):
    """A mesh that could not be made for want of memory leaves the context's
    reduction partials, which its other meshes use, as they were."""
    runtime("""
large = hex2spec(slope_mesh(40, 20, 30))
def make(sp):
    log()
    dm = DeviceMesh(ctx, sp, len(gam))
    return dm, [int(x.split()[1]) for x in log() if x.startswith("malloc")]
dm, sizes = make(large)
dm.close()
ctx.close()
ctx = Context(0)
dm, small = make(spec)
ext, _ = dm.build_stiffness(gam, ym, nu)
# the partials come last: everything before them fits
rt.rt_limit(rt.rt_used() + sum(sizes) - small[-1] - 1)
try:
    DeviceMesh(ctx, large, len(gam))
    assert False, "no room for it"
except RuntimeError as e:
    assert "out of memory" in str(e), e
rt.rt_limit(1 << 40)
rt.rt_watch(b"k_pcg_begin", 2)
log()
try:
    dm.solve(ext, cg_maxiter=1)  # no kernel runs, so no verdict
except RuntimeError:
    pass
begin = [x for x in log() if "k_pcg_begin" in x]
assert len(begin) == 1 and begin[0].split()[-1] != "0", begin
""")


@pytest.mark.parametrize("kprec", ["K_F64", "K_F32"])
def test_operator_whose_storage_failed_is_not_used(runtime, kprec):
    """Where the packed matrices of an operator could not be allocated (an
    upload onto a mesh that had none, a choice of operator), products and
    solves report that instead of reading matrices that are not there, and
    work once there is room."""
    runtime(f"""
dm = DeviceMesh(ctx, spec, len(gam))
ext, dinv = dm.build_stiffness(gam, ym, nu)
if {kprec} == K_F64:
    dm.set_operator(K_F64, KFMT_PACKED)  # from the geometry: nothing stored
    change = lambda: dm.upload_stiffness(np.zeros((81, 81, spec.nelmt), order='F'), dinv)
else:
    change = lambda: dm.set_operator({kprec}, KFMT_PACKED)
room = 20 * spec.neq
for call in (change, lambda: dm.matvec(ext), lambda: dm.solve(ext, cg_maxiter=1)):
    rt.rt_limit(rt.rt_used() + room)
    log()
    try:
        call()
        assert False, "no room for it"
    except RuntimeError as e:
        assert "out of memory" in str(e), e
    assert not [x for x in log() if "k_ebe" in x or "k_mf64" in x]
rt.rt_limit(1 << 40)
rt.rt_watch(b"k_ebe_packed", 1)
dm.matvec(ext)
s = [x for x in log() if "k_ebe_packed" in x]
assert len(s) == 1 and s[0].split()[-1] != "0", s
""")


def test_trials_find_their_matrices_packed(runtime):
    """A trial on the packed operator of a built mesh packs the matrices it
    multiplies when it is made, and a change of the stiffness packs them
    again: a plastic iteration neither allocates nor packs."""
    runtime("""
dm = DeviceMesh(ctx, spec, len(gam))
ext, dinv = dm.build_stiffness(gam, ym, nu)
dm.set_operator(K_F64, KFMT_PACKED)
assert not [x for x in log() if "k_pack_upper" in x]
t = DeviceSlope(dm, ext)
t.begin_srf(ym, nu, phi, coh, psi, 0.1)
assert len([x for x in log() if "k_pack_upper" in x]) == 1
def iterate():
    log()
    try:
        t.plastic_iter(1e-8, 1, 5e-4, False)  # no kernel runs, so no verdict
    except RuntimeError as e:
        assert "verdict" in str(e), e
    s = log()
    assert any("k_ebe_packed" in x for x in s), s
    assert not [x for x in s if "k_pack_upper" in x or x.startswith("malloc")], s
iterate()
for change in (lambda: dm.build_stiffness(gam, 2 * ym, nu),
               lambda: dm.upload_stiffness(np.zeros((81, 81, spec.nelmt), order='F'), dinv),
               lambda: dm.build_stiffness(gam, ym, nu)):
    change()
    assert len([x for x in log() if "k_pack_upper" in x]) == 1
    iterate()
""")


# ncol, elements: by points (reads no geometry), by lanes (the XCD split only)
# and uploaded matrices (both)
@pytest.mark.parametrize("grid,upload,distinct,pick", [((3, 2, 2), False, 1, (3, 1)),
                                                       ((12, 5, 5), False, 2, (3, 0)),
                                                       ((3, 2, 2), True, 8, (1, 0))])
def test_autotune_times_what_differs(runtime, grid, upload, distinct, pick):
    """Candidates that launch the same kernel the same way are timed once,
    and what the product does not read stays as it was (defaults: 3 blocks
    per CU, the XCD split).  Every timing here is shorter than the one
    before it."""
    runtime(f"""
mesh = slope_mesh(*{grid})
spec = hex2spec(mesh)
dm = DeviceMesh(ctx, spec, len(gam))
ext, dinv = dm.build_stiffness(gam, ym, nu)
if {upload}:
    dm.upload_stiffness(np.zeros((81, 81, spec.nelmt), order='F'), dinv)
eng = BatchEngine(dm, ext, 64)
eng.set_graphs(False)
eng.begin(0, ym, nu, phi, coh, psi, 0.1)
eng.advance(1e-8, 100, 1e-4, 5e-4, 10, max_steps=8)
log()
t = eng.autotune(3)
n = sum("k_bm" in x for x in log())
assert n == {distinct} * 4, n
assert (t["blocks_per_cu"], t["xcd_split"]) == {pick}, t
ms = [c["ms"] for c in t["candidates"]]
assert len(ms) == 8 and len(set(ms)) == {distinct} and t["ms"] == min(ms), t
""")


@pytest.mark.parametrize("pinned", [True, False])
def test_large_results_without_pinned_memory(runtime, pinned):
    """Results of several pieces arrive whole, through the pinned pieces or,
    where those cannot be had, by a plain copy that leaves no error behind."""
    runtime(f"""
dm = DeviceMesh(ctx, hex2spec(slope_mesh(10, 5, 3)), len(gam))  # K of 7.9 MB
n = dm.spec.nelmt
k = np.random.default_rng(1).normal(size=(n, 81 * 81))
if not {pinned}:
    rt.rt_host_limit(1 << 16)
dm.upload_stiffness(k, np.ones(dm.spec.neq + 1))
for _ in range(2):
    assert np.array_equal(np.ravel(dm.download_stiffness()), np.ravel(k))
dm.set_operator(K_F64, KFMT_PACKED)
""")
