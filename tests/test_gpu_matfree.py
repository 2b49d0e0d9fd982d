"""Products of built meshes formed from the geometry instead of the stored
element matrices, against the stored full FP64 operator (the reference's
matrices bit for bit) and against uploaded matrices, on element counts at
the edges of the kernels' element groups."""
import numpy as np
import pytest

from specfem3d_geotech_amd.mesh import Material, slope_mesh
from specfem3d_geotech_amd.solver import K_F64, KFMT_FULL, KFMT_PACKED, DeviceMesh
from specfem3d_geotech_amd.spec import hex2spec

pytestmark = pytest.mark.gpu

SOILS = [Material(gam=20.0, ym=1e5, nu=0.3, phi=25.0, coh=8.0),
         Material(gam=19.0, ym=7e4, nu=0.45, phi=30.0, coh=20.0)]


def _mesh(nx, ny, nz):
    return slope_mesh(nx, ny, nz, materials=SOILS, layer_z=[10.0], jitter=0.1, seed=4)


def rel_l2(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


# 1, 8, 9, 10, 63, 72, 73 (nine elements per block, blocks in eights), 1,500
@pytest.mark.parametrize("grid", [(1, 1, 1), (2, 2, 2), (3, 3, 1), (5, 2, 1), (7, 3, 3),
                                  (6, 4, 3), (73, 1, 1), (20, 5, 15)])
def test_packed_product_from_geometry(ctx, grid):
    """K p of the packed operator of a built mesh equals the stored full
    operator's to FP64 rounding: each side sums a few hundred rounded terms
    per entry, of random sign, so well below 1e-14 of the result."""
    mesh = _mesh(*grid)
    spec = hex2spec(mesh)
    gam, ym, nu, *_ = mesh.material_arrays()
    dm = DeviceMesh(ctx, spec, len(gam))
    try:
        _, dinv = dm.build_stiffness(gam, ym, nu)
        p = np.random.default_rng(2).normal(size=spec.neq + 1)
        p[0] = 0.0
        dm.set_operator(K_F64, KFMT_FULL)
        full = dm.matvec(p)
        dm.set_operator(K_F64, KFMT_PACKED)
        assert rel_l2(dm.matvec(p), full) < 1e-14
        # uploaded matrices are applied as they are, not from the geometry
        k = 3.0 * dm.download_stiffness()
        dm.upload_stiffness(k, dinv)
        assert rel_l2(dm.matvec(p), 3.0 * full) < 1e-14
        # and a rebuild applies the new materials
        dm.build_stiffness(gam, 2.0 * ym, nu)
        assert rel_l2(dm.matvec(p), 2.0 * full) < 1e-14
    finally:
        dm.close()


# 2^18 equations is where the blocks of the vector kernels change; the small
# grids have fewer equations than the product has shares of p.Kp
@pytest.mark.parametrize("grid,full", [((1, 1, 1), True), ((2, 1, 1), True), ((4, 2, 3), True),
                                       ((37, 7, 19), False), ((40, 10, 27), False),
                                       ((41, 10, 27), True)])
def test_solve_against_separate_reference_order(ctx, grid, full):
    """The tree-reduced solve equals the reference-order one at a tight
    tolerance: both stop at relative updates of 1e-13, so they differ by a
    few hundred such updates at most."""
    from specfem3d_geotech_amd.solver import REDUCE_SEQUENTIAL, REDUCE_TREE
    mesh = _mesh(*grid)
    spec = hex2spec(mesh)
    gam, ym, nu, *_ = mesh.material_arrays()
    dm = DeviceMesh(ctx, spec, len(gam))
    try:
        ext, _ = dm.build_stiffness(gam, ym, nu)
        dm.set_operator(K_F64, KFMT_FULL if full else KFMT_PACKED)
        cap = 20000 if spec.neq < 5000 else 40
        u, it, ec = dm.solve(ext, cg_tol=1e-13, cg_maxiter=cap)
        ctx.set_reduction(REDUCE_SEQUENTIAL)
        v, jt, fc = dm.solve(ext, cg_tol=1e-13, cg_maxiter=cap)
        # a warm start goes through the first residual's product
        w, _, _ = dm.solve(ext, u0=v, cg_tol=1e-13, cg_maxiter=cap)
        ctx.set_reduction(REDUCE_TREE)
        x, _, _ = dm.solve(ext, u0=v, cg_tol=1e-13, cg_maxiter=cap)
        assert ec == fc and abs(it - jt) <= 0.02 * jt
        assert rel_l2(u, v) < 1e-10
        assert rel_l2(x, w) < 1e-10
        # at most two iterations
        assert dm.solve(ext, cg_tol=1e-13, cg_maxiter=1)[1:] == (2, -1)
        assert dm.solve(ext, cg_tol=1e-13, cg_maxiter=17)[1] <= 18
    finally:
        ctx.set_reduction(REDUCE_TREE)
        dm.close()


def _engine_x(ctx, mesh, spec, ncol, steps, upload=False, cols=1):
    """x of column 0 after exactly `steps` CG steps of `cols` columns of the
    elastic solve."""
    from specfem3d_geotech_amd.batch import DEFAULT_INNER_TOL, BatchEngine, device_mesh
    from specfem3d_geotech_amd.plastic import dt_viscoplas
    _, ym, nu, phi, coh, psi = mesh.material_arrays()
    dm, ext = device_mesh(ctx, mesh, spec)
    try:
        if upload:
            _, dinv = dm.build_stiffness(mesh.material_arrays()[0], ym, nu)
            dm.upload_stiffness(dm.download_stiffness(), dinv)
        eng = BatchEngine(dm, ext, ncol)
        try:
            for j in range(cols):
                eng.begin(j, ym, nu, phi, coh, psi, dt_viscoplas(nu, phi, ym))
            if steps:
                eng.advance(1e-14, 5000, DEFAULT_INNER_TOL, 5e-4, 300, max_steps=steps)
            else:
                eng.plastic_iter(np.zeros(ncol, np.int32), 1e-12, 20000, DEFAULT_INNER_TOL, 5e-4)
            return eng.download(0)[0]
        finally:
            eng.close()
    finally:
        dm.close()


def test_batched_product_same_bits_for_every_column_count(ctx):
    """A column's bits do not depend on the engine's column count: 1 to 64
    columns on 65,600 elements (a lane per element and column) and on 1,025
    (64 columns by lanes, fewer by points), with idle columns beside it."""
    for grid, steps in (((41, 40, 40), 16), ((41, 5, 5), 24)):
        mesh = _mesh(*grid)
        spec = hex2spec(mesh) if mesh.nelmt < 5000 else __import__(
            "specfem3d_geotech_amd.spec", fromlist=["x"]).hex2spec_device(ctx, mesh)
        ref = None
        for ncol in (1, 2, 4, 8, 16, 32, 64):
            x = _engine_x(ctx, mesh, spec, ncol, steps, cols=min(ncol, 3))
            assert np.abs(x).max() > 0
            ref = x if ref is None else ref
            assert np.array_equal(x, ref), ncol


@pytest.mark.parametrize("grid", [(1, 1, 1), (3, 1, 1), (3, 3, 1), (8, 4, 6)])
def test_batched_solve_from_geometry_and_from_uploaded_matrices(ctx, grid):
    """The engine's converged solve is the same on a built mesh and on one
    whose (identical) matrices were uploaded: both end at relative updates
    of 1e-12 from FP64 residuals, so they agree to 1e-10."""
    mesh = _mesh(*grid)
    spec = hex2spec(mesh)
    a = _engine_x(ctx, mesh, spec, 4, 0)
    b = _engine_x(ctx, mesh, spec, 4, 0, upload=True)
    assert rel_l2(a, b) < 1e-10


# equation counts around the tiles' lengths: fewer than one tile, a tile's
# edge, several tiles per wave (1, 2, 4 columns) with a ragged end, and above
# 131,072 equations, where the tiles grow
@pytest.mark.parametrize("grid", [(1, 1, 1), (2, 2, 2), (5, 3, 2), (9, 7, 11), (21, 16, 18)])
def test_engine_steps_same_bits_around_tile_edges(ctx, grid):
    """x after 24 steps (three x writes, FP64 residuals between) has the same
    bits in engines of 1 to 64 columns, and follows the FP64 iterate of the
    drop-in: FP32 directions and residuals keep it within 1e-3 of it over
    so few iterations."""
    mesh = _mesh(*grid)
    spec = hex2spec(mesh)
    xs = [_engine_x(ctx, mesh, spec, ncol, 24, cols=min(ncol, 2)) for ncol in (1, 2, 4, 8, 16, 32, 64)]
    for x in xs[1:]:
        assert np.array_equal(x, xs[0])
    gam, ym, nu, *_ = mesh.material_arrays()
    dm = DeviceMesh(ctx, spec, len(gam))
    try:
        ext, _ = dm.build_stiffness(gam, ym, nu)
        if spec.neq > 100:
            u, _, _ = dm.solve(ext, cg_tol=1e-14, cg_maxiter=24)
            assert rel_l2(xs[0], u) < 1e-3
    finally:
        dm.close()


def test_inverse_map_rows_beside_the_device_sort(ctx):
    """K p where an equation gathers 63, 64, 65 or thousands of element
    entries (rows of up to 64 are sorted on the device, longer ones on the
    host), and a refused equation number: the sums run over the entries in
    ascending element order, so they equal the oracle's bit for bit."""
    import oracle as O
    rng = np.random.default_rng(9)
    for nelmt, neq, shared in ((7, 40, 63), (7, 40, 64), (7, 40, 65), (120, 9, 4000)):
        flat = rng.integers(0, neq, nelmt * 81).astype(np.int32)  # neq itself: shared below
        flat[rng.permutation(flat.size)[:shared]] = neq
        gdof = flat.reshape(nelmt, 81)
        spec = hex2spec(_mesh(nelmt, 1, 1))
        spec.gdof_elmt, spec.neq = gdof, neq
        k = rng.normal(size=(nelmt, 81, 81))
        p = rng.normal(size=neq + 1)
        p[0] = 0.0
        dm = DeviceMesh(ctx, spec, 2)
        try:
            dm.upload_stiffness(k, np.ones(neq + 1))
            assert np.array_equal(dm.matvec(p)[1:], O.ebe_matvec(neq, k, gdof, p)[1:])
        finally:
            dm.close()
        gdof[nelmt - 1, 80] = neq + 1
        with pytest.raises(RuntimeError, match=rf"gdof_elmt\[{nelmt * 81 - 1}\]={neq + 1}"):
            DeviceMesh(ctx, spec, 2)


@pytest.mark.parametrize("grid", [(1, 1, 1), (3, 2, 1), (9, 4, 3)])
def test_stiffness_of_distorted_elements_bits(ctx, grid):
    """K, its diagonal and the gravity load of strongly distorted elements
    are the oracle's bits; where a corner is not finite every entry of that
    element is NaN, as the full sums give it."""
    import oracle as O
    mesh = slope_mesh(*grid, materials=SOILS, layer_z=[10.0], jitter=0.25, seed=11)
    spec = hex2spec(mesh)
    gam, ym, nu, *_ = mesh.material_arrays()
    km, _, ext0 = O.stiffness_bodyload(spec, gam, nu, ym)
    dm = DeviceMesh(ctx, spec, len(gam))
    try:
        ext, _ = dm.build_stiffness(gam, ym, nu)
        assert np.array_equal(dm.download_stiffness(), km)
        assert np.array_equal(ext, ext0)
    finally:
        dm.close()
    spec.corners = spec.corners.copy()
    spec.corners[-1, 3, 1] = np.nan
    dm = DeviceMesh(ctx, spec, len(gam))
    try:
        dm.build_stiffness(gam, ym, nu)
        k = dm.download_stiffness()
        assert np.isnan(k[-1]).all() and np.array_equal(k[:-1], km[:-1])
    finally:
        dm.close()


def test_matrices_buffer_of_a_closed_mesh_serves_the_next(ctx):
    """Meshes made one after another on one context, each closed before the
    next: equal, a little smaller (the kept buffer serves it), much smaller
    and larger (it does not).  Each has the oracle's matrices, and two alive
    at once do not share a buffer."""
    import oracle as O
    alive = []
    for nelmt in (60, 60, 50, 20, 80, 60):
        spec = hex2spec(_mesh(nelmt, 1, 1))
        gam, ym, nu, *_ = _mesh(nelmt, 1, 1).material_arrays()
        km, _, _ = O.stiffness_bodyload(spec, gam, nu, ym)
        dm = DeviceMesh(ctx, spec, len(gam))
        dm.build_stiffness(gam, ym, nu)
        assert np.array_equal(dm.download_stiffness(), km)
        alive.append((dm, km))
        if len(alive) == 2:  # the one before is still what it was
            old, old_km = alive.pop(0)
            assert np.array_equal(old.download_stiffness(), old_km)
            old.close()
    alive[0][0].close()


@pytest.mark.parametrize("built", [True, False])
@pytest.mark.parametrize("ncol", [1, 64])
def test_autotune_after_the_stiffness_changed_hands(ctx, built, ncol):
    """Mid-solve the mesh gets the same matrices uploaded (or built again
    from the geometry) and the engine tunes the product that it now has; the
    solve goes on to the solution of an engine that was left alone (both end
    at relative updates of 1e-12 from FP64 residuals: 1e-10)."""
    from specfem3d_geotech_amd.batch import DEFAULT_INNER_TOL, BatchEngine, device_mesh
    from specfem3d_geotech_amd.plastic import dt_viscoplas
    mesh = _mesh(8, 4, 6)
    spec = hex2spec(mesh)
    gam, ym, nu, phi, coh, psi = mesh.material_arrays()
    ref = _engine_x(ctx, mesh, spec, ncol, 0)
    dm, ext = device_mesh(ctx, mesh, spec)
    try:
        _, dinv = dm.build_stiffness(gam, ym, nu)
        k = dm.download_stiffness()
        if not built:
            dm.upload_stiffness(k, dinv)
        eng = BatchEngine(dm, ext, ncol)
        try:
            eng.begin(0, ym, nu, phi, coh, psi, dt_viscoplas(nu, phi, ym))
            eng.advance(1e-12, 20000, DEFAULT_INNER_TOL, 5e-4, 1, max_steps=40)
            if built:
                dm.upload_stiffness(k, dinv)
            else:
                dm.build_stiffness(gam, ym, nu)
            t = eng.autotune(2)
            assert t["ms"] > 0
            while not eng.advance(1e-12, 20000, DEFAULT_INNER_TOL, 5e-4, 1)["ended"][0]:
                pass
            assert rel_l2(eng.download(0)[0], ref) < 1e-10
        finally:
            eng.close()
    finally:
        dm.close()


@pytest.mark.parametrize("ncol,grid", [(1, (4, 3, 2)), (64, (12, 5, 5))])
@pytest.mark.parametrize("exp", [-40, 48])
def test_engine_in_other_units_of_length(ctx, ncol, grid, exp):
    """The same slope in a unit of length 2^exp times as large (unit weights
    smaller by it, moduli kept): every number of the solve is a power of two
    times that of the plain one, so x is, bit for bit.  E / h^3 and h^2 leave
    the range of FP32 here, E h does not."""
    mesh = _mesh(*grid)
    x = _engine_x(ctx, mesh, hex2spec(mesh), ncol, 24)
    assert np.abs(x).max() > 0 and np.isfinite(x).all()
    s = 2.0 ** exp
    mesh.coord = mesh.coord * s
    mesh.materials = [Material(gam=m.gam / s, ym=m.ym, nu=m.nu, phi=m.phi, coh=m.coh)
                      for m in SOILS]
    assert np.array_equal(_engine_x(ctx, mesh, hex2spec(mesh), ncol, 24), x * s)
