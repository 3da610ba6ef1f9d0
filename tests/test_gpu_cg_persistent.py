"""The persistent CG and BiCGStab kernels against the kernel-by-kernel form ("graph": False), bit for
bit: both add every dot product in the same order, so the solutions, the iteration counts
and the residuals are the same numbers.  The sizes sit at the edges of what the kernel
distinguishes: tiles of 256 rows (the last one ragged), 64 workgroups of up to 256 tiles or
256 workgroups beyond, 1, 2, 4 and 8 rows per thread, slices of 4 (plane meshes) and 6
entries, and solves of several launches (for BiCGStab, solves that go on where a launch ended)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [
    # dims, iteration limit
    ((3, 3, 3), 200),          # one ragged tile
    ((16, 16, 1), 200),        # one whole tile, 4 entries a row
    ((17, 16, 16), 400),       # 17 tiles: a second tile in one workgroup
    ((65, 16, 16), 2000),      # 65 tiles: the second wave of slots begins
    ((256, 16, 16), 700),      # 256 tiles: the last grid of 64 workgroups
    ((257, 16, 16), 700),      # 257: 256 workgroups, all but one with one tile
    ((64, 32, 32), 2000),      # the same two, converging
    ((41, 40, 40), 2000),
    ((64, 64, 65), 60),        # 2 rows per thread
    ((700, 500, 1), 60),       # the same, 4 entries a row
    ((101, 100, 61), 40),      # 3 rows per thread (kernel of 4), last slice ragged
    ((128, 128, 70), 30),      # 5 rows per thread (kernel of 8)
]


@pytest.fixture(scope="module")
def ctx():
    import foamadapter_amd as fa
    with fa.Context(0) as c:
        yield c


def _system(ctx, dims):
    import foamadapter_amd as fa
    from foamadapter_amd import dsl, fvcc
    poly = fa.PolyMesh.hex(dims, jitter=0.2 if min(dims) > 1 else 0.0, jitter_seed=5)
    if min(dims) == 1:  # a plane mesh: no finite-volume faces on its two sides
        for p in poly.patches[4:]:
            p.type = "empty"
    m = fa.Mesh.from_poly(ctx, poly, renumber=len(dims) == 3 and min(dims) > 40)
    N, F, B = m.n_cells, m.n_internal_faces, m.n_boundary_faces
    bc = fa.BoundaryConditions(m, ["fixedValue"] + ["zeroGradient"] * (m.n_patches - 1))
    p = fvcc.VolumeField(m, ctx.zeros((N,)), ctx.zeros((B,)), bc, "p")
    gamma = fvcc.SurfaceField(m, ctx.uniform(F + B, 0.5, 2.0, 11, 0))
    phi = fvcc.SurfaceField(m, ctx.uniform(F + B, -1.0, 1.0, 11, 1))
    return m, dsl.assemble(dsl.imp.laplacian(gamma, p) - dsl.exp.div(phi), p, 0.0, 1.0)


@pytest.mark.parametrize("precision", ["double", "mixed"])
@pytest.mark.parametrize("dims,limit", CASES, ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_persistent_is_bitwise_the_kernel_by_kernel_form(ctx, dims, limit, precision):
    from foamadapter_amd import la
    print(dims, limit, precision, flush=True)
    m, ls = _system(ctx, dims)
    got = []
    # eager first, then the persistent form three times: a first solve, and repeats of it
    for graph in (False, True, True, True):
        x = ctx.zeros((m.n_cells,))
        st = la.solve_cg(ls, x, {"relTol": 1e-8, "maxIter": limit, "precision": precision, "graph": graph},
                         raise_on_noconverge=False)
        got.append((x.numpy(), st.numIter, st.finalResNorm, st.status))
    assert got[0][1] >= 12  # fewer iterations in the solve before run kernel by kernel
    for g in got[1:]:
        if precision == "mixed" and got[0][3] != 0 and got[0][1] < limit:
            # cut by its limit after a residual replacement: the kernel-by-kernel form
            # counts the iterations it had queued behind the replacement's stop towards
            # the limit, the persistent one runs as many as it was given
            assert g[1] == limit and g[3] == got[0][3]
            continue
        assert g[1:] == got[0][1:]
        assert np.array_equal(g[0], got[0][0])
    m.close()


GHOST_CASES = [
    ((64, 64, 63), "random"),     # one row per thread: up to 1536 ghosts for 256 rows
    ((64, 64, 65), "random"),     # 2 rows per thread: a tile of 512 rows has up to 3072 ghosts
    ((101, 100, 61), "random"),   # 3 rows: more ghosts than fit in FP64, not in FP32
    ((128, 128, 70), "block"),    # 5 rows: the same
    ((128, 128, 70), "random"),   # more than fit in either
]


@pytest.mark.parametrize("method", ["double", "mixed", "bicgstab"])
@pytest.mark.parametrize("dims,order", GHOST_CASES, ids=str)
def test_many_ghosts(ctx, dims, order, method):
    """Tiles whose rows refer to many rows of other tiles: in LDS while they fit, else read
    where the product meets them.  Fewer iterations than one replacement takes."""
    import foamadapter_amd as fa
    from foamadapter_amd import dsl, fvcc, la
    print(dims, order, method, flush=True)
    m = fa.Mesh.from_poly(ctx, fa.PolyMesh.hex(dims, **({"perm_seed": 3} if order == "random" else {})))
    N, F, B = m.n_cells, m.n_internal_faces, m.n_boundary_faces
    p = fvcc.VolumeField(m, ctx.zeros((N,)), ctx.zeros((B,)),
                         fa.BoundaryConditions(m, ["fixedValue"] * m.n_patches), "p")
    gamma = fvcc.SurfaceField(m, ctx.uniform(F + B, 0.5, 2.0, 11, 0))
    phi = fvcc.SurfaceField(m, ctx.uniform(F + B, -1.0, 1.0, 11, 1))
    ls = dsl.assemble(dsl.imp.laplacian(gamma, p) - dsl.exp.div(phi), p, 0.0, 1.0)
    got = []
    for graph in (False, True, True):
        x = ctx.uniform(N, -1, 1, 12, 4)
        opts = {"solver": "PBiCGStab"} if method == "bicgstab" else {"precision": method}
        st = la.solve_cg(ls, x, dict(opts, relTol=1e-12, maxIter=20, graph=graph), raise_on_noconverge=False)
        got.append((x.numpy(), st.numIter, st.finalResNorm))
    for g in got[1:]:
        assert g[1:] == got[0][1:] and np.array_equal(g[0], got[0][0])
    m.close()


BI_CASES = [
    ((3, 3, 3), 100), ((16, 16, 1), 200), ((17, 16, 16), 100), ((65, 16, 16), 400), ((64, 32, 32), 400),
    ((41, 40, 40), 400),
    ((64, 64, 65), 130),       # 2 rows per thread, two launches
    ((700, 500, 1), 130),      # the same, 4 entries a row
    ((101, 100, 61), 130),     # 3 rows per thread (kernel of 4), last slice ragged
]


@pytest.mark.parametrize("kind", ["advection", "diffusion"])
@pytest.mark.parametrize("dims,limit", BI_CASES, ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_persistent_bicgstab_is_bitwise_the_kernel_by_kernel_form(ctx, dims, limit, kind):
    from foamadapter_amd import dsl, fvcc, la
    print(dims, limit, kind, flush=True)
    m, ls = _system(ctx, dims)
    N, F, B = m.n_cells, m.n_internal_faces, m.n_boundary_faces
    if kind == "advection":  # non-symmetric, a few iterations
        import foamadapter_amd as fa
        T = fvcc.VolumeField(m, ctx.uniform(N, -1, 1, 12, 0), ctx.uniform(B, -1, 1, 12, 1),
                             fa.BoundaryConditions(m, ["fixedValue"] * m.n_patches), "T")
        phi = fvcc.SurfaceField(m, ctx.uniform(F + B, -1e-6, 1e-6, 12, 2))
        gamma = fvcc.SurfaceField(m, ctx.uniform(F + B, 0.5, 2.0, 12, 3))
        dt = 0.5 * float(m.get("V").mean()) ** (2.0 / 3.0)
        dsl.assemble(dsl.imp.ddt(T) + dsl.imp.div(phi, T, "upwind") - dsl.imp.laplacian(gamma, T), T, 0.0, dt, ls)
    got = []
    for graph in (False, True, True):
        x = ctx.uniform(N, -1, 1, 12, 4)
        st = la.solve_cg(ls, x, {"solver": "PBiCGStab", "relTol": 1e-9, "maxIter": limit, "graph": graph},
                         raise_on_noconverge=False)
        got.append((x.numpy(), st.numIter, st.initResNorm, st.finalResNorm, st.trueResNorm, st.status))
    for g in got[1:]:
        assert g[1:] == got[0][1:]
        assert np.array_equal(g[0], got[0][0])
    m.close()


VEC_CASES = [((3, 3, 3), 100), ((17, 16, 16), 100), ((16, 16, 1), 200),
             ((41, 40, 40), 400),     # components of several launches
             ((64, 64, 65), 130),     # 2 rows per thread; the limit ends the first component
             ((17, 16, 16), 1)]       # no component converges


@pytest.mark.parametrize("kind", ["advection", "diffusion"])
@pytest.mark.parametrize("dims,limit", VEC_CASES, ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_vec_components_are_bitwise_the_single_solves(ctx, dims, limit, kind):
    """The components of a Vec3 equation solved from interleaved arrays against the kernel-by-kernel
    solves of component copies: solutions, stats, the system's right-hand side, and what an error leaves."""
    import foamadapter_amd as fa
    from foamadapter_amd import _lib, dsl, fvcc
    print(dims, limit, kind, flush=True)
    m, ls = _system(ctx, dims)
    N, F, B = m.n_cells, m.n_internal_faces, m.n_boundary_faces
    if kind == "advection":
        T = fvcc.VolumeField(m, ctx.uniform(N, -1, 1, 12, 0), ctx.uniform(B, -1, 1, 12, 1),
                             fa.BoundaryConditions(m, ["fixedValue"] * m.n_patches), "T")
        phi = fvcc.SurfaceField(m, ctx.uniform(F + B, -1e-6, 1e-6, 12, 2))
        gamma = fvcc.SurfaceField(m, ctx.uniform(F + B, 0.5, 2.0, 12, 3))
        dt = 0.5 * float(m.get("V").mean()) ** (2.0 / 3.0)
        dsl.assemble(dsl.imp.ddt(T) + dsl.imp.div(phi, T, "upwind") - dsl.imp.laplacian(gamma, T), T, 0.0, dt, ls)
    b3 = ctx.uniform(3 * N, -1, 1, 13, 1)
    b3.shape = (N, 3)
    got = []
    for graph in (False, True, True):
        x3 = ctx.uniform(3 * N, -1, 1, 13, 2)
        x3.shape = (N, 3)
        ls.rhs3 = b3
        st = err = None
        try:
            st = dsl._solve_vec(ls, fvcc.VolumeField(m, x3, None), {"solver": "PBiCGStab", "relTol": 1e-9,
                                                                    "maxIter": limit, "graph": graph})
        except _lib.FvError as e:
            err = str(e)
        got.append((x3.numpy(), ls.rhs(), st, err))
    assert (got[0][3] is not None) == (limit == 1 or got[0][2] is None)
    for g in got[1:]:
        assert g[2:] == got[0][2:]
        assert np.array_equal(g[0], got[0][0]) and np.array_equal(g[1], got[0][1])
    m.close()


@pytest.mark.parametrize("dims", [(1, 1, 1), (17, 16, 1), (61, 60, 59)], ids=str)
def test_vec_boundary_and_mean_magnitude(ctx, dims):
    import ctypes as C
    import foamadapter_amd as fa
    from foamadapter_amd import _lib, fvcc
    print(dims, flush=True)
    m = fa.Mesh.from_poly(ctx, fa.PolyMesh.hex(dims, jitter=0.2, jitter_seed=2))
    N, B = m.n_cells, m.n_boundary_faces
    kinds = (["fixedGradient", "fixedValue", "zeroGradient"] * m.n_patches)[:m.n_patches]
    bc = fa.BoundaryConditions(m, kinds)
    u, ub, ug = (ctx.uniform(3 * n, -1, 1, 14, i) for i, n in enumerate((N, B, B)))
    u.shape, ub.shape, ug.shape = (N, 3), (B, 3), (B, 3)
    ref, po, fc, dc = ub.numpy().copy(), m.get("patchOffsets"), m.get("faceCells"), m.get("deltaCoeffs_b")
    for i, k in enumerate(kinds):
        if k != "fixedValue":
            r = slice(po[i], po[i + 1])
            ref[r] = u.numpy()[fc[r]] + ug.numpy()[r] / dc[r, None]
    fvcc.VolumeField(m, u, ub, bc, "U", ug).correct_boundary_conditions()
    assert np.array_equal(ub.numpy(), ref)
    d = ctx.uniform(N, -1, 1, 14, 5)
    mean = C.c_double()
    _lib.call("fv_mean_magnitude", ctx.handle, m.handle, d.ptr, C.byref(mean))
    V = m.get("V")
    want = np.sum(V * np.abs(d.numpy())) / np.sum(V)
    assert abs(mean.value - want) <= 4 * N * 2.3e-16 * want  # two pairs of sums of N terms
    m.close()


def test_solves_of_several_threads(ctx):
    """Small solves are plain launches whose workgroups meet; beside the solves of other threads,
    one of which fills the device, they may not, and are launched again: the same bits."""
    import threading
    import foamadapter_amd as fa
    from foamadapter_amd import la
    cases = [((128, 128, 70), "PCG", 2, 40), ((41, 40, 40), "PCG", 12, 2000), ((33, 32, 32), "PCG", 12, 2000),
             ((64, 32, 32), "PBiCGStab", 12, 400)]
    out, errors = {}, []

    def run(i):
        try:
            dims, method, reps, limit = cases[i]
            with fa.Context(0) as c:
                m, ls = _system(c, dims)
                opts = {"solver": method, "relTol": 1e-8, "maxIter": limit}
                got = []
                for graph in [False] + [True] * reps:
                    x = c.zeros((m.n_cells,))
                    st = la.solve_cg(ls, x, dict(opts, graph=graph), raise_on_noconverge=False)
                    got.append((x.numpy(), st.numIter, st.finalResNorm))
                    x.close()
                out[i] = got
                m.close()
        except Exception as e:  # noqa: BLE001
            errors.append((i, e))

    threads = [threading.Thread(target=run, args=(i,)) for i in range(len(cases))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
    for i, got in out.items():
        for g in got[1:]:
            assert g[1:] == got[0][1:] and np.array_equal(g[0], got[0][0]), cases[i]


@pytest.mark.parametrize("method", ["double", "mixed", "bicgstab"])
def test_a_solve_without_iterations(ctx, method):
    """maxIter 0, first and repeated, before and after a solve: the forms agree, x stays, and a
    residual above the tolerance is not reported as convergence (FP64 CG, which reads no state
    when it runs nothing, reports the residual of x as its explicit one)."""
    from foamadapter_amd import la
    print(method, flush=True)
    opts = {"solver": "PBiCGStab"} if method == "bicgstab" else {"precision": method}
    got = []
    for graph in (False, True):
        m, ls = _system(ctx, (17, 16, 16))
        A, b = ls.scipy(), ls.rhs()
        x = ctx.uniform(m.n_cells, -1, 1, 12, 4)
        x0 = x.numpy()
        res = np.linalg.norm(b - A @ x0) / np.linalg.norm(b)
        out = []
        for limit in (0, 0, 30, 0):
            if limit:
                la.solve_cg(ls, ctx.uniform(m.n_cells, -1, 1, 12, 5), dict(opts, relTol=1e-12, maxIter=limit, graph=graph),
                            raise_on_noconverge=False)
                continue
            st = la.solve_cg(ls, x, dict(opts, relTol=1e-8, maxIter=0, graph=graph), raise_on_noconverge=False)
            assert np.array_equal(x.numpy(), x0) and abs(st.trueResNorm - res) <= m.n_cells * 2.3e-16 * res
            if method != "double":
                assert st.status != 0 and st.finalResNorm == st.trueResNorm
            out.append((st.numIter, st.initResNorm, st.finalResNorm, st.trueResNorm, st.status))
        got.append(out)
        m.close()
    assert got[0] == got[1]


def test_a_solve_without_iterations_leaves_x(ctx):
    """A diagonal of both signs, which the scaling cannot take: x is not touched and its residual
    reported all the same."""
    import foamadapter_amd as fa
    from foamadapter_amd import dsl, fvcc, la
    m = fa.Mesh.from_poly(ctx, fa.PolyMesh.hex((11, 9, 8)))
    N, F, B = m.n_cells, m.n_internal_faces, m.n_boundary_faces
    T = fvcc.VolumeField(m, ctx.uniform(N, -1, 1, 3, 0), ctx.uniform(B, -1, 1, 3, 1),
                         fa.BoundaryConditions(m, ["fixedValue"] * m.n_patches), "T")
    phi = fvcc.SurfaceField(m, ctx.uniform(F + B, -1, 1, 3, 2))
    ls = dsl.assemble(dsl.imp.ddt(T) + dsl.imp.div(phi, T), T, 0.0, 1.0)
    A, b = ls.scipy(), ls.rhs()
    assert A.diagonal().min() < 0 < A.diagonal().max()
    for graph in (False, True):
        x = ctx.uniform(N, -1, 1, 12, 4)
        x0 = x.numpy()
        st = la.solve_cg(ls, x, {"relTol": 1e-8, "maxIter": 0, "graph": graph}, raise_on_noconverge=False)
        res = np.linalg.norm(b - A @ x0) / np.linalg.norm(b)
        assert np.array_equal(x.numpy(), x0) and abs(st.trueResNorm - res) <= N * 2.3e-16 * res
    m.close()
