"""The kernels that take a matrix's rows by blocks of 256 (residual A x - b, rAU with HbyA,
the solver's explicit residual) against the same sums in Python floats, in column order, bit
for bit: blocks that fit the LDS, one that does not (a coarse cell with 400 neighbours), a
last block of one row."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    import foamadapter_amd as fa
    with fa.Context(0) as c:
        yield c


def _poly(name):
    import foamadapter_amd as fa
    from skewed_meshes import refined_block
    if name == "refined":
        r = refined_block(20)
        return r[0] if isinstance(r, tuple) else r
    return fa.PolyMesh.hex({"one": (1, 1, 1), "line": (257, 1, 1), "box": (11, 9, 8)}[name])


@pytest.mark.parametrize("name", ["one", "line", "box", "refined"])
def test_rows_by_blocks(ctx, name):
    import foamadapter_amd as fa
    from foamadapter_amd import coupling, dsl, fvcc, la
    print(name, flush=True)
    m = fa.Mesh.from_poly(ctx, _poly(name))
    N, F, B = m.n_cells, m.n_internal_faces, m.n_boundary_faces
    bc = fa.BoundaryConditions(m, ["fixedValue"] * m.n_patches)
    T = fvcc.VolumeField(m, ctx.uniform(N, -1, 1, 3, 0), ctx.uniform(B, -1, 1, 3, 1), bc, "T")
    phi = fvcc.SurfaceField(m, ctx.uniform(F + B, -1, 1, 3, 2))
    gamma = fvcc.SurfaceField(m, ctx.uniform(F + B, 0.5, 2, 3, 3))
    ls = dsl.assemble(dsl.imp.ddt(T) + dsl.imp.div(phi, T) - dsl.imp.laplacian(gamma, T), T, 0.0, 0.01)
    ro, ci, va, b = ls.sp.rowOffs(), ls.sp.colIdxs(), ls.values(), ls.rhs()
    if name == "refined":
        assert ro[256] - ro[0] > 2048
    x = T.numpy()
    res = np.empty(N)
    for i in range(N):
        s = 0.0
        for k in range(ro[i], ro[i + 1]):
            s += va[k] * x[ci[k]]
        res[i] = s - b[i]
    assert np.array_equal(ls.residual(T.internal).numpy(), res)
    # the solver's own, ||b - A x|| / ||b|| of a solve that may not iterate (the
    # kernel-by-kernel form reads no state then and reports the final residual only)
    st = la.solve_cg(ls, T.internal, {"relTol": 1e-30, "maxIter": 0}, raise_on_noconverge=False)
    ref = np.linalg.norm(res) / np.linalg.norm(b)
    assert abs((st.initResNorm or st.trueResNorm) - ref) <= 4 * N * 2.3e-16 * ref  # two sums of N squares

    u3, b3 = ctx.uniform(3 * N, -1, 1, 3, 4), ctx.uniform(3 * N, -1, 1, 3, 5)
    u3.shape = b3.shape = (N, 3)
    U = fvcc.VolumeField(m, u3, ctx.zeros((B, 3)), bc, "U")
    V, d = m.get("V"), ls.sp.diagOffset()
    rau = V / va[ro[:-1] + d]
    uh, bh = u3.numpy(), b3.numpy()
    h = np.empty((N, 3))
    for i in range(N):
        s = np.zeros(3)
        for k in range(ro[i], ro[i + 1]):
            if k != ro[i] + d[i]:
                s -= va[k] * uh[ci[k]]
        h[i] = (s + bh[i]) * (rau[i] / V[i])
    rAU, HbyA = coupling.computeRAUandHByA(ls, b3, U)
    fc = m.get("faceCells")
    assert np.array_equal(rAU.internal.numpy(), rau) and np.array_equal(rAU.boundary.numpy(), rau[fc])
    assert np.array_equal(HbyA.internal.numpy(), h) and np.array_equal(HbyA.boundary.numpy(), h[fc])
    one = coupling.computeRAU(ls)  # the separate form
    assert np.array_equal(one.internal.numpy(), rau)
    m.close()


@pytest.mark.parametrize("gather", [0, 1])  # staged: in one pass; stencil walk: in two
def test_velocity_update(ctx, gather):
    import foamadapter_amd as fa
    from foamadapter_amd import coupling, fvcc
    print(gather, flush=True)
    m = fa.Mesh.from_poly(ctx, fa.PolyMesh.hex((19, 17, 13), jitter=0.2, jitter_seed=2, perm_seed=1), renumber=True)
    m.set_gather(gather)
    N, B = m.n_cells, m.n_boundary_faces
    p = fvcc.VolumeField(m, ctx.uniform(N, -1, 1, 4, 0), ctx.uniform(B, -1, 1, 4, 1))
    h3 = ctx.uniform(3 * N, -1, 1, 4, 2)
    h3.shape = (N, 3)
    rau = ctx.uniform(N, 0.5, 2, 4, 3)
    U = fvcc.VolumeField(m, ctx.zeros((N, 3)), ctx.zeros((B, 3)))
    coupling.updateVelocity(fvcc.VolumeField(m, h3, None), fvcc.VolumeField(m, rau, None), p, U)
    g = fvcc.GaussGreenGrad(ctx, m).grad(p).numpy()
    assert np.array_equal(U.numpy(), h3.numpy() - rau.numpy()[:, None] * g)
    m.close()


@pytest.mark.parametrize("precision", ["double", "mixed"])
@pytest.mark.parametrize("name", ["one", "line", "box", "refined"])
def test_batch_start(ctx, name, precision):
    """The start of a batched solve (row residual, scaling, first residual) and the fused
    heat assembly: two CG iterations from a nonzero x against the same two in FP64 numpy.
    A row sum of n terms is off by n * eps of its terms; the scaled system is diagonally
    dominant, so two iterations keep errors at a few times that: bounds 64 and, where
    vectors are FP32, 64 * 2^-24 of the first correction."""
    import scipy.sparse as sp
    import foamadapter_amd as fa
    from foamadapter_amd import fvcc, la
    print(name, precision, flush=True)
    m = fa.Mesh.from_poly(ctx, _poly(name))
    N, F, B = m.n_cells, m.n_internal_faces, m.n_boundary_faces
    bc = fa.BoundaryConditions(m, ["fixedValue"] * m.n_patches)
    T = fvcc.VolumeField(m, ctx.uniform(N, -1, 1, 3, 0), ctx.uniform(B, -1, 1, 3, 1), bc, "T")
    gam = ctx.upload(np.full(F + B, 1e-2 * float(m.get("V").mean()) ** (2 / 3)))
    ls = la.LinearSystem(la.SparsityPattern(m))
    la.HeatAssembly([(ls, T.internal, 1.0, gam, bc, T.boundary, None)]).assemble(-1.0)
    A, b = ls.scipy(), ls.rhs()
    if name == "refined":
        assert A.indptr[256] - A.indptr[0] > 2048
    x0 = ctx.uniform(N, -1, 1, 3, 7)
    xh = x0.numpy()
    bt = la.Batch(ctx, precision, 2048, 2)  # tiles of two kScaleRows, one chunk
    bt.add(ls, x0)
    st = bt.solve({"relTol": 1e-30, "maxIter": 2, "innerRelTol": 1e-30}, use_graph=False,
                  raise_on_noconverge=False)[0]
    g = np.sqrt(A.diagonal())
    G = sp.diags(1 / g)
    As = G @ A @ G
    r = (b - A @ xh) / g
    ref0 = np.linalg.norm(r * g) / np.linalg.norm(b)
    d, p = np.zeros(N), r.copy()
    rho = r @ r
    for _ in range(st.numIter):
        if rho == 0.0:  # one row: solved by the first iteration
            break
        q = As @ p
        a = rho / (p @ q)
        d, r = d + a * p, r - a * q
        rho, old = r @ r, rho
        p = r + rho / old * p
    eps = 2.0 ** -52 if precision == "double" else 2.0 ** -24
    assert 1 <= st.numIter <= 2
    assert abs(st.initResNorm - ref0) <= 64 * N * 2.0 ** -52 * ref0
    ref = xh + d / g
    scale = np.abs(xh).max() + np.abs(d / g).max()
    assert np.abs(x0.numpy() - ref).max() <= 64 * (eps * np.abs(d / g).max() + 2.0 ** -52 * scale)
    bt.close()
    m.close()
