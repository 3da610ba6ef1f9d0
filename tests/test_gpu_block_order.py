"""The cell operators on meshes in a block mesher's order (lines of cells, not
renumbered), whose 256-cell workgroups have more lower and boundary faces than the default
lists hold and run in the wide form: bit for bit the per-cell stencil walk, which is the
oracle's order.  The sizes sit at the edges of the wide lists: lines shorter and longer
than a workgroup, planes of less than one, and a mesh whose sides have all faces on the
boundary."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DIMS = [(257, 20, 9), (300, 7, 12), (40, 33, 21), (16, 15, 40), (97, 83, 6)]


@pytest.fixture(scope="module")
def ctx():
    import foamadapter_amd as fa
    with fa.Context(0) as c:
        yield c


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("dims", DIMS)
def test_wide_workgroups_bitwise_the_stencil_walk(ctx, dims, dtype):
    import foamadapter_amd as fa
    from foamadapter_amd import fvcc
    print(dims, dtype, flush=True)
    m = fa.Mesh.from_poly(ctx, fa.PolyMesh.hex(dims, jitter=0.2, jitter_seed=3))
    N, F, B = m.n_cells, m.n_internal_faces, m.n_boundary_faces
    kinds = ["fixedValue", "fixedGradient"] * 3
    T = fvcc.VolumeField(m, ctx.uniform(N, -1, 1, 1, 0, dtype), ctx.uniform(B, -1, 1, 1, 1, dtype),
                         fa.BoundaryConditions(m, kinds), "T", ctx.uniform(B, -1, 1, 1, 2, dtype))
    phi = fvcc.SurfaceField(m, ctx.uniform(F + B, -1, 1, 1, 3, dtype))
    gamma = fvcc.SurfaceField(m, ctx.uniform(F + B, 0.5, 2, 1, 4, dtype))

    def ops():
        return [fvcc.GaussGreenGrad(ctx, m).grad(T, 1.5).numpy(),
                fvcc.GaussGreenDiv(ctx, m, ["linear"]).div(None, phi, T, 0.5).numpy(),
                fvcc.GaussGreenDiv(ctx, m, ["upwind"]).div(None, phi, T).numpy(),
                fvcc.GaussGreenDiv(ctx, m).div(None, phi).numpy(),
                fvcc.GaussGreenLaplacian(ctx, m).laplacian(None, gamma, T, 2.0).numpy()]

    m.set_gather(1)
    walk = ops()
    m.set_gather(0)
    for name, a, b in zip(("grad", "div", "upwind", "integrate", "laplacian"), ops(), walk):
        assert np.array_equal(a, b), name
    m.close()


def test_block_order_takes_the_staged_path(ctx):
    """Lines of 97 cells: all but a few corner workgroups fit the wide lists."""
    import foamadapter_amd as fa
    m = fa.Mesh.from_poly(ctx, fa.PolyMesh.hex((97, 83, 61)))
    blocks, over = m.gather_stats(256)
    assert over * 100 <= blocks
    m.close()


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("dims", DIMS + [(1, 1, 1), "refined", (64, 32, 32), (61, 33, 33), (64, 64, 64), (65, 65, 63)], ids=str)
def test_walk_and_staged_at_the_edges_of_the_rule(ctx, dims, dtype):
    """Small meshes walk the stencil by themselves (65536 cells, 262144 in a block mesher's
    order), six entries at a time (the refined mesh has a cell with 400): every mode against the
    sums over the faces in Python's order (small meshes) and against each other."""
    import foamadapter_amd as fa
    from foamadapter_amd import fvcc
    import oracle_cpu as orc
    from skewed_meshes import refined_block
    print(dims, dtype, flush=True)
    poly = refined_block(20) if dims == "refined" else fa.PolyMesh.hex(dims, jitter=0.0 if dims == (1, 1, 1) else 0.2, jitter_seed=3)
    poly = poly[0] if isinstance(poly, tuple) else poly
    m = fa.Mesh.from_poly(ctx, poly)
    N, F, B = m.n_cells, m.n_internal_faces, m.n_boundary_faces
    kinds = (["fixedValue", "fixedGradient"] * m.n_patches)[:m.n_patches]
    T = fvcc.VolumeField(m, ctx.uniform(N, -1, 1, 1, 0, dtype), ctx.uniform(B, -1, 1, 1, 1, dtype),
                         fa.BoundaryConditions(m, kinds), "T", ctx.uniform(B, -1, 1, 1, 2, dtype))
    phi = fvcc.SurfaceField(m, ctx.uniform(F + B, -1, 1, 1, 3, dtype))
    gamma = fvcc.SurfaceField(m, ctx.uniform(F + B, 0.5, 2, 1, 4, dtype))

    def ops():
        return [fvcc.GaussGreenGrad(ctx, m).grad(T, 1.5).numpy(),
                fvcc.GaussGreenDiv(ctx, m, ["linear"]).div(None, phi, T, 0.5).numpy(),
                fvcc.GaussGreenDiv(ctx, m, ["upwind"]).div(None, phi, T).numpy(),
                fvcc.GaussGreenDiv(ctx, m).div(None, phi).numpy(),
                fvcc.GaussGreenLaplacian(ctx, m).laplacian(None, gamma, T, 2.0).numpy()]

    got = {}
    for mode in (1, 0, 2):
        m.set_gather(mode)
        got[mode] = ops()
    for mode in (0, 2):
        for name, a, b in zip(("grad", "div", "upwind", "integrate", "laplacian"), got[mode], got[1]):
            assert np.array_equal(a, b), (mode, name)
    if dtype == np.float64 and N <= 10000:
        g = orc.geometry(poly)
        Th, Tb, ph = T.numpy(), T.boundary.numpy(), phi.values.numpy()
        assert np.array_equal(got[1][0], 1.5 * orc.grad(g, Th, Tb))
        assert np.array_equal(got[1][1], 0.5 * orc.div(g, ph, Th, Tb))
    m.close()


def _crowded(poly, cells=256):
    """The workgroups of `cells` cells that the default lists do not hold: more than 256 lower
    faces from outside, 128 boundary faces or 8 lower faces of a cell from inside."""
    F = len(poly.neighbour)
    ow, nb = poly.owner[:F] // cells, poly.neighbour // cells
    n = -(-poly.n_cells // cells)
    live = np.concatenate([np.zeros(0, np.int64)] + [np.arange(p.start, p.start + p.size) for p in poly.patches if not p.empty])
    outside = np.bincount(nb[ow != nb], minlength=n)
    boundary = np.bincount(poly.owner[live] // cells, minlength=n)
    inside = np.zeros(n, np.int64)
    np.maximum.at(inside, np.arange(poly.n_cells) // cells, np.bincount(poly.neighbour[ow == nb], minlength=poly.n_cells))
    owned = np.bincount(ow, minlength=n)
    return int(np.sum((outside > 256) | (boundary > 128) | (inside > 8) | (owned > 832))), n


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("dims,order", [(d, "block") for d in DIMS] + [((97, 83, 61), "block"), ((33, 20, 27), "zorder"),
                                                                      ((65, 65, 63), "zorder")], ids=str)
def test_every_form_gives_the_bits_of_the_walk(ctx, dims, order, dtype):
    """Each workgroup size asked for (small meshes walk the stencil unless it is), the wide form
    of the 256-cell workgroup where a mesh in lines takes it, and mode 0's own choice, on the two
    large meshes a staged one."""
    import foamadapter_amd as fa
    from foamadapter_amd import fvcc
    print(dims, order, dtype, flush=True)
    poly = fa.PolyMesh.hex(dims, jitter=0.2, jitter_seed=3, **({"perm_seed": 2} if order == "zorder" else {}))
    m = fa.Mesh.from_poly(ctx, poly, renumber=order == "zorder")
    if order == "block":
        crowded, n = _crowded(poly)
        _, over = m.gather_stats(256)
        assert crowded * 100 > n and over < crowded  # the rule of the wide form
    N, F, B = m.n_cells, m.n_internal_faces, m.n_boundary_faces
    T = fvcc.VolumeField(m, ctx.uniform(N, -1, 1, 1, 0, dtype), ctx.uniform(B, -1, 1, 1, 1, dtype),
                         fa.BoundaryConditions(m, ["fixedValue", "fixedGradient"] * 3), "T",
                         ctx.uniform(B, -1, 1, 1, 2, dtype))
    phi = fvcc.SurfaceField(m, ctx.uniform(F + B, -1, 1, 1, 3, dtype))
    gamma = fvcc.SurfaceField(m, ctx.uniform(F + B, 0.5, 2, 1, 4, dtype))
    got = {}
    for mode in (1, 0, 2, 3, 4):
        m.set_gather(mode)
        got[mode] = [fvcc.GaussGreenGrad(ctx, m).grad(T, 1.5).numpy(),
                     fvcc.GaussGreenDiv(ctx, m, ["linear"]).div(None, phi, T, 0.5).numpy(),
                     fvcc.GaussGreenDiv(ctx, m, ["upwind"]).div(None, phi, T).numpy(),
                     fvcc.GaussGreenDiv(ctx, m).div(None, phi).numpy(),
                     fvcc.GaussGreenLaplacian(ctx, m).laplacian(None, gamma, T, 2.0).numpy()]
    for mode in (0, 2, 3, 4):
        for name, a, b in zip(("grad", "div", "upwind", "integrate", "laplacian"), got[mode], got[1]):
            assert np.array_equal(a, b), (mode, name)
    m.close()
