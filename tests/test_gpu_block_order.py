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
