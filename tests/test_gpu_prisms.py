"""Meshes whose rows have 5 or 3 off-diagonal entries (prisms, plane triangles): the persistent
solvers read slices padded to 6 or 4, the others slices as wide as their longest row.  The
sizes: one ragged slice, more than 256 tiles, 2 and 3 rows per thread."""
import numpy as np
import pytest

from skewed_meshes import prism_block

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    import foamadapter_amd as fa
    with fa.Context(0) as c:
        yield c


def _system(ctx, dims):
    import foamadapter_amd as fa
    from foamadapter_amd import dsl, fvcc
    m = fa.Mesh.from_poly(ctx, prism_block(*dims), renumber=True)
    N, F, B = m.n_cells, m.n_internal_faces, m.n_boundary_faces
    T = fvcc.VolumeField(m, ctx.uniform(N, -1, 1, 3, 0), ctx.uniform(B, -1, 1, 3, 1),
                         fa.BoundaryConditions(m, ["fixedValue"] * m.n_patches), "T")
    gamma = fvcc.SurfaceField(m, ctx.uniform(F + B, 0.5, 2.0, 3, 2))
    return m, T, dsl.assemble(dsl.imp.ddt(T) - dsl.imp.laplacian(gamma, T), T, 0.0, 3.0)


@pytest.mark.parametrize("method", ["double", "mixed", "bicgstab"])
@pytest.mark.parametrize("dims", [(3, 2, 2), (9, 8, 7), (60, 50, 1), (40, 40, 33), (65, 64, 64), (70, 60, 75), (500, 300, 1)],
                         ids=str)
def test_the_forms_of_a_solve_agree(ctx, dims, method):
    from foamadapter_amd import la
    print(dims, method, flush=True)
    m, T, ls = _system(ctx, dims)
    got = []
    for graph in (False, True, True, False):
        x = ctx.uniform(m.n_cells, -1, 1, 12, 4)
        opts = {"solver": "PBiCGStab"} if method == "bicgstab" else {"precision": method}
        st = la.solve_cg(ls, x, dict(opts, relTol=1e-10, maxIter=500, graph=graph))
        got.append((x.numpy(), st))
    for x, st in got[1:]:
        assert (st.numIter, st.initResNorm, st.finalResNorm) == \
            (got[0][1].numIter, got[0][1].initResNorm, got[0][1].finalResNorm)
        assert np.array_equal(x, got[0][0])
    A, b = ls.scipy(), ls.rhs()
    assert np.diff(A.indptr).max() == (4 if dims[2] == 1 else 6) or dims == (3, 2, 2)
    assert np.linalg.norm(b - A @ got[0][0]) <= 1.01e-10 * np.linalg.norm(b)
    m.close()


@pytest.mark.parametrize("precision", ["double", "mixed"])
@pytest.mark.parametrize("dims,width", [((30, 30, 30), 5), ((150, 100, 1), 3)], ids=str)
def test_a_batch_holds_no_padding(ctx, dims, width, precision):
    """A member's vectors and its scaled matrix, `width` entries a row."""
    from foamadapter_amd import la
    print(dims, precision, flush=True)
    m, T, ls = _system(ctx, dims)
    b = la.Batch(ctx, precision, 256, 8)
    x = ctx.uniform(m.n_cells, -1, 1, 12, 4)
    used = ctx.bytes_in_use
    b.add(ls, x)
    size = 8 if precision == "double" else 4
    assert ctx.bytes_in_use - used <= (6 * size + 8 + width * size) * m.n_cells + (1 << 16)
    assert b.solve({"relTol": 1e-8, "maxIter": 500})[0].finalResNorm <= 1e-8
    b.close()
    m.close()
