"""An equation assembled in one pass against the same equation assembled term by term, bit
for bit: the one-pass kernel adds every term's faces, and the terms, in the same order.
The meshes sit at the edges of its workgroups: two cells, lines of 257, a renumbered brick
mesh, lines in block order (the wide lists), and a random numbering that fits no list."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    import foamadapter_amd as fa
    with fa.Context(0) as c:
        yield c


def _mesh(ctx, name):
    import foamadapter_amd as fa
    if name == "one":
        return fa.Mesh.from_poly(ctx, fa.PolyMesh.hex((2, 1, 1)))
    if name == "edge":
        return fa.Mesh.from_poly(ctx, fa.PolyMesh.hex((257, 1, 3), jitter=0.0))
    if name == "bricks":
        return fa.Mesh.from_poly(ctx, fa.PolyMesh.hex((33, 20, 27), jitter=0.2, jitter_seed=2, perm_seed=4),
                                 renumber=True)
    if name == "lines":
        return fa.Mesh.from_poly(ctx, fa.PolyMesh.hex((70, 31, 17), jitter=0.2, jitter_seed=2))
    if name == "walk":  # no list holds a random numbering: every workgroup walks its cells
        return fa.Mesh.from_poly(ctx, fa.PolyMesh.hex((21, 22, 23), jitter=0.2, jitter_seed=2, perm_seed=9))
    raise KeyError(name)


def _fields(ctx, m, ncomp, kinds):
    import foamadapter_amd as fa
    from foamadapter_amd import fvcc
    N, F, B = m.n_cells, m.n_internal_faces, m.n_boundary_faces

    def arr(n, stream, lo=-1.0, hi=1.0):
        a = ctx.uniform(n * ncomp, lo, hi, 21, stream)
        if ncomp > 1:
            a.shape = (n, ncomp)
        return a
    psi = fvcc.VolumeField(m, arr(N, 0), arr(B, 1), fa.BoundaryConditions(m, kinds), "psi", arr(B, 2))
    psi.old_time = fvcc.VolumeField(m, arr(N, 3), None)
    phi = fvcc.SurfaceField(m, ctx.uniform(F + B, -1, 1, 21, 4))
    gamma = fvcc.SurfaceField(m, ctx.uniform(F + B, 0.5, 2, 21, 5))
    other = fvcc.SurfaceField(m, ctx.uniform(F + B, -1, 1, 21, 6))
    sp = ctx.uniform(N, 0.0, 1.0, 21, 7)
    return psi, phi, gamma, other, sp


def _equations(dsl, psi, phi, gamma, other, sp):
    imp, exp = dsl.imp, dsl.exp
    eqs = {"heat": imp.ddt(psi) - imp.laplacian(gamma, psi),
           "momentum": imp.ddt(psi) + imp.div(phi, psi, "upwind") - imp.laplacian(gamma, psi),
           "linear": imp.ddt(psi) * 2.0 + imp.div(phi, psi, "linear") * 0.5 - imp.laplacian(gamma, psi),
           "convection": imp.div(phi, psi, "upwind") + imp.source(sp, psi),
           "diffusion": dsl.Expression(imp.laplacian(gamma, psi) * 3.0)}
    if psi.ncomp == 1:
        eqs["pressure"] = imp.laplacian(gamma, psi) - exp.div(other)
        eqs["sources"] = imp.ddt(psi) - imp.laplacian(gamma, psi) + imp.source(sp, psi) - exp.div(other) * 0.7
    return eqs


@pytest.mark.parametrize("ncomp", [1, 3])
@pytest.mark.parametrize("mesh", ["one", "edge", "bricks", "lines", "walk"])
def test_one_pass_is_bitwise_the_terms_one_by_one(ctx, mesh, ncomp, monkeypatch):
    from foamadapter_amd import dsl, la
    print(mesh, ncomp, flush=True)
    m = _mesh(ctx, mesh)
    kinds = [("fixedValue", "fixedGradient", "zeroGradient")[i % 3] for i in range(m.n_patches)]
    psi, phi, gamma, other, sp = _fields(ctx, m, ncomp, kinds)
    fused = dsl._assemble_fused
    taken = []
    for name, eq in _equations(dsl, psi, phi, gamma, other, sp).items():
        got = []
        for one_pass in (True, False):
            monkeypatch.setattr(dsl, "_assemble_fused",
                                (lambda *a: taken.append(fused(*a)) or taken[-1]) if one_pass else (lambda *a: False))
            ls = la.LinearSystem(la.SparsityPattern.readOrCreate(m))
            if one_pass:  # every entry is written, whatever the system held
                dsl.assemble(dsl.Expression(dsl.imp.laplacian(gamma, psi) * 7.0), psi, 0.0, 0.5, ls)
            dsl.assemble(eq, psi, 0.0, 0.125, ls)
            bm, br = _boundary_coeffs(ctx, m, ls)
            got.append([ls.values(), ls.rhs(), bm, br] + ([ls.rhs3.numpy()] if ncomp > 1 else []))
        for k, (a, b) in enumerate(zip(*got)):
            assert np.array_equal(a, b), (name, k)
    assert taken and all(taken)
    m.close()


def _boundary_coeffs(ctx, m, ls):
    import ctypes as C
    from foamadapter_amd._lib import call
    bm, br = C.c_void_p(), C.c_void_p()
    call("fv_linsys_boundary_coeffs", ls.handle, C.byref(bm), C.byref(br))
    out = []
    for p in (bm, br):
        h = np.empty(m.n_boundary_faces)
        call("fv_memcpy_d2h", ctx.handle, C.c_void_p(h.ctypes.data), p, h.nbytes)
        out.append(h)
    return out


def test_other_orders_are_assembled_term_by_term(ctx):
    """A laplacian before the ddt, a second laplacian, an explicit div of a field: the library
    has no pass for them, and the result is still the equation's."""
    from foamadapter_amd import dsl, la
    m = _mesh(ctx, "bricks")
    psi, phi, gamma, other, sp = _fields(ctx, m, 1, ["fixedValue"] * m.n_patches)
    imp, exp = dsl.imp, dsl.exp
    for eq in (imp.laplacian(gamma, psi) + imp.ddt(psi),
               imp.laplacian(gamma, psi) + imp.laplacian(gamma, psi),
               imp.laplacian(gamma, psi) - exp.div(phi, psi)):
        ls = la.LinearSystem(la.SparsityPattern.readOrCreate(m))
        assert not dsl._assemble_fused(eq, psi, 0.1, ls)
        dsl.assemble(eq, psi, 0.0, 0.1, ls)
        assert np.all(np.isfinite(ls.values())) and np.any(ls.values() != 0.0)
    m.close()


@pytest.mark.parametrize("coefficient", ["psi", "other"])
def test_source_with_a_vector_coefficient(ctx, coefficient, monkeypatch):
    """A Vec3 equation whose source coefficient is the field itself (each component's equation
    has that component) or an array of another shape than one value a cell: not one for the
    one-pass kernel, which reads one value a cell for all components."""
    from foamadapter_amd import dsl, la
    m = _mesh(ctx, "bricks")
    psi, phi, gamma, other, sp = _fields(ctx, m, 3, ["fixedValue"] * m.n_patches)
    wide = ctx.uniform(3 * m.n_cells, 0.0, 1.0, 21, 8)
    eq = dsl.imp.ddt(psi) - dsl.imp.laplacian(gamma, psi) + dsl.imp.source(psi if coefficient == "psi" else wide, psi)
    fused = dsl._assemble_fused
    got = []
    for one_pass in (True, False):
        monkeypatch.setattr(dsl, "_assemble_fused", fused if one_pass else (lambda *a: False))
        ls = la.LinearSystem(la.SparsityPattern.readOrCreate(m))
        dsl.assemble(eq, psi, 0.0, 0.125, ls)
        got.append([ls.values(), ls.rhs(), ls.rhs3.numpy()])
    for a, b in zip(*got):
        assert np.array_equal(a, b)
    m.close()
