"""What a persistent solve does when its launches fail: a plain launch whose workgroups do not
meet is launched again cooperatively, a system whose buffers find no room, a refused launch
and a launch whose workgroups lose each other go on kernel by kernel.  The failures are asked
for from the host (fv_linsys_persist_fault); every kernel ends by itself.  A solve that failed
before its x was written gives the bits of the kernel-by-kernel form."""
import ctypes as C

import numpy as np
import pytest

from test_gpu_cg_persistent import _system

pytestmark = pytest.mark.gpu

APART, REFUSED, LOST = 1, 2, 3
SOLVER = {"double": 0, "mixed": 1, "bicgstab": 2}
ONE = (17, 16, 16)      # a launch does the whole solve (FP64)
MANY = (256, 16, 16)    # a solve of several launches
LARGE = (101, 100, 61)  # 3 rows per thread: no whole solves


@pytest.fixture(scope="module")
def ctx():
    import foamadapter_amd as fa
    with fa.Context(0) as c:
        yield c


def _counts(ls, method):
    from foamadapter_amd._lib import call
    h = np.zeros(4, np.int64)
    call("fv_linsys_persist_counts", ls.handle, SOLVER[method], C.c_void_p(h.ctypes.data))
    return dict(zip(("launches", "apart", "refused", "lost"), h.tolist()))


def _fault(ls, method, fault, after=0, exchange=0):
    from foamadapter_amd._lib import call
    call("fv_linsys_persist_fault", ls.handle, SOLVER[method], fault, after, exchange)


def _solve(ctx, m, ls, method, graph=True, limit=4000):
    from foamadapter_amd import la
    x = ctx.uniform(m.n_cells, -1, 1, 12, 4)
    opts = {"solver": "PBiCGStab"} if method == "bicgstab" else {"precision": method}
    st = la.solve_cg(ls, x, dict(opts, relTol=1e-8, maxIter=limit, graph=graph))
    return x.numpy(), st


def _same(got, ref):
    a, b = got[1], ref[1]
    assert (a.numIter, a.initResNorm, a.finalResNorm, a.trueResNorm) == \
        (b.numIter, b.initResNorm, b.finalResNorm, b.trueResNorm)
    assert np.array_equal(got[0], ref[0])


def _short(ctx, dims):
    """A system solved in a few iterations, in one launch also beside other contexts."""
    import foamadapter_amd as fa
    from foamadapter_amd import dsl, fvcc
    m, ls = _system(ctx, dims)
    T = fvcc.VolumeField(m, ctx.uniform(m.n_cells, -1, 1, 12, 0), ctx.zeros((m.n_boundary_faces,)),
                         fa.BoundaryConditions(m, ["fixedValue"] * m.n_patches), "T")
    gamma = fvcc.SurfaceField(m, ctx.uniform(m.n_internal_faces + m.n_boundary_faces, 0.5, 2.0, 12, 3))
    dt = 0.05 * float(m.get("V").mean()) ** (2.0 / 3.0)
    dsl.assemble(dsl.imp.ddt(T) - dsl.imp.laplacian(gamma, T), T, 0.0, dt, ls)
    return m, ls


@pytest.mark.parametrize("method", ["double", "bicgstab"])
@pytest.mark.parametrize("dims,after", [(ONE, 0), (MANY, 0), (MANY, 1)], ids=str)
def test_a_plain_launch_that_does_not_meet(ctx, dims, after, method):
    print(dims, after, method, flush=True)
    m, ls = _system(ctx, dims)
    ref = _solve(ctx, m, ls, method, graph=False)
    _fault(ls, method, APART, after)
    got = _solve(ctx, m, ls, method)
    c = _counts(ls, method)
    assert c["apart"] == 1 and c["refused"] == c["lost"] == 0 and c["launches"] >= after + 2
    _same(got, ref)
    _same(_solve(ctx, m, ls, method), ref)
    m.close()


def test_plain_launches_are_tried_again(ctx):
    """After a miss 128 launches are cooperative ones, which cannot miss; the next is plain."""
    m, ls = _system(ctx, (3, 3, 3))
    ref = _solve(ctx, m, ls, "double", graph=False)
    _fault(ls, "double", APART)
    for i in range(128):
        if i == 127:
            _fault(ls, "double", APART)  # of no effect on the last cooperative one
        _same(_solve(ctx, m, ls, "double"), ref)
    assert _counts(ls, "double") == {"launches": 129, "apart": 1, "refused": 0, "lost": 0}
    _fault(ls, "double", APART)
    _same(_solve(ctx, m, ls, "double"), ref)
    assert _counts(ls, "double") == {"launches": 131, "apart": 2, "refused": 0, "lost": 0}
    m.close()


@pytest.mark.parametrize("after", [0, 1, 2])
def test_a_component_whose_launch_does_not_meet(ctx, after):
    import foamadapter_amd as fa
    from foamadapter_amd import dsl, fvcc
    print(after, flush=True)
    m, ls = _short(ctx, ONE)
    N = m.n_cells
    got = []
    for graph in (False, True):
        x3, b3 = ctx.uniform(3 * N, -1, 1, 13, 2), ctx.uniform(3 * N, -1, 1, 13, 1)
        x3.shape = b3.shape = (N, 3)
        ls.rhs3 = b3
        if graph:
            _fault(ls, "bicgstab", APART, after)
        st = dsl._solve_vec(ls, fvcc.VolumeField(m, x3, None), {"solver": "PBiCGStab", "relTol": 1e-9,
                                                                "maxIter": 400, "graph": graph})
        got.append((x3.numpy(), ls.rhs(), st))
    assert _counts(ls, "bicgstab")["apart"] == 1
    assert got[1][2] == got[0][2]
    assert np.array_equal(got[1][0], got[0][0]) and np.array_equal(got[1][1], got[0][1])
    m.close()


@pytest.mark.parametrize("after,fault", [(0, REFUSED), (1, REFUSED), (2, REFUSED), (2, LOST)])
def test_a_component_goes_on_kernel_by_kernel(ctx, after, fault):
    """The components behind a refused or lost launch are solved one by one: each to its
    tolerance, the system's right-hand side that of the last."""
    from foamadapter_amd import dsl, fvcc
    print(after, fault, flush=True)
    m, ls = _short(ctx, ONE)
    N = m.n_cells
    A = ls.scipy()
    x3, b3 = ctx.uniform(3 * N, -1, 1, 13, 2), ctx.uniform(3 * N, -1, 1, 13, 1)
    x3.shape = b3.shape = (N, 3)
    ls.rhs3 = b3
    _fault(ls, "bicgstab", fault, after)
    st = dsl._solve_vec(ls, fvcc.VolumeField(m, x3, None), {"solver": "PBiCGStab", "relTol": 1e-9, "maxIter": 400})
    c = _counts(ls, "bicgstab")
    assert c["refused" if fault == REFUSED else "lost"] == 1 and len(st) == 3
    x, b = x3.numpy(), b3.numpy()
    for k in range(3):
        res = np.linalg.norm(b[:, k] - A @ x[:, k]) / np.linalg.norm(b[:, k])
        assert st[k].status == 0 and res <= 1.01e-9 and abs(st[k].trueResNorm - res) <= 1e-12
    assert np.array_equal(ls.rhs(), b[:, 2])
    m.close()


CASES = [("double", ONE, 0), ("double", MANY, 0), ("double", MANY, 1), ("double", LARGE, 0), ("double", LARGE, 1),
         ("mixed", ONE, 0), ("mixed", ONE, 1), ("bicgstab", ONE, 0), ("bicgstab", MANY, 0), ("bicgstab", MANY, 1)]


@pytest.mark.parametrize("fault", ["refused", "lost"])
@pytest.mark.parametrize("method,dims,after", CASES, ids=str)
def test_a_solve_goes_on_kernel_by_kernel(ctx, method, dims, after, fault):
    """After a first launch, x of a system without whole solves holds that launch's
    iterations, and the solve goes on from there: its own count, the same tolerance.  (Lost:
    the host takes a launch's state for that of a lost one.)"""
    print(method, dims, after, fault, flush=True)
    m, ls = _system(ctx, dims)
    ref = _solve(ctx, m, ls, method, graph=False)
    _fault(ls, method, REFUSED if fault == "refused" else LOST, after)
    got = _solve(ctx, m, ls, method)
    c = _counts(ls, method)
    assert c[fault] == 1 and sum(c.values()) == c["launches"] + 1
    A, b = ls.scipy(), ls.rhs()
    res = np.linalg.norm(b - A @ got[0]) / np.linalg.norm(b)
    # the CG recurrence estimates the residual: its bound is that of the reference's
    assert res <= max(1.01e-8, 2 * ref[1].trueResNorm) and abs(got[1].trueResNorm - res) <= 1e-10
    if fault == "refused" or dims == MANY and (after or method == "double"):
        assert got[1].initResNorm == ref[1].initResNorm
    if method == "double" and dims == MANY or fault == "refused" and after == 0:
        _same(got, ref)  # x was not written before
    _, later = _solve(ctx, m, ls, method)  # kernel by kernel
    assert later.finalResNorm <= 1e-8 and _counts(ls, method) == c
    m.close()


@pytest.mark.parametrize("method", ["double", "bicgstab"])
def test_a_group_without_one_of_its_workgroups(ctx, method):
    """More than 256 tiles: the sums of 32 workgroups each are collected and published by one of
    them.  One of each group is missing from the last exchange, the result's residual: the
    launch is lost, and the residual reported is the result's, not one of the others' rows."""
    print(method, flush=True)
    m, ls = _short(ctx, (64, 64, 17))
    ref = _solve(ctx, m, ls, method, graph=False)
    n = ref[1].numIter
    _same(_solve(ctx, m, ls, method), ref)
    assert _counts(ls, method)["launches"] == 1
    _fault(ls, method, LOST, 0, 2 * n + 2 if method == "double" else 3 * n + 2)
    x, st = _solve(ctx, m, ls, method)
    assert _counts(ls, method)["lost"] == 1
    A, b = ls.scipy(), ls.rhs()
    res = np.linalg.norm(b - A @ x) / np.linalg.norm(b)
    # every sum is of N terms of one sign: within N eps
    assert np.array_equal(x, ref[0]) and abs(st.trueResNorm - res) <= m.n_cells * 2.3e-16 * res
    m.close()


@pytest.mark.parametrize("method", ["double", "mixed", "bicgstab"])
def test_no_room_for_the_persistent_buffers(method):
    """Room for x and a solver's own vectors and scaled matrix, but not for what the persistent
    form needs beside them (12 bytes a row and more): the same solve, kernel by kernel."""
    import foamadapter_amd as fa
    print(method, flush=True)
    budget, out = 4 << 30, []
    for tight in (False, True):
        with fa.Context(0, hbm_budget=budget) as c:
            m, ls = _system(c, (64, 64, 64))
            rows = m.n_cells
            need = {"double": 8 * 13, "mixed": 4 * 12 + 8, "bicgstab": 8 * 13}[method] * rows + 8 * rows
            if tight:
                rest = c.empty((budget - c.bytes_in_use - need - (1 << 18),), np.uint8)
            out.append(_solve(c, m, ls, method, graph=tight))
            if tight:
                assert _counts(ls, method)["launches"] == 0
                rest.close()
            m.close()
    _same(out[1], out[0])


def test_systems_of_one_pattern_share_the_plan(ctx):
    """What depends on the pattern alone is made once: a second system takes less memory than
    the first, and the BiCGStab of a third uses what the CG made."""
    from foamadapter_amd import la
    m, ls = _system(ctx, (64, 64, 40))
    x = ctx.uniform(m.n_cells, -1, 1, 12, 4)
    took = []
    for method in ("double", "double", "bicgstab"):
        two = la.LinearSystem(ls.sp)
        from foamadapter_amd._lib import call, lib
        call("fv_memcpy_d2d", ctx.handle, lib.fv_linsys_values(two.handle), lib.fv_linsys_values(ls.handle), 8 * ls.sp.nnz)
        call("fv_memcpy_d2d", ctx.handle, lib.fv_linsys_rhs(two.handle), lib.fv_linsys_rhs(ls.handle), 8 * m.n_cells)
        used = ctx.bytes_in_use
        opts = {"solver": "PBiCGStab"} if method == "bicgstab" else {}
        la.solve_cg(two, x, dict(opts, relTol=1e-3, maxIter=2000))
        assert _counts(two, method)["launches"] >= 1
        took.append(ctx.bytes_in_use - used)
        two.close()
    vectors = 8 * 13 * m.n_cells  # of either solver, with its scaled matrix
    assert took[0] >= vectors + 12 * m.n_cells
    assert took[1] <= vectors + (1 << 18) and took[2] <= vectors + (1 << 18)
    m.close()


@pytest.mark.parametrize("method", ["double", "mixed", "bicgstab"])
def test_launches_are_short_beside_another_thread(ctx, method):
    """While another thread uses a context of its own a launch holds the device for a quarter of
    a millisecond (an iteration takes 5 us and more): the same bits.  A context that is idle, or
    used by this thread, changes nothing."""
    import threading
    import time
    import foamadapter_amd as fa
    print(method, flush=True)
    m, ls = _system(ctx, MANY)
    ref = _solve(ctx, m, ls, method, graph=False)

    def launches():
        before = _counts(ls, method)["launches"]
        got = _solve(ctx, m, ls, method)
        _same(got, ref)
        return _counts(ls, method)["launches"] - before

    with fa.Context(0) as other:
        other.sync()
        time.sleep(0.1)  # other tests' threads are long gone
        idle = launches()
        stop = threading.Event()

        def use():
            while not stop.is_set():
                other.sync()
                time.sleep(0.001)
        t = threading.Thread(target=use)
        t.start()
        time.sleep(0.05)
        busy = launches()
        stop.set()
        t.join()
        time.sleep(0.1)
        launches()  # (a mixed solve queues as many as the one before)
        again = launches()
    assert busy >= ref[1].numIter / 50 and idle <= ref[1].numIter / 100 + 8
    assert again <= idle + 2
    m.close()


def test_a_mixed_solve_queues_the_launches_it_needs(ctx):
    """A solve queues as many launches as the one before took, at once: after one of many, a
    short one queues as many once, and the next as many as that took."""
    from foamadapter_amd import la
    m, ls = _system(ctx, MANY)
    took = []
    for tol in (1e-8, 1e-8, 1e-1, 1e-1, 1e-1):
        before = _counts(ls, "mixed")["launches"]
        x = ctx.uniform(m.n_cells, -1, 1, 12, 4)
        st = la.solve_cg(ls, x, {"relTol": tol, "maxIter": 4000, "precision": "mixed"})
        assert st.finalResNorm <= tol and st.numIter >= 12
        took.append(_counts(ls, "mixed")["launches"] - before)
    print(took, flush=True)
    assert took[0] > 3 and took[1] <= took[0] and took[2] == took[1]
    assert took[3] < took[2] and took[4] == took[3]
    m.close()


@pytest.mark.parametrize("dims,limit", [((256, 16, 16), 700), ((257, 16, 16), 700), ((64, 32, 32), 150),
                                        ((41, 40, 40), 130)], ids=str)
def test_a_mixed_solve_cut_by_its_limit_reports_its_residual(ctx, dims, limit):
    """The persistent form runs the iterations it was given, whatever replacements came before
    them, and reports the FP64 residual of the x it leaves.  The rows are summed in the host's
    order: the norms differ by a sum of N terms."""
    from foamadapter_amd import la
    print(dims, limit, flush=True)
    m, ls = _system(ctx, dims)
    A, b = ls.scipy(), ls.rhs()
    for _ in range(2):
        x = ctx.uniform(m.n_cells, -1, 1, 12, 4)
        st = la.solve_cg(ls, x, {"relTol": 1e-12, "maxIter": limit, "precision": "mixed"},
                         raise_on_noconverge=False)
        res = np.linalg.norm(b - A @ x.numpy()) / np.linalg.norm(b)
        assert st.status != 0 and st.numIter == limit and _counts(ls, "mixed")["launches"] > 0
        assert abs(st.finalResNorm - res) <= m.n_cells * 2.3e-16 * res
    m.close()
