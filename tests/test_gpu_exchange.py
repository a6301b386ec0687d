"""Vectors crossing the C ABI (afx_exchange.hip): the device permutation, the
direct and the pieced transfer on both sides of their limits, and calls from
several threads at once."""
import ctypes as C
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def make(ni, nj, renumber, model="inviscid"):
    from aeroflex_amd import rans
    m = rans.Mesh.naca_ogrid(ni, nj, r_far=20.0, first_h=2e-3)
    s = rans.Solver(m, viscosity_model=model, renumber=renumber)
    far = rans.BoundaryVariables(mach=0.5, angle=0.03)
    s.set_bcs({"farfield": rans.BoundaryCondition("farfield", far), "wall": rans.BoundaryCondition("slip-wall")})
    return s


# 2 ni nj cells in all: less than a block of the layout kernels (256), one full
# block, two cells more; below the last direct vector (131 072 cells, 4 MB) and on
# it, pieced with a last piece of 128 rows and of 6 144, several pieces per worker
# (and the vectors of one value per cell pieced too)
@pytest.mark.parametrize("ni,nj", [(8, 3), (8, 16), (43, 3), (64, 1023), (64, 1024), (64, 1025), (67, 1024),
                                   (128, 2050)])
def test_rows_keep_their_cells(ni, nj):
    s, f = make(ni, nj, True), make(ni, nj, False)   # f: file order on the device
    rng = np.random.default_rng(ni * nj)
    s.init()
    q = s.get_q().reshape(-1, 4)
    q[:] = q[0] * (1.0 + 0.01 * rng.standard_normal(q.shape))
    s.set_q(q)
    f.set_q(q.ravel())
    assert np.array_equal(s.get_q(), q.ravel())
    assert np.array_equal(f.get_q(), q.ravel())
    for a, b in ((s.calc_dt(), f.calc_dt()), (s.fillRhoRHS()[0], f.fillRhoRHS()[0])):
        # the same operations in the same order per cell: the same bits
        assert np.array_equal(a[:len(a) - 8 * ni], b[:len(b) - 8 * ni])
    n64, n32 = s.fillRhoRHS(0)[1], s.fillRhoRHS(1)[1]
    R64, R32 = s.fillRhoRHS(0)[0], s.fillRhoRHS(1)[0]
    # norms in another summation order: n eps, below 1e-12 at 1e6 entries
    assert abs(np.linalg.norm(R64) - n64) <= 1e-12 * n64
    assert abs(np.linalg.norm(R32) - n32) <= 1e-12 * n32
    # rows out of place differ by about sqrt(2) |R|; the FP32 form itself by
    # 6e-8 sum |flux len| / |R|, below 1e-2 even on the cells of many chords
    # that the coarsest of these grids have
    assert np.linalg.norm(R32 - R64) <= 0.1 * np.linalg.norm(R64)


def test_threads_do_not_mix_their_vectors():
    solvers = [make(64, 400 + 300 * k, True, "spalart-allmaras") for k in range(4)]
    bad = []

    def work(k):
        s, rng = solvers[k], np.random.default_rng(k)
        for _ in range(6):
            q, nu = rng.standard_normal(4 * s.n_cells), rng.standard_normal(s.n_cells)
            s.set_q(q)
            s.set_nu(nu)
            if not (np.array_equal(s.get_q(), q) and np.array_equal(s.get_nu(), nu)):
                bad.append(k)
    team = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in team:
        t.start()
    for t in team:
        t.join()
    assert not bad


# direct and pieced vectors, one and two norms, both operators of the implicit
# step: without pinned memory the same values cross
@pytest.mark.parametrize("model,nj", [("inviscid", 16), ("spalart-allmaras", 16), ("spalart-allmaras", 1100)])
def test_vectors_cross_without_pinned_memory(model, nj):
    from aeroflex_amd import rans
    ni = 64

    def values():
        s = make(ni, nj, True, model)
        s.init()
        s.refill_bcs()
        s.set_cfl(2.0)
        q = s.get_q().reshape(-1, 4)
        q[:s.n_real] *= 1.0 + 1e-3 * np.random.default_rng(nj).standard_normal((s.n_real, 4))
        s.set_q(q.ravel())
        out = [s.get_q(), s.calc_dt()]
        for precision in (rans.AFX_FP64, rans.AFX_FP32):
            out += s.fillRhoRHS(precision)
        if model != "inviscid":
            s.set_nu(s.get_nu() * 1.5)
            out += [s.get_nu(), s.nu_residual()]
        err = s.explicit_solve(0.5)
        if nj < 100:
            for matrix_free in (False,) if model != "inviscid" else (False, True):
                s.set_matrix_free(matrix_free)
                s.fill()
                assert s.compute() == 0
                assert s.solve(relaxation=0.5, tol=0.0, rhs_iterations=2) >= 0
                out.append(s.linear_iterations())
        return out + [err, s.get_q()]
    want = values()
    try:
        assert rans.lib.afx_no_pinned(1) == 0
        got = values()
    finally:
        rans.lib.afx_no_pinned(0)
    assert len(got) == len(want)
    for a, b in zip(got, want):
        assert np.array_equal(a, b)


def test_a_failed_allocation_is_reported_once():
    """The state's first large transfer allocates its device rows; where that
    fails, the next call goes through."""
    from aeroflex_amd import rans
    s, t = make(64, 1100, True), make(64, 1100, True)
    s.init()
    t.init()
    rans.lib.afx_fail_alloc(1)
    with pytest.raises(rans.RansError, match="out of memory"):
        s.get_q()
    rans.lib.afx_fail_alloc(0)
    assert np.array_equal(s.get_q(), t.get_q())


def _free_bytes():
    """Free device memory, from the runtime that the library is linked with."""
    from aeroflex_amd import rans
    free, total = C.c_size_t(), C.c_size_t()
    assert C.CDLL(rans.LIB_PATH).hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def _implicit(s, kind):
    s.set_preconditioner(kind)
    s.set_cfl(2.0)
    s.fill()
    s.compute()
    s.solve(relaxation=0.5, tol=0.0, rhs_iterations=1)
    return s.get_q()


def _batch(s):
    from aeroflex_amd import rans
    s.set_cfl(0.1)
    b = rans.Batch([s])
    b.run(2, 0)
    b.close()
    return s.get_q()


# every set-up that a first call makes: each of its allocations fails once, and
# the call after that goes through with the same result.  Once the solver is closed
# nothing of them is left, to a few of the runtime's chunks of 2 MB; an array of the
# set-ups kept by mistake is 4 MB and more.
@pytest.mark.parametrize("model,call", [
    ("inviscid", lambda s: _implicit(s, "dilu")), ("inviscid", lambda s: _implicit(s, "block-jacobi")),
    ("spalart-allmaras", lambda s: _implicit(s, "dilu")), ("inviscid", lambda s: s.explicit_solve(0.5)),
    ("laminar", lambda s: s.adjoint(np.ones(4 * s.n_cells))), ("inviscid", lambda s: s.tangent(np.ones(4 * s.n_cells))),
    ("inviscid", lambda s: s.adjoint_nodes(np.ones(4 * s.n_cells))[1]), ("inviscid", lambda s: s.get_wall_profile("wall")),
    ("spalart-allmaras", _batch)])
def test_a_set_up_that_failed_halfway_is_run_again(model, call):
    from aeroflex_amd import rans

    def prepared():
        s = make(64, 270, True, model)
        s.init()
        s.refill_bcs()
        q = s.get_q().reshape(-1, 4)
        q[:s.n_real] *= 1.0 + 1e-3 * np.random.default_rng(7).standard_normal((s.n_real, 4))
        s.set_q(q.ravel())
        return s, q.ravel()
    # (five at once: every hardware queue gets its scratch memory, which the runtime keeps)
    warm = [prepared() for _ in range(5)]
    want = [call(w) for w, _ in warm][0]
    before = _free_bytes()
    s, q = prepared()
    failed = 0
    for again in range(80):
        print("attempt", again, flush=True)
        # a solver keeps what the last attempt got, so the second allocation is a
        # new one; a batch that could not be made starts again
        rans.lib.afx_fail_alloc(again + 1 if call is _batch else min(again, 1) + 1)
        try:
            s.set_q(q)
            got = call(s)
            break
        except rans.RansError as e:
            assert "out of memory" in str(e)
            failed += 1
        finally:
            rans.lib.afx_fail_alloc(0)
    assert failed > 0
    assert np.array_equal(np.asarray(got), np.asarray(want))
    s.close()
    assert before - _free_bytes() <= 3 << 21


def test_a_call_that_fails_leaves_no_work_on_its_staging_buffer():
    """The norm's kernels write into the pinned buffer that the call gives back
    when the residual's device rows cannot be had: behind 20 ms of residuals on
    the stream, they have ended by the time of the error."""
    from aeroflex_amd import rans
    s = make(64, 1100, True)
    s.init()
    hip = C.CDLL(rans.LIB_PATH)
    stream = C.c_void_p(s.stream())
    s.launch_stage(0, 0, 400)
    assert hip.hipStreamQuery(stream) != 0   # (not yet done: the queue is longer than the call below)
    rans.lib.afx_fail_alloc(1)
    try:
        with pytest.raises(rans.RansError, match="out of memory"):
            s.fillRhoRHS()
    finally:
        rans.lib.afx_fail_alloc(0)
    assert hip.hipStreamQuery(stream) == 0


@pytest.mark.parametrize("model", ["inviscid", "spalart-allmaras"])
def test_boundary_conditions_that_were_set_in_part_are_refused(model):
    """Setting them again allocates their tables anew (here with other patches of
    wall): where that fails the solver refuses to go on until they are set."""
    from aeroflex_amd import rans
    far = rans.BoundaryVariables(mach=0.5, angle=0.03)
    one = {"farfield": rans.BoundaryCondition("farfield", far), "wall": rans.BoundaryCondition("slip-wall")}
    both = {"farfield": rans.BoundaryCondition("wall"), "wall": rans.BoundaryCondition("slip-wall")}
    s = make(64, 33, True, model)
    s.init()
    s.refill_bcs()
    q = s.get_q()
    want = s.fillRhoRHS()
    failed = 0
    for nth in range(1, 12):
        rans.lib.afx_fail_alloc(nth)
        try:
            s.set_bcs(both)
            break
        except rans.RansError as e:
            assert "out of memory" in str(e)
            failed += 1
            rans.lib.afx_fail_alloc(0)
            with pytest.raises(rans.RansError, match="boundary conditions not set"):
                s.fillRhoRHS()
        finally:
            rans.lib.afx_fail_alloc(0)
        s.set_bcs(one)
        s.set_q(q)
        assert np.array_equal(s.fillRhoRHS()[0], want[0])
    assert failed >= 2
