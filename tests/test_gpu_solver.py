"""GPU tests of the device solve of the decoupled Stokes system (KillerSolver,
Solvers.c:2226-2751, with kspgcr, Solvers.c:100-227), against the oracle's
step-by-step restatement (oracle/orc_solver.py) on the blocks the GPU
assembled: the same Powell-Hestenes and GCR iteration counts, a solution that
meets the reference's stopping rule, and the oracle's solution within 1e-5.
These run at penalty 1e5, the value most of the reference's input files set.
At the input default 1e10 the penalty entries exceed the viscous ones by
about 1e13, the momentum residual the stopping rule tests sits at the
rounding floor of the penalised operator, and the iteration counts depend on
the rounding of the factor: the oracle alone, with only its LU column
ordering changed, goes from 2 to 20 Powell-Hestenes iterations and moves the
solution by 100 % on the inclusion model.  There the test asks only for a
solution that meets the stopping rule with a residual like the oracle's.
The drop-in KillerSolver takes host blocks and returns what the context
solve returns; the line search takes the device correction as it takes a
host one."""
import ctypes as C
import os
import sys

import numpy as np
import pytest
import scipy.sparse as sp

import newton_driver as nd

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "oracle"))
import orc_solver  # noqa: E402

pytestmark = pytest.mark.gpu
DP = C.POINTER(C.c_double)
IP = C.POINTER(C.c_int)


def _model(mdz, name, penalty=1e5):
    if name == "inclusion":
        m = mdz.Model.inclusion(41, 41, 1)
    elif name == "pwl":
        m = mdz.Model.pwl_inclusion(60, 60)
    else:
        m = mdz.Model.lithosphere(129, 65, 1)
    m.m.model.penalty = penalty
    return m


def _download(mdz, hot, ctx, i):
    neq, nnz = C.c_int(), C.c_int()
    mdz.check(hot.mdz_ctx_block_info(ctx, i, C.byref(neq), C.byref(nnz)))
    Ic = np.zeros(neq.value + 1, np.int32)
    J = np.zeros(max(nnz.value, 1), np.int32)
    A = np.zeros(max(nnz.value, 1))
    mdz.check(hot.mdz_ctx_download_block(ctx, i, Ic.ctypes.data_as(IP), J.ctypes.data_as(IP), A.ctypes.data_as(DP),
                                         None, None))
    return Ic, J[:nnz.value], A[:nnz.value]


class System:
    """The blocks, residual and penalty diagonals of the context's last unit."""

    def __init__(self, mdz, hot, ctx, it, model):
        nu, npr = it.neq_mom, it.neq_cont
        shapes = [(nu, nu), (nu, npr), (npr, nu)]
        self.raw = [_download(mdz, hot, ctx, i) for i in (0, 1, 2, 4, 5, 6)]
        mats = [sp.csr_matrix((A, J, Ic), shape=shapes[q % 3]) for q, (Ic, J, A) in enumerate(self.raw)]
        self.A, self.B, self.C, self.AJ, self.BJ, self.CJ = mats
        Fm, Fc = np.zeros(nu), np.zeros(npr)
        mdz.check(hot.mdz_ctx_download_residual(ctx, Fm.ctypes.data_as(DP), Fc.ctypes.data_as(DP)))
        self.bu, self.bp = Fm, Fc
        cont = np.zeros(npr, np.int64)
        for c, e in enumerate(it.ep):
            if e >= nu:
                cont[e - nu] = c
        mp = model.m.model
        self.Dpen, self.D1, self.inc = orc_solver.penalty_diagonals(cont, None, None, np.ones(npr),
                                                                    mp.penalty if mp.penalty > 0 else 1e10,
                                                                    mp.dx * mp.dz, mp.dt)
        self.nu, self.np = nu, npr

    def oracle(self, pc_type=0):
        return orc_solver.killer_solver(self.A, self.B, self.C, self.AJ, self.BJ, self.CJ, self.Dpen, self.D1,
                                        self.inc, self.bu, self.bp, pc_type=pc_type)

    def residual(self, x):
        du, dp = x[:self.nu], x[self.nu:]
        return self.bu - self.AJ @ du - self.BJ @ dp, self.bp - self.CJ @ du - self.D1 * dp


def _solve(mdz, hot, ctx, n, nb):
    dx = np.zeros(n)
    info = mdz.solve_info()
    mdz.check(hot.mdz_ctx_solve(ctx, nb, dx.ctypes.data_as(DP), C.byref(info)))
    return dx, info


@pytest.mark.parametrize("nb", [64, 0])
@pytest.mark.parametrize("name", ["inclusion", "pwl", "litho"])
def test_device_solve_matches_oracle(mdz, orc, hot, name, nb):
    print("case", name, "nb", nb, flush=True)
    m = _model(mdz, name)
    gpu = None
    try:
        it = nd.Iterate(mdz, orc, m)
        gpu = nd.GpuAssembler(mdz, hot, m, it)
        gpu()
        sysm = System(mdz, hot, gpu.ctx, it, m)
        dx, info = _solve(mdz, hot, gpu.ctx, it.neq_mom + it.neq_cont, nb)
        du, dp, oi = sysm.oracle()
        ksp = list(info.ksp_its[:info.ph_its])
        print(name, "ph", info.ph_its, oi["ph_its"], "ksp", ksp, oi["ksp_its"], "kd", info.kd, "nb", info.nb,
              "factor ms %.2f iterate ms %.2f" % (info.factor_ms, info.iterate_ms))
        assert info.ph_its == oi["ph_its"]
        assert ksp == oi["ksp_its"]
        # the reference's stopping rule holds for the device solution (recomputed here)
        fu, fp = sysm.residual(dx)
        assert abs(fp.max() - info.maxdiv) <= 1e-9 * max(abs(info.maxdiv0), 1e-300) + 1e-30
        assert np.isclose(info.maxru0, sysm.bu.max(), rtol=1e-14, atol=0)
        assert (abs(fp.max()) < 1e-14 or fp.max() / info.maxdiv0 < 1e-5)
        assert (abs(fu.max()) < 1e-14 or fu.max() / info.maxru0 < 1e-5)
        # both solutions reduce the residual equally far, and agree to the
        # accuracy the tolerances leave
        ox = np.concatenate([du, dp])
        ofu, ofp = sysm.residual(ox)
        b = np.linalg.norm(sysm.bu)
        print(name, "rel residual momentum: device %.3e oracle %.3e" % (np.linalg.norm(fu) / b,
                                                                        np.linalg.norm(ofu) / b))
        assert np.linalg.norm(fu) <= 2 * np.linalg.norm(ofu) + 1e-12 * b
        ddu = np.linalg.norm(dx[:it.neq_mom] - du) / np.linalg.norm(du)
        ddp = np.linalg.norm(dx[it.neq_mom:] - dp) / np.linalg.norm(dp)
        print(name, "device vs oracle du %.3e dp %.3e" % (ddu, ddp))
        assert ddu < 1e-5 and ddp < 1e-5
        # final rms of the residual per equation family (the reference's printout)
        nequ = int((it.eu >= 0).sum())
        assert np.isclose(info.resx, np.sqrt(np.mean(fu[:nequ] ** 2)), rtol=1e-9)
        assert np.isclose(info.resz, np.sqrt(np.mean(fu[nequ:] ** 2)), rtol=1e-9)
        assert np.isclose(info.resp, np.sqrt(np.mean(fp ** 2)), rtol=1e-9, atol=1e-300)
    finally:
        if gpu:
            gpu.close()
        m.free()


@pytest.mark.parametrize("name", ["pwl", "litho"])
def test_symmetrised_jacobian_preconditioner(mdz, orc, hot, name):
    """pc_type 1: the factor is that of (AJ + AJ^T)/2 - B Dpen C
    (Solvers.c:2404-2408); the oracle's iteration counts and solution."""
    print("case pc_type 1", name, flush=True)
    m = _model(mdz, name)
    m.m.model.pc_type = 1
    gpu = None
    try:
        it = nd.Iterate(mdz, orc, m)
        gpu = nd.GpuAssembler(mdz, hot, m, it)
        gpu()
        sysm = System(mdz, hot, gpu.ctx, it, m)
        dx, info = _solve(mdz, hot, gpu.ctx, it.neq_mom + it.neq_cont, 0)
        du, dp, oi = sysm.oracle(pc_type=1)
        ksp = list(info.ksp_its[:info.ph_its])
        print(name, "pc_type 1: ph", info.ph_its, oi["ph_its"], "ksp", ksp, oi["ksp_its"])
        assert info.ph_its == oi["ph_its"]
        assert ksp == oi["ksp_its"]
        ddu = np.linalg.norm(dx[:it.neq_mom] - du) / np.linalg.norm(du)
        print(name, "pc_type 1: device vs oracle du %.3e" % ddu)
        assert ddu < 1e-5
    finally:
        if gpu:
            gpu.close()
        m.free()


@pytest.mark.parametrize("name", ["pwl"])
def test_default_penalty_meets_the_stopping_rule(mdz, orc, hot, name):
    """Penalty 1e10 (the input default): the device solution meets the
    reference's stopping rule, with a momentum residual like the oracle's."""
    m = _model(mdz, name, penalty=0.0)
    gpu = None
    try:
        it = nd.Iterate(mdz, orc, m)
        gpu = nd.GpuAssembler(mdz, hot, m, it)
        gpu()
        sysm = System(mdz, hot, gpu.ctx, it, m)
        dx, info = _solve(mdz, hot, gpu.ctx, it.neq_mom + it.neq_cont, 0)
        du, dp, oi = sysm.oracle()
        fu, fp = sysm.residual(dx)
        ofu, _ = sysm.residual(np.concatenate([du, dp]))
        print(name, "penalty 1e10: ph", info.ph_its, oi["ph_its"], "ksp", list(info.ksp_its[:info.ph_its]),
              oi["ksp_its"], "residual %.3e oracle %.3e" % (np.linalg.norm(fu), np.linalg.norm(ofu)))
        assert (abs(fp.max()) < 1e-14 or fp.max() / info.maxdiv0 < 1e-5)
        assert (abs(fu.max()) < 1e-14 or fu.max() / info.maxru0 < 1e-5)
        assert np.linalg.norm(fu) <= 10 * np.linalg.norm(ofu) + 1e-12 * np.linalg.norm(sysm.bu)
    finally:
        if gpu:
            gpu.close()
        m.free()


def test_factor_is_an_exact_inverse(mdz, orc, hot):
    """On a linear model the Jacobian equals the Picard operator, so the
    factor inverts Js exactly: one GCR direction per Powell-Hestenes
    iteration (kspgcr counts it as 1), for every block size."""
    m = _model(mdz, "inclusion")
    gpu = None
    try:
        it = nd.Iterate(mdz, orc, m)
        gpu = nd.GpuAssembler(mdz, hot, m, it)
        gpu()
        sysm = System(mdz, hot, gpu.ctx, it, m)
        assert abs(sysm.AJ - sysm.A).max() <= 1e-15 * abs(sysm.A).max()
        assert abs(sysm.BJ - sysm.B).max() == 0.0
        for nb in (64, 128, 512):
            _, info = _solve(mdz, hot, gpu.ctx, it.neq_mom + it.neq_cont, nb)
            assert list(info.ksp_its[:info.ph_its]) == [1] * info.ph_its, (nb, list(info.ksp_its[:info.ph_its]))
    finally:
        if gpu:
            gpu.close()
        m.free()


def test_killer_solver_dropin(mdz, orc, hot):
    """The drop-in on host blocks returns the context solve's correction
    (to 1e-10)."""
    m = mdz.Model.lithosphere(96, 48, 2)
    m.m.model.penalty = 1e5
    gpu = None
    try:
        it = nd.Iterate(mdz, orc, m)
        gpu = nd.GpuAssembler(mdz, hot, m, it)
        gpu()
        sysm = System(mdz, hot, gpu.ctx, it, m)
        n = it.neq_mom + it.neq_cont
        dx, info = _solve(mdz, hot, gpu.ctx, n, 0)
        keep = []

        def smat(Ic, J, A, neq):
            s = mdz.SparseMat()
            Ic, J, A = np.ascontiguousarray(Ic, np.int32), np.ascontiguousarray(J, np.int32), np.ascontiguousarray(A)
            keep.extend([Ic, J, A])
            s.Ic, s.J, s.A = Ic.ctypes.data_as(IP), J.ctypes.data_as(IP), A.ctypes.data_as(DP)
            s.neq, s.nnz = neq, len(A)
            return s

        nu, npr = it.neq_mom, it.neq_cont
        neqs = [nu, nu, npr, nu, nu, npr]
        mats = [smat(Ic, J, A, neqs[q]) for q, (Ic, J, A) in enumerate(sysm.raw)]
        D = smat(np.zeros(npr + 1, np.int32), np.zeros(1, np.int32), np.zeros(1), npr)
        D.nnz = 0
        st = mdz.SparseMat()
        st.eqn_u, st.eqn_v, st.eqn_p = (it.eu.ctypes.data_as(IP), it.ev.ctypes.data_as(IP), it.ep.ctypes.data_as(IP))
        st.neq_mom, st.neq_cont, st.neq = nu, npr, nu + npr
        sol = np.zeros(n)
        bu, bp = sysm.bu.copy(), sysm.bp.copy()
        hot.KillerSolver(C.byref(mats[0]), C.byref(mats[1]), C.byref(mats[2]), C.byref(D), None,
                         bu.ctypes.data_as(DP), bp.ctypes.data_as(DP), sol.ctypes.data_as(DP), m.m.model, m.m.mesh,
                         m.m.scaling, C.byref(st), C.byref(st), C.byref(mats[3]), C.byref(mats[4]), C.byref(mats[5]))
        assert hot.mdz_last_status() == 0, hot.mdz_last_error()
        assert np.allclose(sol, dx, rtol=0, atol=1e-10 * np.abs(dx).max())
    finally:
        if gpu:
            gpu.close()
        m.free()


def test_line_search_takes_the_device_correction(mdz, orc, hot):
    """mdz_ctx_line_search(dx = NULL) after a solve equals the call with the
    solve's correction passed from the host, bit for bit."""
    m = mdz.Model.lithosphere(96, 48, 3)
    m.m.model.penalty = 1e5
    gpu = None
    try:
        it = nd.Iterate(mdz, orc, m)
        gpu = nd.GpuAssembler(mdz, hot, m, it)
        gpu()
        dx, _ = _solve(mdz, hot, gpu.ctx, it.neq_mom + it.neq_cont, 0)
        a = -np.array([0.25, 0.5, 1.0])
        r_dev, r_host = np.zeros((3, 3)), np.zeros((3, 3))
        mdz.check(hot.mdz_ctx_line_search(gpu.ctx, None, 3, a.ctypes.data_as(DP), r_dev.ctypes.data_as(DP)))
        mdz.check(hot.mdz_ctx_line_search(gpu.ctx, dx.ctypes.data_as(DP), 3, a.ctypes.data_as(DP),
                                          r_host.ctypes.data_as(DP)))
        assert np.array_equal(r_dev, r_host)
        print("line search after the device solve", r_dev[:, 0])
    finally:
        if gpu:
            gpu.close()
        m.free()


def test_device_solve_matches_oracle_513x257(mdz, orc, hot):
    """A larger lithosphere (264 k momentum unknowns, kd about 513): the
    Picard-preconditioned GCR needs tens of directions per Powell-Hestenes
    iteration here; the device takes the oracle's counts."""
    print("case lithosphere 513x257", flush=True)
    m = mdz.Model.lithosphere(513, 257, 1)
    m.m.model.penalty = 1e5
    gpu = None
    try:
        it = nd.Iterate(mdz, orc, m)
        gpu = nd.GpuAssembler(mdz, hot, m, it)
        gpu()
        sysm = System(mdz, hot, gpu.ctx, it, m)
        dx, info = _solve(mdz, hot, gpu.ctx, it.neq_mom + it.neq_cont, 0)
        du, dp, oi = sysm.oracle()
        ksp = list(info.ksp_its[:info.ph_its])
        print("513x257 ph", info.ph_its, oi["ph_its"], "ksp", ksp, oi["ksp_its"],
              "factor ms %.1f iterate ms %.1f" % (info.factor_ms, info.iterate_ms))
        assert info.ph_its == oi["ph_its"]
        assert all(abs(a - b) <= 1 for a, b in zip(ksp, oi["ksp_its"])), (ksp, oi["ksp_its"])
        ddu = np.linalg.norm(dx[:it.neq_mom] - du) / np.linalg.norm(du)
        print("513x257 device vs oracle du %.3e" % ddu)
        assert ddu < 1e-4
    finally:
        if gpu:
            gpu.close()
        m.free()


def _fill_freed_memory(hot, byte=0xFF):
    """Device memory for the next small and large allocations to find: buffers
    filled with `byte` (0xFF: NaN), every other one freed -- the others, returned, keep
    the freed ones from going back to the system."""
    kept = []
    for size, count in ((1 << 10, 4096), (1 << 18, 64), (1 << 22, 32)):
        ptrs = [C.c_void_p() for _ in range(count)]
        for q in ptrs:
            assert hot.hipMalloc(C.byref(q), C.c_size_t(size)) == 0
            assert hot.hipMemset(q, C.c_int(byte), C.c_size_t(size)) == 0
        assert hot.hipDeviceSynchronize() == 0
        for q in ptrs[::2]:
            assert hot.hipFree(q) == 0
        kept += ptrs[1::2]
    return kept


def test_restarted_gcr_in_used_memory(mdz, orc, hot):
    """One GCR call of three cycles (77 directions), the solver's buffers in
    memory that held NaN before: the oracle's counts.  kspgcr subtracts
    val[i1] of the cycle before, which is never set for the last direction
    of a cycle: 0 there, whatever the buffer held."""
    print("case pwl, rel_tol_KSP 3e-7", flush=True)
    m = mdz.Model.pwl_inclusion(60, 60)
    m.m.model.penalty = 1e5
    m.m.model.rel_tol_KSP = 3e-7
    gpu, kept = None, []
    try:
        it = nd.Iterate(mdz, orc, m)
        gpu = nd.GpuAssembler(mdz, hot, m, it)
        gpu()
        sysm = System(mdz, hot, gpu.ctx, it, m)
        du, dp, oi = orc_solver.killer_solver(sysm.A, sysm.B, sysm.C, sysm.AJ, sysm.BJ, sysm.CJ, sysm.Dpen, sysm.D1,
                                              sysm.inc, sysm.bu, sysm.bp, rel_tol_KSP=3e-7)
        assert max(oi["ksp_its"]) > 2 * orc_solver.RESTART
        kept = _fill_freed_memory(hot)
        dx, info = _solve(mdz, hot, gpu.ctx, it.neq_mom + it.neq_cont, 0)
        ksp = list(info.ksp_its[:info.ph_its])
        ddu = np.linalg.norm(dx[:it.neq_mom] - du) / np.linalg.norm(du)
        print("ksp", ksp, oi["ksp_its"], "du %.2e" % ddu)
        assert ksp == oi["ksp_its"]
        assert ddu < 1e-5
    finally:
        for q in kept:
            hot.hipFree(q)
        if gpu:
            gpu.close()
        m.free()
