"""GPU tests of the sparse factor behind mdz_ctx_solve at the sizes and
boundary conditions where its tiles and fronts have edges: on linear models
the factor is an exact inverse (one GCR direction per Powell-Hestenes
iteration), on the others the counts and the correction are the oracle's."""
import ctypes as C

import numpy as np
import pytest

import newton_driver as nd
import test_gpu_solver as sv

pytestmark = pytest.mark.gpu


def _solve_case(mdz, orc, hot, m, pc_type=0):
    m.m.model.penalty = 1e5
    m.m.model.pc_type = pc_type
    gpu = None
    try:
        it = nd.Iterate(mdz, orc, m)
        gpu = nd.GpuAssembler(mdz, hot, m, it)
        gpu()
        sysm = sv.System(mdz, hot, gpu.ctx, it, m)
        dx, info = sv._solve(mdz, hot, gpu.ctx, it.neq_mom + it.neq_cont, 0)
        return it, sysm, dx, info, sysm.oracle(pc_type=pc_type)
    finally:
        if gpu:
            gpu.close()
        m.free()


# one tile, tiles of one row, more columns than rows, more than one panel per front
@pytest.mark.parametrize("nx,nz", [(3, 3), (4, 9), (7, 40), (33, 5), (31, 33), (64, 64), (65, 63), (130, 20), (96, 97)])
def test_factor_inverts_linear_models(mdz, orc, hot, nx, nz):
    print("case inclusion", nx, nz, flush=True)
    it, sysm, dx, info, (du, dp, oi) = _solve_case(mdz, orc, hot, mdz.Model.inclusion(nx, nz, 3))
    ksp = list(info.ksp_its[:info.ph_its])
    print(nx, nz, "unknowns", it.neq_mom, "kd", info.kd, ksp, oi["ksp_its"])
    assert ksp == oi["ksp_its"] == [1] * info.ph_its
    # the solutions' accuracy: the viscosity contrast 1e5 under the penalty leaves about 1e-6 (another
    # ordering of the oracle's own factor moves du by 1.4e-6 at 41 x 41)
    assert np.linalg.norm(dx[:it.neq_mom] - du) <= 1e-5 * np.linalg.norm(du)


# walls, free surface with air, Neumann top, with the preconditioners whose matrix
# has a factor (the others are not positive definite: eigenvalues on the host)
@pytest.mark.parametrize("bc,pc_type", [(0, 0), (0, 1), (3, 0), (3, 1), (4, 1)])
def test_factor_of_boundary_families(mdz, orc, hot, bc, pc_type):
    print("case edge", bc, "pc_type", pc_type, flush=True)
    it, sysm, dx, info, (du, dp, oi) = _solve_case(mdz, orc, hot, mdz.Model.edgecase(37, 29, 5, bc, 0), pc_type)
    ksp = list(info.ksp_its[:info.ph_its])
    d = np.linalg.norm(dx[:it.neq_mom] - du) / np.linalg.norm(du)
    print("bc", bc, "pc_type", pc_type, ksp, oi["ksp_its"], "du %.2e" % d)
    assert ksp == oi["ksp_its"]
    assert d < 1e-5


@pytest.mark.parametrize("nx,nz,seed", [(37, 29, 5), (20, 45, 3), (64, 40, 5)])
def test_factor_around_periodic_walls(mdz, orc, hot, nx, nz, seed):
    """The symmetrised Jacobian of a periodic model is positive definite.  Its
    velocities do not conserve volume over the whole box, so the
    divergence only falls to a share of its first value: rel_tol_div = 0.5."""
    print("case periodic", nx, nz, flush=True)
    m = mdz.Model.edgecase(nx, nz, seed, 1, 0)
    m.m.model.penalty, m.m.model.pc_type, m.m.model.rel_tol_div = 1e5, 1, 0.5
    gpu = None
    try:
        it = nd.Iterate(mdz, orc, m)
        gpu = nd.GpuAssembler(mdz, hot, m, it)
        gpu()
        s = sv.System(mdz, hot, gpu.ctx, it, m)
        dx, info = sv._solve(mdz, hot, gpu.ctx, it.neq_mom + it.neq_cont, 0)
        du, dp, oi = sv.orc_solver.killer_solver(s.A, s.B, s.C, s.AJ, s.BJ, s.CJ, s.Dpen, s.D1, s.inc, s.bu, s.bp,
                                                 pc_type=1, rel_tol_div=0.5)
        ksp = list(info.ksp_its[:info.ph_its])
        d = np.linalg.norm(dx[:it.neq_mom] - du) / np.linalg.norm(du)
        print("periodic", nx, nz, ksp, oi["ksp_its"], "du %.2e" % d)
        assert ksp == oi["ksp_its"]
        assert d < 1e-5
    finally:
        if gpu:
            gpu.close()
        m.free()


@pytest.mark.parametrize("bc", [2, 4])
def test_matrix_without_a_factor_is_refused(mdz, orc, hot, bc):
    m = mdz.Model.edgecase(37, 29, 5, bc, 0)
    m.m.model.penalty = 1e5
    gpu = None
    try:
        it = nd.Iterate(mdz, orc, m)
        gpu = nd.GpuAssembler(mdz, hot, m, it)
        gpu()
        dx = np.zeros(it.neq_mom + it.neq_cont)
        rc = hot.mdz_ctx_solve(gpu.ctx, 0, dx.ctypes.data_as(sv.DP), None)
        assert rc == -8 and b"not positive" in hot.mdz_last_error()
    finally:
        if gpu:
            gpu.close()
        m.free()
