"""GPU tests of the marker binning where it has edges, each against the
oracle's sequential sums: bins longer than the counting sort orders, no
markers or none active, the smallest grids, markers outside the box, periodic
walls (the strain's mean between the strain and the softening) and more
phases than the step keeps in registers."""
import ctypes as C

import numpy as np
import pytest

from markers_util import DP, Markers, node_types, seed_markers
from test_gpu_markers import CFD, _cmp_fields, _ctx_step, _oracle_marker_step, _softening

pytestmark = pytest.mark.gpu


def _check_step(mdz, orc, hot, m, mk, nph):
    mo = m.clone()
    try:
        _ctx_step(mdz, hot, m, mk)
        _oracle_marker_step(orc, mo, mk)
        for f in "ns":
            for p in range(nph):
                name = "phase_perc_%s:%d" % (f, p)
                assert np.array_equal(m.field(name), mo.field(name)), name
        _cmp_fields(m, mo, CFD, 1e-14)
    finally:
        mo.free()


@pytest.mark.parametrize("itp", [1, 9])
@pytest.mark.parametrize("active", [511, 512, 513, 3000])
def test_crowded_bin(mdz, orc, hot, active, itp):
    """One bin -- the quarter cell of the 1-node stencil, the centroid's and
    the vertex's of the 9-node one -- holds `active` active markers: up to
    512 are ordered in place, more go through the radix sort."""
    print("case active", active, itp, flush=True)
    m = mdz.Model.lithosphere(30, 20, 4)
    _softening(m)
    m.m.model.itp_stencil = itp
    mk = seed_markers(mdz, m, (2, 2), seed=3, phase="layers")
    g, p = m.m.mesh.contents, m.m.model
    rng = np.random.default_rng(1)

    def in_bins(k):
        """active markers of k in each of the stencil's bins around cell (7, 5)'s upper left quarter"""
        x, z = (k.x - p.xmin) / g.dx, (k.z - p.zmin) / g.dz
        cell, vertex = (np.floor(x) == 7) & (np.floor(z) == 5), (np.rint(x) == 7) & (np.rint(z) == 6)
        return [int((b & (k.phase != -1)).sum()) for b in ([cell & vertex] if itp == 1 else [cell, vertex])]

    crowd = active - in_bins(mk)[0]
    n = crowd + 200  # (200 inactive ones among them)
    x = p.xmin + (7 + rng.uniform(0.05, 0.45, n)) * g.dx
    z = p.zmin + (5 + rng.uniform(0.55, 0.95, n)) * g.dz
    phase = np.concatenate([rng.integers(0, 3, crowd), np.full(n - crowd, -1)])
    perm = rng.permutation(mk.n + n)
    mk = Markers(mdz, np.concatenate([mk.x, x])[perm], np.concatenate([mk.z, z])[perm],
                 np.concatenate([mk.phase, phase])[perm],
                 np.concatenate([mk.strain_pl, rng.exponential(1.0, n)])[perm])
    assert in_bins(mk) == [active] * (1 if itp == 1 else 2)
    try:
        _check_step(mdz, orc, hot, m, mk, 3)
    finally:
        m.free()


@pytest.mark.parametrize("itp,per_cell", [(1, (11, 11)), (1, (12, 12)), (9, (5, 6)), (9, (6, 6))])
def test_dense_bins(mdz, orc, hot, itp, per_cell):
    """Markers a bin below and above the 32 at which the radix sort takes
    over: 30.25 and 36 a quarter cell, 30 and 36 a centroid."""
    m = mdz.Model.lithosphere(14, 11, 4)
    _softening(m)
    m.m.model.itp_stencil = itp
    mk = seed_markers(mdz, m, per_cell, seed=6, phase="layers", inactive=0.05, outside=10)
    try:
        _check_step(mdz, orc, hot, m, mk, 3)
    finally:
        m.free()


@pytest.mark.parametrize("nx,nz", [(3, 3), (4, 3), (33, 3), (65, 17)])
def test_small_grids_and_markers_outside(mdz, orc, hot, nx, nz):
    m = mdz.Model.lithosphere(nx, nz, 4)
    _softening(m)
    mk = seed_markers(mdz, m, (3, 3), seed=nx, phase="layers", inactive=0.1, outside=20)
    try:
        _check_step(mdz, orc, hot, m, mk, 3)
    finally:
        m.free()


@pytest.mark.parametrize("n", [0, 5])
def test_no_active_markers(mdz, orc, hot, n):
    m = mdz.Model.lithosphere(12, 9, 4)
    mk = Markers(mdz, np.zeros(n), np.zeros(n), np.full(n, -1), np.zeros(n))
    try:
        _check_step(mdz, orc, hot, m, mk, 3)
    finally:
        m.free()


@pytest.mark.parametrize("bc", [1, 3])
def test_periodic_walls_and_air(mdz, orc, hot, bc):
    m = mdz.Model.edgecase(40, 24, 6, bc, 1)
    _softening(m)
    mk = seed_markers(mdz, m, (4, 4), seed=9, inactive=0.05)
    try:
        _check_step(mdz, orc, hot, m, mk, 3)
    finally:
        m.free()


def test_more_phases_than_registers_hold(mdz, orc, hot):
    """Six phases: the fractions against P2Mastah's drop-in, which takes the
    general gather of its own bins."""
    m = mdz.Model.lithosphere(40, 20, 4)
    mesh, nph = m.m.mesh.contents, 6
    keep = [np.zeros(n) for n in (40 * 20, 41 * 21) for _ in range(nph)]
    ptrs = [(DP * nph)(*[a.ctypes.data_as(DP) for a in keep[q * nph:(q + 1) * nph]]) for q in (0, 1)]
    old = [C.cast(q, C.c_void_p).value for q in (mesh.phase_perc_n, mesh.phase_perc_s)]
    mk = seed_markers(mdz, m, (4, 4), seed=2)
    mk.phase[:] = np.random.default_rng(5).integers(0, nph, mk.n)
    mesh.phase_perc_n, mesh.phase_perc_s = [C.cast(q, C.POINTER(DP)) for q in ptrs]
    m.m.model.Nb_phases = m.m.materials.Nb_phases = nph
    for p in range(3, nph):
        m.m.materials.C[p], m.m.materials.phi[p] = m.m.materials.C[0], 0.1 * p
    try:
        _ctx_step(mdz, hot, m, mk)
        step = [a.copy() for a in keep]
        assert max(a.max() for a in step) == 1.0
        for centroid in (1, 0):
            hot.P2Mastah(C.byref(m.m.model), mk.m, None, m.m.mesh, None, node_types(m, centroid), 0, 0, 1, centroid, 1)
            assert hot.mdz_last_status() == 0, hot.mdz_last_error()
        for a, b in zip(step, keep):
            assert np.array_equal(a, b)
    finally:
        mesh.phase_perc_n, mesh.phase_perc_s = [C.cast(q, C.POINTER(DP)) for q in old]
        m.free()
