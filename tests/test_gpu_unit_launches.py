"""GPU test of the 64-row value passes, whose one launch takes the listed general
waves, the tag-free waves and the continuity rows as block ranges -- of one
block family, or of both -- against the pass with one lane per row and no
staging: CSR values and right-hand sides are the same bit for bit.  The grids
lie on both sides of the 2048 blocks up to which both families share a launch
(180 x 120 cells: 2018 and the general waves) and up to which the Jacobian
pass runs at two waves per SIMD (300 x 200 cells: 2800 blocks), down to grids
without a tag-free wave, with ragged last waves."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
DP = C.POINTER(C.c_double)


def _values(mdz, hot, ctx, which):
    neq, nnz = C.c_int(), C.c_int()
    mdz.check(hot.mdz_ctx_block_info(ctx, which, C.byref(neq), C.byref(nnz)))
    A, b, bbc = np.zeros(max(nnz.value, 1)), np.zeros(max(neq.value, 1)), np.zeros(max(neq.value, 1))
    mdz.check(hot.mdz_ctx_download_block(ctx, which, None, None, A.ctypes.data_as(DP), b.ctypes.data_as(DP),
                                         bbc.ctypes.data_as(DP)))
    return A, b, bbc


@pytest.mark.parametrize("cells", [(5, 4), (33, 16), (140, 90), (180, 120), (300, 200)], ids=lambda c: "%dx%d" % c)
def test_one_launch_of_the_value_pass_equals_the_direct_pass(mdz, hot, cells):
    m = mdz.Model.lithosphere(cells[0], cells[1], 6)
    c = C.c_void_p()
    try:
        mdz.check(hot.mdz_ctx_create(C.byref(c), m.m.mesh, C.byref(m.m.materials), C.byref(m.m.model),
                                     C.byref(m.m.scaling)))
        out = []
        for rows in (0, 64):
            mdz.check(hot.mdz_ctx_set_launch_shape(c, 64, rows, rows))
            r = (C.c_double * 3)()
            mdz.check(hot.mdz_ctx_newton_unit(c, r))
            out.append((list(r), [_values(mdz, hot, c, w) for w in range(8)]))
        assert out[0][0] == out[1][0]
        for w, (x, y) in enumerate(zip(out[0][1], out[1][1])):
            for p, q in zip(x, y):
                assert np.array_equal(p, q), w
    finally:
        if c:
            hot.mdz_ctx_destroy(c)
        m.free()
