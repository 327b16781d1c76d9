"""GPU test of the 64-row value passes, whose one launch takes the listed general
waves, the tag-free waves and the continuity rows as block ranges -- of one
block family, or of both -- against the pass with one lane per row and no
staging: CSR values and right-hand sides are the same bit for bit.  The grids
lie on both sides of the 2048 blocks up to which both families share a launch
(180 x 120 cells: 2018 and the general waves) and up to which the Jacobian
pass runs at two waves per SIMD (300 x 200 cells: 2800 blocks), down to grids
without a tag-free wave, with ragged last waves."""
import ctypes as C
import os
import subprocess
import sys

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


# units of one context, each behind a line on stderr, where the runtime logs every kernel's name
UNITS = """
import ctypes as C, sys
sys.path.insert(0, sys.argv[1])
from conftest import load_pkg
mdz = load_pkg()
hot = mdz.lib_hot()
m = mdz.Model.lithosphere(33, 16, 6)
c, r = C.c_void_p(), (C.c_double * 3)()
mdz.check(hot.mdz_ctx_create(C.byref(c), m.m.mesh, C.byref(m.m.materials), C.byref(m.m.model), C.byref(m.m.scaling)))
for shape in ((), (64, 64, 64), (64, 128, 64), (64, 256, 64), (64, 64, 128)):
    if shape:
        mdz.check(hot.mdz_ctx_set_launch_shape(c, *shape))
    print("unit with", shape, file=sys.stderr, flush=True)
    mdz.check(hot.mdz_ctx_newton_unit(c, r))
print("done", file=sys.stderr, flush=True)
hot.mdz_ctx_destroy(c)
"""


def test_a_set_launch_shape_is_the_one_that_runs():
    """The value pass of both families in one launch of 64-row blocks is for
    contexts that left the shape to the library, or asked for 64 rows."""
    here = os.path.dirname(os.path.abspath(__file__))
    r = subprocess.run([sys.executable, "-c", UNITS, here], env=dict(os.environ, AMD_LOG_LEVEL="3"), text=True,
                       capture_output=True, timeout=100)
    assert r.returncode == 0, r.stderr[-2000:]
    units = r.stderr[:r.stderr.index("done")].split("unit with ")[1:]
    assert len(units) == 5
    if "k_norms_final" not in units[0]:
        pytest.skip("the runtime logs no kernel names")
    launched = [[k for k in ("k_values_pair", "k_values_split", "k_values_mom") if k in u] for u in units]
    print(launched)
    assert launched == [["k_values_pair"], ["k_values_pair"], ["k_values_split", "k_values_mom"],
                        ["k_values_split", "k_values_mom"], ["k_values_split", "k_values_mom"]]
