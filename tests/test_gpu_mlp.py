"""GPU tests of the surrogate network: training data against the oracle's
Viscosity, the BF16 matrix-core forward / backward / Adam kernels against the
CPU network oracle (tests/mlp_oracle.py, FP64 with the kernels' BF16
rounding points), training, and the learned initial guess in the
device-resident Newton unit.

Tolerances: forward outputs 5e-4 absolute for 99.9 % of the samples (FP32
accumulation order; outputs are O(1)) and 1e-2 for all (a hidden activation
can round to the neighbouring BF16 value);
gradients 5e-3 relative in norm per parameter group against the BF16-rounded
oracle, 5e-2 against the plain FP64 gradient; Adam 1e-6 relative."""
import ctypes as C

import numpy as np
import pytest

import mlp_oracle as mo
from helpers import point_viscosity

pytestmark = pytest.mark.gpu

FP = C.POINTER(C.c_float)


@pytest.fixture(scope="module")
def litho(mdz):
    m = mdz.Model.lithosphere(64, 32, 7)
    yield m
    m.free()


@pytest.fixture
def net(mdz, hot, litho):
    h = C.c_void_p()
    mdz.check(hot.mdz_mlp_create(C.byref(h), C.byref(litho.m.materials), C.byref(litho.m.model),
                                 C.byref(litho.m.scaling)))
    yield h
    hot.mdz_mlp_destroy(h)


def _samples(mdz, hot, net, n, first=0):
    X = np.zeros((n, 9), np.float32)
    Y = np.zeros((n, 2), np.float32)
    mdz.check(hot.mdz_mlp_download_samples(net, first, n, X.ctypes.data_as(FP), Y.ctypes.data_as(FP)))
    return X, Y


def _weights(mdz, hot, net):
    w = np.zeros(mo.NPARAMS, np.float32)
    mdz.check(hot.mdz_mlp_get_weights(net, w.ctypes.data_as(FP), mo.NPARAMS))
    return w


def test_training_labels_are_the_reference_root(mdz, orc, hot, net, litho):
    """Label y0 = 4 log10(eta_ve / eta_ref) from the oracle's Viscosity at the
    decoded inputs (root and initial guess of its visco-elastic solve)."""
    mdz.check(hot.mdz_mlp_generate(net, 4096, 11))
    X, Y = _samples(mdz, hot, net, 4096)
    s = litho.m.scaling
    mt = litho.m.materials
    dt0 = litho.m.model.dt
    try:
        for i in range(0, 4096, 64):
            f = X[i].astype(np.float64)
            E = 10 ** (3 * f[0] - 15) / s.E
            T = (850 * f[1] + 1123) / s.T
            P = (5 * f[2] + 5) * 1e9 / s.S
            tau0 = (250 * f[3] + 250) * 1e6 / s.S
            litho.m.model.dt = 10 ** (f[4] + 11) / s.t
            ph = int(np.argmax(f[5:8]))
            r = point_viscosity(orc, litho, ph, mt.mu[ph], T, P, E, -E, 0.0, d=mt.gs_ref[ph], Txx0=tau0, Tzz0=-tau0,
                                fric=0.5, C_coh=1e30, P0=P, beta=mt.bet[ph])
            # features are stored in FP32: inputs carry ~1e-7 relative rounding
            assert Y[i, 0] == pytest.approx(4 * np.log10(r["eta_ve"] / r["eta_up"]), abs=1e-4), i
            assert Y[i, 0] <= 1e-6  # the root lies below the smallest isolated viscosity
    finally:
        litho.m.model.dt = dt0


def test_forward_and_gradient_against_oracle(mdz, hot, net):
    mdz.check(hot.mdz_mlp_generate(net, 4096, 5))
    mdz.check(hot.mdz_mlp_init(net, 3))
    X, Y = _samples(mdz, hot, net, 4096)
    w = _weights(mdz, hot, net).astype(np.float64)
    yg = np.zeros((4096, 2), np.float32)
    mdz.check(hot.mdz_mlp_predict(net, 0, 4096, yg.ctypes.data_as(FP)))
    yo, _ = mo.forward(w, X, bf=True)
    err = np.abs(yg - yo)
    print("forward max abs err %.2e, 99.9th percentile %.2e" % (err.max(), np.quantile(err, 0.999)))
    assert np.quantile(err, 0.999) <= 5e-4  # FP32 accumulation order
    assert err.max() <= 1e-2                # hidden activations one BF16 ulp apart
    g = np.zeros(mo.NPARAMS, np.float32)
    loss = C.c_double()
    mdz.check(hot.mdz_mlp_gradient(net, 0, 4096, g.ctypes.data_as(FP), C.byref(loss)))
    go, lo = mo.gradient(w, X, Y, bf=True)
    gx, _ = mo.gradient(w, X, Y, bf=False)
    assert loss.value == pytest.approx(lo, rel=1e-3)
    for k, (o, n) in mo.OFF.items():
        a, b, c = g[o:o + n], go[o:o + n], gx[o:o + n]
        e_bf = np.linalg.norm(a - b) / np.linalg.norm(b)
        e_64 = np.linalg.norm(a - c) / np.linalg.norm(c)
        print("%s: rel err vs BF16 oracle %.2e, vs FP64 %.2e" % (k, e_bf, e_64))
        assert e_bf <= 5e-3, k
        assert e_64 <= 5e-2, k


def _gradient(mdz, hot, net, first, count):
    g, loss = np.zeros(mo.NPARAMS, np.float32), C.c_double()
    mdz.check(hot.mdz_mlp_gradient(net, first, count, g.ctypes.data_as(FP), C.byref(loss)))
    return g.astype(np.float64), loss.value


@pytest.mark.parametrize("count", [64, 1024, 8192, 8256])
def test_gradient_of_small_batches(mdz, hot, net, count):
    """Batches up to 8192 take a block for each tile of 32 samples, larger
    ones four tiles a block; here with ragged last blocks (258 tiles).  A
    BF16 rounding that falls the other way moves a sample's term by 2^-8 in
    each of the four layers at most."""
    mdz.check(hot.mdz_mlp_generate(net, 9000, 7))
    mdz.check(hot.mdz_mlp_init(net, 4))
    X, Y = _samples(mdz, hot, net, count, 128)
    g, loss = _gradient(mdz, hot, net, 128, count)
    go, lo = mo.gradient(_weights(mdz, hot, net).astype(np.float64), X, Y, bf=True)
    assert loss == pytest.approx(lo, rel=1e-3)
    for k, (o, n) in mo.OFF.items():
        e = np.linalg.norm(g[o:o + n] - go[o:o + n]) / np.linalg.norm(go[o:o + n])
        print(count, k, "%.2e" % e)
        assert e <= 4 * 2.0 ** -8, k


def test_gradient_is_the_mean_of_its_halves(mdz, hot, net):
    """16384 samples (four tiles a block) against their halves (a block for
    each tile), and those against batches of 64: the same terms -- the
    counts' ratios are powers of two -- in another order of FP32 sums
    (512 partials: 512 x 6e-8)."""
    mdz.check(hot.mdz_mlp_generate(net, 16384, 8))
    mdz.check(hot.mdz_mlp_init(net, 5))
    whole, loss = _gradient(mdz, hot, net, 0, 16384)
    for size in (8192, 64):
        parts = [_gradient(mdz, hot, net, k, size) for k in range(0, 16384, size)]
        assert loss == pytest.approx(sum(p[1] for p in parts), rel=3e-5)
        mean = sum(p[0] for p in parts) / len(parts)
        e = np.linalg.norm(whole - mean) / np.linalg.norm(mean)
        print(size, "%.2e" % e)
        assert e <= 3e-5


def test_inference_form_against_oracle(mdz, hot, net):
    """The network the grid guess evaluates (inference form: log2(e) folded
    into the weights, K-permuted rows on 16x16x32 tiles) against the
    oracle's inference form, with the training forward's bounds; and within
    BF16 noise of the training forward itself.  Random initial weights make
    a wrong permutation or scale an O(1) error."""
    mdz.check(hot.mdz_mlp_generate(net, 4096, 6))
    mdz.check(hot.mdz_mlp_init(net, 8))
    X, _ = _samples(mdz, hot, net, 4096)
    w = _weights(mdz, hot, net).astype(np.float64)
    yi = np.zeros((4096, 2), np.float32)
    mdz.check(hot.mdz_mlp_predict_inference(net, 0, 4096, yi.ctypes.data_as(FP)))
    yo = mo.forward_inference(w, X, bf=True)
    err = np.abs(yi - yo)
    print("inference form: max abs err %.2e, 99.9th percentile %.2e" % (err.max(), np.quantile(err, 0.999)))
    assert np.quantile(err, 0.999) <= 5e-4
    assert err.max() <= 1e-2
    yg = np.zeros((4096, 2), np.float32)
    mdz.check(hot.mdz_mlp_predict(net, 0, 4096, yg.ctypes.data_as(FP)))
    assert np.abs(yi - yg).max() <= 3e-2 * np.abs(yg).max()


def test_adam_step_against_oracle(mdz, hot, net):
    mdz.check(hot.mdz_mlp_init(net, 4))
    w0 = _weights(mdz, hot, net).astype(np.float64)
    rng = np.random.default_rng(0)
    g1 = rng.standard_normal(mo.NPARAMS).astype(np.float32)
    g2 = rng.standard_normal(mo.NPARAMS).astype(np.float32)
    mdz.check(hot.mdz_mlp_adam_step(net, g1.ctypes.data_as(FP), 1e-3))
    mdz.check(hot.mdz_mlp_adam_step(net, g2.ctypes.data_as(FP), 1e-3))
    w, m, v = mo.adam(w0, 0.0, 0.0, g1.astype(np.float64), 1, 1e-3)
    w, m, v = mo.adam(w, m, v, g2.astype(np.float64), 2, 1e-3)
    wg = _weights(mdz, hot, net)
    assert np.abs(wg - w).max() <= 1e-6 * np.abs(w).max() + 1e-7


def test_training_reduces_the_loss(mdz, hot, net):
    mdz.check(hot.mdz_mlp_generate(net, 1 << 17, 9))
    mdz.check(hot.mdz_mlp_init(net, 1))
    hist = (C.c_double * 4)()
    mdz.check(hot.mdz_mlp_train(net, 4, 4096, 1e-3, 2, hist))
    print("loss per epoch", list(hist))
    assert hist[3] < hist[0] and hist[3] < 0.5 * hist[0]


def test_learned_guess_in_the_newton_unit(mdz, orc, hot, net, litho):
    """Learned mode: the network's correction of the reference's guess
    starts the FP32 iteration and FP64 finishes to the reference tolerance;
    fields stay within the mixed-precision bounds; the iteration counts of
    both modes are printed."""
    from helpers import numbering, blocks
    # the training of the benchmark configuration: 2^24 samples, 20 epochs,
    # batch 65536, Adam lr 1e-3 (about 2 s on the GPU)
    mdz.check(hot.mdz_mlp_generate(net, 1 << 24, 21))
    mdz.check(hot.mdz_mlp_init(net, 5))
    hist = (C.c_double * 20)()
    mdz.check(hot.mdz_mlp_train(net, 20, 65536, 1e-3, 3, hist))
    print("loss per epoch", list(hist))
    w = _weights(mdz, hot, net)
    mo_ = litho.clone()
    S = numbering(orc, mdz, mo_)
    bo = blocks(orc, mdz, S, 8)
    orc.orc_newton_unit(mo_.m.mesh, C.byref(mo_.m.materials), C.byref(mo_.m.model), C.byref(mo_.m.Nmodel),
                        C.byref(mo_.m.scaling), C.byref(S), *[C.byref(b) for b in bo])
    counts = {}
    for mode in (1, 2):
        mg = litho.clone()
        ctx = C.c_void_p()
        mdz.check(hot.mdz_ctx_create(C.byref(ctx), mg.m.mesh, C.byref(mg.m.materials), C.byref(mg.m.model),
                                     C.byref(mg.m.scaling)))
        try:
            mdz.check(hot.mdz_ctx_set_network(ctx, w.ctypes.data_as(FP), mo.NPARAMS))
            mdz.check(hot.mdz_ctx_set_rheology_mode(ctx, mode))
            mdz.check(hot.mdz_ctx_collect_histogram(ctx, 1))
            res = (C.c_double * 3)()
            mdz.check(hot.mdz_ctx_newton_unit(ctx, res))
            h = (C.c_longlong * 192)()
            mdz.check(hot.mdz_ctx_iteration_histogram(ctx, h))
            it = np.arange(64)
            counts[mode] = (float((it * np.array(h[128:192])).sum() / sum(h[128:192])),
                            float((it * np.array(h[0:64])).sum() / sum(h[0:64])))
            for k, v in zip(("resx", "resz", "resp"), res):
                ref = getattr(mo_.m.Nmodel, k)
                assert abs(v - ref) <= 1e-10 * abs(ref), (mode, k)
            mdz.check(hot.mdz_ctx_download_grid(ctx, mg.m.mesh))
            from helpers import relerr
            for f in ("eta_n", "eta_s", "sxxd", "sxz", "detadexx_n"):
                e = relerr(mg.field(f), mo_.field(f), 1e-6 if f.startswith("detad") else 1e-8)
                assert e <= 1e-10, (mode, f, e)
        finally:
            hot.mdz_ctx_destroy(ctx)
            mg.free()
    print("mean FP32 / FP64 local iterations: reference guess %.2f / %.2f, learned %.2f / %.2f"
          % (counts[1] + counts[2]))
    # (the reference's guess is within ~1e-3 of the root at most nodes of
    # this model; the gain is asserted where it is poor, in the test below)
    for b in bo:
        orc.orc_free_block(C.byref(b))
    mo_.free()


def _transition_lithosphere(mdz, ncx=256, ncz=128, seed=9):
    """The lithosphere with each layer near its Maxwell transition at the
    background rate (600, 900 and 1200 K for the upper crust, lower crust
    and mantle, +- 40 K seeded noise): the dislocation-creep and elastic
    viscosities are comparable, and the reference's guess -- the smaller of
    the isolated viscosities -- lies up to ~40 % above the root (4-5 FP64
    Newton steps instead of 2-3)."""
    m = mdz.Model.lithosphere(ncx, ncz, seed)
    g = m.m.mesh.contents
    s = m.m.scaling
    nc = (g.Nx - 1) * (g.Nz - 1)
    zc = np.ctypeslib.as_array(g.zc_coord, shape=(g.Nz - 1,))
    depth = -np.repeat(zc, g.Nx - 1) * s.L
    layer = np.where(depth < 20e3, 0, np.where(depth < 35e3, 1, 2))
    T = np.array([600.0, 900.0, 1200.0])[layer] + 40.0 * np.random.default_rng(seed).standard_normal(nc)
    np.ctypeslib.as_array(g.T, shape=(nc,))[:] = T / s.T
    return m


def _unit_counts(mdz, hot, m, w, mode):
    """(total local iterations, mean FP32, mean FP64, mean plastic, norms) of
    one unit in `mode` with the network w."""
    mg = m.clone()
    ctx = C.c_void_p()
    mdz.check(hot.mdz_ctx_create(C.byref(ctx), mg.m.mesh, C.byref(mg.m.materials), C.byref(mg.m.model),
                                 C.byref(mg.m.scaling)))
    try:
        mdz.check(hot.mdz_ctx_set_network(ctx, w.ctypes.data_as(FP), mo.NPARAMS))
        mdz.check(hot.mdz_ctx_set_rheology_mode(ctx, mode))
        mdz.check(hot.mdz_ctx_collect_histogram(ctx, 1))
        res = (C.c_double * 3)()
        mdz.check(hot.mdz_ctx_newton_unit(ctx, res))
        h = (C.c_longlong * 192)()
        mdz.check(hot.mdz_ctx_iteration_histogram(ctx, h))
        h = np.array(h[:])
        it = np.arange(64)
        n = h[0:64].sum()
        f64, pl, f32 = (it * h[0:64]).sum(), (it * h[64:128]).sum(), (it * h[128:192]).sum()
        return f64 + pl + f32, f32 / n, f64 / n, pl / n, list(res)
    finally:
        hot.mdz_ctx_destroy(ctx)
        mg.free()


def test_learned_guess_reduces_local_iterations_where_the_reference_guess_is_poor(mdz, orc, hot):
    """The gain of the trained network over the method without it (mixed
    precision from the reference's guess), on the lithosphere near its
    Maxwell transition (256 x 128): the total number of local iterations
    (FP32 + FP64 + plastic, all node-phase evaluations of one unit) is at
    least 5 % lower, the FP32 iterations strictly lower, and the residual
    norms of both modes equal the oracle's to 1e-10 (every node polished to
    the reference's tolerance).  Training: the C3 configuration on this
    model's flow laws (2^24 samples, 20 epochs, batch 65536)."""
    from helpers import numbering, blocks
    m = _transition_lithosphere(mdz)
    try:
        h = C.c_void_p()
        mdz.check(hot.mdz_mlp_create(C.byref(h), C.byref(m.m.materials), C.byref(m.m.model), C.byref(m.m.scaling)))
        try:
            mdz.check(hot.mdz_mlp_generate(h, 1 << 24, 31))
            mdz.check(hot.mdz_mlp_init(h, 7))
            hist = (C.c_double * 20)()
            mdz.check(hot.mdz_mlp_train(h, 20, 65536, 1e-3, 5, hist))
            w = _weights(mdz, hot, h)
        finally:
            hot.mdz_mlp_destroy(h)
        mixed = _unit_counts(mdz, hot, m, w, 1)
        learned = _unit_counts(mdz, hot, m, w, 2)
        fp64 = _unit_counts(mdz, hot, m, w, 0)
        print("total local iterations: FP64 %d, mixed %d, learned %d (%.1f %% fewer than mixed)"
              % (fp64[0], mixed[0], learned[0], 100.0 * (1.0 - learned[0] / mixed[0])))
        print("means FP32 / FP64 / plastic: mixed %.3f / %.3f / %.3f, learned %.3f / %.3f / %.3f"
              % (mixed[1:4] + learned[1:4]))
        assert learned[0] <= 0.95 * mixed[0]
        assert learned[1] < mixed[1]
        mo_ = m.clone()
        S = numbering(orc, mdz, mo_)
        bo = blocks(orc, mdz, S, 8)
        try:
            orc.orc_newton_unit(mo_.m.mesh, C.byref(mo_.m.materials), C.byref(mo_.m.model), C.byref(mo_.m.Nmodel),
                                C.byref(mo_.m.scaling), C.byref(S), *[C.byref(b) for b in bo])
            for run in (mixed, learned):
                for k, v in zip(("resx", "resz", "resp"), run[4]):
                    ref = getattr(mo_.m.Nmodel, k)
                    assert abs(v - ref) <= 1e-10 * abs(ref), k
        finally:
            for b in bo:
                orc.orc_free_block(C.byref(b))
            mo_.free()
    finally:
        m.free()


def test_error_per_field_by_precision_mode(mdz, orc, hot, net):
    """The error of each precision mode against the FP64 oracle, field by
    field, on the 256x128 lithosphere: plain FP64, FP32 iterations + FP64
    polish, and the same from the network's guess.  Bounds: eta, tau_II and
    the tangent 1e-10 relative (elementwise, floor 1e-8 of the field's scale,
    1e-6 for the sign-changing tangent), CSR values 1e-10 relative to the
    row's largest entry, residual norms 1e-10 relative."""
    from helpers import numbering, blocks, relerr, row_relerr
    mdz.check(hot.mdz_mlp_generate(net, 1 << 22, 31))
    mdz.check(hot.mdz_mlp_init(net, 7))
    hist = (C.c_double * 10)()
    mdz.check(hot.mdz_mlp_train(net, 10, 65536, 1e-3, 5, hist))
    w = _weights(mdz, hot, net)
    mref = mdz.Model.lithosphere(256, 128, 9)
    S = numbering(orc, mdz, mref)
    bo = blocks(orc, mdz, S, 8)
    orc.orc_newton_unit(mref.m.mesh, C.byref(mref.m.materials), C.byref(mref.m.model), C.byref(mref.m.Nmodel),
                        C.byref(mref.m.scaling), C.byref(S), *[C.byref(b) for b in bo])
    tau_o = np.hypot(mref.field("sxxd"), mref.field("sxz_n"))
    rows = []
    try:
        for mode, name in ((0, "fp64"), (1, "mixed"), (2, "learned")):
            mg = mref.clone()
            ctx = C.c_void_p()
            mdz.check(hot.mdz_ctx_create(C.byref(ctx), mg.m.mesh, C.byref(mg.m.materials), C.byref(mg.m.model),
                                         C.byref(mg.m.scaling)))
            try:
                mdz.check(hot.mdz_ctx_set_network(ctx, w.ctypes.data_as(FP), 9090))
                mdz.check(hot.mdz_ctx_set_rheology_mode(ctx, mode))
                res = (C.c_double * 3)()
                mdz.check(hot.mdz_ctx_newton_unit(ctx, res))
                mdz.check(hot.mdz_ctx_download_grid(ctx, mg.m.mesh))
                e = {"eta_n": relerr(mg.field("eta_n"), mref.field("eta_n"), 1e-8),
                     "eta_s": relerr(mg.field("eta_s"), mref.field("eta_s"), 1e-8),
                     "tau_II": relerr(np.hypot(mg.field("sxxd"), mg.field("sxz_n")), tau_o, 1e-8),
                     "detadexx_n": relerr(mg.field("detadexx_n"), mref.field("detadexx_n"), 1e-6),
                     "D11_n": relerr(mg.field("D11_n"), mref.field("D11_n"), 1e-8)}
                for i, lab in ((0, "picard_A"), (4, "jacobian_A"), (5, "jacobian_B")):
                    neq, nnz = C.c_int(), C.c_int()
                    mdz.check(hot.mdz_ctx_block_info(ctx, i, C.byref(neq), C.byref(nnz)))
                    A = np.zeros(max(nnz.value, 1))
                    mdz.check(hot.mdz_ctx_download_block(ctx, i, None, None, A.ctypes.data_as(C.POINTER(C.c_double)),
                                                         None, None))
                    Io, _, Ao, _, _ = mdz.csr_arrays(bo[i])
                    e[lab] = row_relerr(Io, A[:nnz.value], Ao)
                for k, v in zip(("resx", "resz", "resp"), res):
                    ref = getattr(mref.m.Nmodel, k)
                    e[k] = abs(v - ref) / abs(ref)
                rows.append((name, e))
            finally:
                hot.mdz_ctx_destroy(ctx)
                mg.free()
    finally:
        for b in bo:
            orc.orc_free_block(C.byref(b))
        mref.free()
    keys = list(rows[0][1])
    print("\n| mode | " + " | ".join(keys) + " |")
    for name, e in rows:
        print("| %s | " % name + " | ".join("%.1e" % e[k] for k in keys) + " |")
    for name, e in rows:
        for k, v in e.items():
            assert v <= 1e-10, (name, k, v)
