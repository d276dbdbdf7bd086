"""Sigma_c in frequency modes (sigmodes.hip), the form of large calls with 8 to
24 frequencies, here asked for at small sizes (tuner mode 13), against the
FP64 oracle and the plain contraction."""
import numpy as np
import pytest

from ecalj_amd import synth

pytestmark = pytest.mark.gpu

# bf16x3: each of the two products in a row errs by at most ~2^-16 of its
# factors (the dropped lo*lo term and the two lo roundings); the mode form adds
# 2^-25 of a column's weights; 3.1e-5 is that bound with no averaging (one
# element: 2.1e-5 in the plain form too).  f32:
# 2^-24 per step of sums of up to 24 x 257 and then 257 x 150 terms of random
# sign, 2^-24 sqrt(45 000) = 1.3e-5 (the plain form reaches 2.6e-6).  f64: the
# same count of 2^-53 is 2.4e-14, and residuals of 2^-51.
TOLS = {"bf16x3": 3.1e-5, "f32": 1.3e-5, "f64": 1e-13}
TOL = TOLS["bf16x3"]
MODES = 13


@pytest.fixture(scope="module")
def orc():
    import oracle

    oracle.build()
    return oracle


def crand(rng, *sh):
    return np.asfortranarray(rng.standard_normal(sh) + 1j * rng.standard_normal(sh))


def relerr(a, b):
    return np.abs(a - b).max() / np.abs(b).max()


def physical_weights(orc, rng, nm, ntq, nf):
    t, w = np.polynomial.legendre.leggauss(nf)
    x, wx = 0.5 * (t + 1.0), 0.5 * w
    om = (1.0 - x) / x
    no = max(1, nm // 10)
    ek = np.concatenate([np.sort(rng.uniform(-12, 0, no)), np.sort(rng.uniform(0.5, 60, nm - no))]) / synth.RYDBERG_EV
    eq = np.sort(rng.uniform(-11, 12, ntq)) / synth.RYDBERG_EV
    return orc.wgtim(eq, ek, 0.003, 0.25, x, wx, np.exp(-om ** 2))


def case(orc, seed, ngb, nm, ntq, nf, weights):
    rng = np.random.default_rng(seed)
    z = crand(rng, ngb, nm, ntq)
    w = crand(rng, ngb, ngb, nf + 1) / (1.0 + np.arange(nf + 1)) ** 2  # used through the upper triangle
    if weights == "physical":
        g = physical_weights(orc, rng, nm, ntq, nf)
    elif weights == "random":  # every frequency needed: the plane pool overflows, plain contraction
        g = rng.standard_normal((nf + 1, nm, ntq))
    elif weights == "rank1":
        g = rng.standard_normal((nf + 1, 1, 1)) * rng.standard_normal((1, nm, ntq))
    else:
        g = np.zeros((nf + 1, nm, ntq))
        g[:, nm // 2, 0] = 1.0
    return z, np.asfortranarray(w), np.asfortranarray(g)


# rows: tile remainders and a full tile; columns: a whole number of tiles, one
# more, one group and several; frequencies: both ends and the plane kernel's edges
@pytest.mark.parametrize("prec", ["bf16x3", "f32", "f64"])
@pytest.mark.parametrize("weights", ["physical", "random", "rank1", "one_column"])
@pytest.mark.parametrize("ngb,nm,ntq,nf", [(128, 128, 8, 7), (161, 129, 9, 11), (130, 67, 16, 12), (200, 113, 10, 17),
                                           (257, 150, 7, 18), (131, 80, 33, 23), (33, 9, 5, 9),
                                            (1, 3, 1, 1)])
def test_modes_against_oracle(orc, prec, weights, ngb, nm, ntq, nf):
    import ecalj_amd

    z, w, g = case(orc, ngb + nf, ngb, nm, ntq, nf, weights)
    ref = orc.sigc_imag(z, w, g)
    h = ecalj_amd.Handle(0, prec)
    try:
        h.set_tuning(MODES)
        got = h.sigc(z, w, g)
        again = h.sigc(z, w, g)
        h.set_tuning(6)
        plain = h.sigc(z, w, g)
    finally:
        h.close()
    print(prec, weights, ngb, nm, ntq, nf, relerr(got, ref), relerr(plain, ref), flush=True)
    assert relerr(got, ref) < TOLS[prec]
    assert np.array_equal(got, again)
    assert relerr(got, plain) < TOLS[prec]


@pytest.mark.parametrize("prec", ["bf16x3", "f32", "f64"])
@pytest.mark.parametrize("nms", [[140, 0, 70, 211], [200]])
def test_modes_grouped(orc, nms, prec):
    import ecalj_amd

    ngb, ntq, nf = 150, 11, 14
    zs, ws, gs = zip(*[case(orc, 7 + k, ngb, max(nm, 1), ntq, nf, "physical") for k, nm in enumerate(nms)])
    ref = np.zeros((ntq, ntq), complex, order="F")
    for nm, z, w, g in zip(nms, zs, ws, gs):
        if nm:
            ref = orc.sigc_imag(z, w, g, ref)
    h = ecalj_amd.Handle(0, prec)
    try:
        h.set_tuning(MODES)
        cat = lambda xs: np.concatenate([x.ravel(order="F") for nm, x in zip(nms, xs) if nm])
        dz, dg = h.to_dev(cat(zs).astype(np.complex128 if prec == "f64" else np.complex64)), h.to_dev(cat(gs))
        dw = h.to_dev(np.concatenate([w.ravel(order="F") for w in ws]))
        s = h.array((ntq, ntq))
        s.zero()
        h.sigc_grouped_dev(nms, dz, ngb, ntq, nf, dw, dg, s)
        got = s.download()
    finally:
        h.close()
    print(nms, relerr(got, ref), flush=True)
    assert relerr(got, ref) < TOLS[prec]


def test_modes_more_columns_than_one_sort(orc):
    """17 000 columns: two sorts per k; the oracle's contraction is linear in
    the columns of one middle state, so a few states are compared."""
    import ecalj_amd

    ngb, nm, ntq, nf = 128, 1000, 17, 8
    z, w, g = case(orc, 3, ngb, nm, ntq, nf, "physical")
    keep = np.zeros(nm, bool)
    keep[[0, 3, 499, 963, 964, 999]] = True
    g[:, ~keep, :] = 0.0
    ref = orc.sigc_imag(np.asfortranarray(z[:, keep]), w, np.asfortranarray(g[:, keep]))
    h = ecalj_amd.Handle(0, "bf16x3")
    try:
        h.set_tuning(MODES)
        got = h.sigc(z, w, g)
    finally:
        h.close()
    print(relerr(got, ref), flush=True)
    assert relerr(got, ref) < TOL


def test_modes_non_finite_inputs_reach_the_result(orc):
    import ecalj_amd

    z, w, g = case(orc, 5, 130, 130, 8, 9, "physical")
    h = ecalj_amd.Handle(0, "bf16x3")
    try:
        h.set_tuning(MODES)
        for bad in (np.inf, np.nan):
            w2 = w.copy(order="F")
            w2[3, 70, 4] = bad
            assert not np.isfinite(h.sigc(z, w2, g)).any()
            g2 = g.copy(order="F")
            g2[2, 11, 5] = bad
            s = h.sigc(z, w, g2)
            assert not np.isfinite(s[5]).any() and np.isfinite(np.delete(s, 5, axis=0)).all()
        assert np.array_equal(h.sigc(z, w, np.zeros_like(g)), np.zeros((8, 8)))
    finally:
        h.close()


def test_modes_graph_replay_follows_its_inputs(orc):
    """The ranks are found on the device: a captured call replays with those of
    the weights it meets, also when they need more modes than at capture."""
    import ecalj_amd

    ngb, nm, ntq, nf = 130, 130, 9, 12
    z, w, g1 = case(orc, 21, ngb, nm, ntq, nf, "rank1")
    h = ecalj_amd.Handle(0, "bf16x3")
    try:
        h.set_tuning(MODES)
        dz, dw, dg, s = h.to_dev(z.astype(np.complex64)), h.to_dev(w), h.to_dev(g1), h.array((ntq, ntq))

        def call():
            s.zero()
            h.sigc_dev(1, dz, ngb, nm, ntq, nf, dw, dg, s)

        call()
        h.graph_begin()
        try:
            call()
        finally:
            gr = h.graph_end()
        for weights in ("rank1", "physical", "random", "rank1"):
            g = case(orc, 21, ngb, nm, ntq, nf, weights)[2]
            dg.upload(g)
            call()
            eager = s.download()
            gr.launch()
            h.sync()
            assert np.array_equal(s.download(), eager)
            assert relerr(eager, orc.sigc_imag(z, w, g)) < TOL
        gr.close()
    finally:
        h.close()


@pytest.mark.parametrize("wscale,gscale", [(1e-40, 1.0), (1e-170, 1.0), (1e170, 1e-20), (1.0, 1e-170), (1.0, 1e170)])
def test_modes_f64_do_not_depend_on_the_scale(orc, wscale, gscale):
    """FP64: W or the weights far from 1 in size, as the plain contraction takes
    them; and frequencies whose W is zero or far smaller than the others'."""
    import ecalj_amd

    z, w, g = case(orc, 31, 130, 70, 6, 10, "physical")
    w[:, :, 3] = 0.0
    w[:, :, 4] *= 1e-60
    ref = orc.sigc_imag(z, w, g)
    h = ecalj_amd.Handle(0, "f64")
    try:
        h.set_tuning(MODES)
        got = h.sigc(z, np.asfortranarray(wscale * w), np.asfortranarray(gscale * g))
    finally:
        h.close()
    err = relerr(got / wscale / gscale, ref)
    print(wscale, gscale, err, flush=True)
    assert err < TOLS["f64"]


@pytest.mark.parametrize("prec", ["bf16x3", "f32", "f64"])
def test_modes_with_w_zero(orc, prec):
    import ecalj_amd

    z, w, g = case(orc, 32, 130, 70, 6, 10, "physical")
    h = ecalj_amd.Handle(0, prec)
    try:
        h.set_tuning(MODES)
        assert (h.sigc(z, np.zeros_like(w), g) == 0.0).all()
    finally:
        h.close()


@pytest.mark.parametrize("prec,exact", [("f64", np.longdouble), ("f32", np.float64)])
@pytest.mark.parametrize("ngb,nf", [(64, 16), (96, 20), (40, 9)])
def test_modes_err_no_more_than_the_plain_form(orc, prec, exact, ngb, nf):
    """Few rows per element of Sigma, so that the contraction's rounding shows
    beside the final product's; W positive, as screened interactions are, so
    that its sums over the frequencies grow.  The elements' errors in norm
    against wider sums (some 1500 of them, so their norm scatters by 3%)."""
    import ecalj_amd

    rng = np.random.default_rng(ngb)
    nm, ntq = 8, 40
    b = crand(rng, ngb, ngb)
    x = np.concatenate([[0.0], (1.0 - np.polynomial.legendre.leggauss(nf)[0]) / (1.0 + np.polynomial.legendre.leggauss(nf)[0])])
    w = np.asfortranarray((b @ b.conj().T)[:, :, None] / (1.0 + x ** 2))
    z = crand(rng, ngb, nm, ntq)
    if prec == "f32":
        z = z.astype(np.complex64).astype(np.complex128)
    g = np.asfortranarray(physical_weights(orc, rng, nm, ntq, nf))
    for v in range(nf + 1):  # Hermitian to the last bit: the contraction reads the upper triangle
        w[:, :, v] = np.triu(w[:, :, v], 1) + np.triu(w[:, :, v], 1).conj().T + np.diag(np.diag(w[:, :, v]).real)
    zr, zi = (a.reshape(ngb, -1, order="F").astype(exact) for a in (z.real, z.imag))
    cr, ci = np.zeros_like(zr), np.zeros_like(zr)
    for v in range(nf + 1):
        wr, wi, gv = w[:, :, v].real.astype(exact), w[:, :, v].imag.astype(exact), g[v].ravel(order="F").astype(exact)
        cr += gv * (wr @ zr - wi @ zi)
        ci += gv * (wr @ zi + wi @ zr)
    a, b = (cr + 1j * ci).reshape(ngb * nm, ntq, order="F"), (zr + 1j * zi).reshape(ngb * nm, ntq, order="F")
    ref = a.conj().T @ b
    off = ~np.eye(ntq, dtype=bool)  # (the diagonal's imaginary part is clipped)
    err = {}
    h = ecalj_amd.Handle(0, prec)
    try:
        for name, mode in (("modes", MODES), ("plain", 6)):
            h.set_tuning(mode)
            d = (h.sigc(z, w, g) - ref)[off]
            err[name] = float(np.sqrt((np.abs(d) ** 2).sum()) / np.sqrt((np.abs(ref[off]) ** 2).sum()))
    finally:
        h.close()
    print(prec, ngb, nf, err, flush=True)
    assert err["modes"] < err["plain"]


def test_modes_f64_zmel_at_an_odd_multiple_of_8_bytes(orc):
    """The FP64 modes load zmel in whole 16-byte elements; one that starts between
    them takes the plain contraction (as the FP64 GEMM's rule does)."""
    import ecalj_amd

    ngb, nm, ntq, nf = 130, 70, 6, 10
    z, w, g = case(orc, 33, ngb, nm, ntq, nf, "physical")
    h = ecalj_amd.Handle(0, "f64")
    try:
        flat = np.concatenate([[0.0], z.ravel(order="F").view(float)])
        dz, da, dw, dg, s = h.to_dev(flat), h.to_dev(z), h.to_dev(w), h.to_dev(g), h.array((ntq, ntq))
        out = []
        for mode, p in ((6, da.ptr), (MODES, dz.ptr + 8)):
            h.set_tuning(mode)
            s.zero()
            h.sigc_dev(1, p, ngb, nm, ntq, nf, dw, dg, s)
            out.append(s.download())
    finally:
        h.close()
    assert relerr(out[1], orc.sigc_imag(z, w, g)) < TOLS["f64"]
    assert np.array_equal(out[0], out[1])  # the plain form's digits


@pytest.mark.parametrize("prec", ["bf16x3", "f32", "f64"])
def test_tuner_mode_chooses_the_form(orc, prec):
    """A call large enough for the modes: mode 0 takes them, as 13 does; any other
    forced variant takes the plain contraction."""
    import ecalj_amd

    ngb, nm, ntq, nf = (512, 420, 24, 20) if prec == "bf16x3" else (300, 205, 16, 16)
    z, w, g = case(orc, 34, ngb, nm, ntq, nf, "physical")
    h = ecalj_amd.Handle(0, prec)
    try:
        out = {}
        for mode in (6, 0, MODES):
            h.set_tuning(mode)
            out[mode] = h.sigc(z, w, g)
            # the report names the shapes that ran over the modes, once each
            assert h.tuning_report().count(f"sigc_modes [{ngb} ") == (0 if mode == 6 else 1)
    finally:
        h.close()
    assert np.array_equal(out[0], out[MODES])
    assert (out[6] != out[0]).any() and relerr(out[6], out[0]) < TOLS[prec]
