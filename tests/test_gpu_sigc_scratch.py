"""Scratch of the Sigma_c mode form: groups of k below a limit, and the plain
contraction for a k whose mode planes pass it or for which there is no room."""
import numpy as np
import pytest

from test_gpu_sigc_modes import MODES, TOLS, case, orc, relerr  # noqa: F401  (orc: fixture)

pytestmark = pytest.mark.gpu


def uniform(h, prec, nk, ngb, nm, ntq, nf, data):
    z, w, g = (np.concatenate([d[i].ravel(order="F") for d in data]) for i in range(3))
    dz = h.to_dev(z.astype(np.complex128 if prec == "f64" else np.complex64))
    dw, dg, s = h.to_dev(w), h.to_dev(g), h.array((ntq, ntq))

    def call(form):
        s.zero()
        if form == "grouped":
            h.sigc_grouped_dev([nm] * nk, dz, ngb, ntq, nf, dw, dg, s)
        else:
            h.sigc_dev(nk, dz, ngb, nm, ntq, nf, dw, dg, s)
        return s

    return call


# one k takes 43 (bf16x3), 16 (f32) and 58 MB (f64) with its czmelwc: no limit (all five in one group), then
# a limit for two (groups of 2, 2, 1) and for none (plain contraction)
@pytest.mark.parametrize("form", ["uniform", "grouped"])
@pytest.mark.parametrize("prec,limits", [("bf16x3", (100 << 20, 8 << 20)), ("f32", (40 << 20, 8 << 20)),
                                         ("f64", (130 << 20, 8 << 20))])
def test_groups_and_fallback(orc, monkeypatch, prec, form, limits):  # noqa: F811
    import ecalj_amd

    nk, ngb, nm, ntq, nf = 5, 150, 60, 9, 13
    data = [case(orc, 40 + k, ngb, nm, ntq, nf, "physical") for k in range(nk)]
    ref = np.zeros((ntq, ntq), complex, order="F")
    for z, w, g in data:
        ref = orc.sigc_imag(z, w, g, ref)
    h = ecalj_amd.Handle(0, prec)
    try:
        h.set_tuning(MODES)
        call = uniform(h, prec, nk, ngb, nm, ntq, nf, data)
        monkeypatch.delenv("ECALJ_SIG_MODE_SCRATCH", raising=False)
        whole = call(form).download()
        monkeypatch.setenv("ECALJ_SIG_MODE_SCRATCH", str(limits[0]))
        parts = call(form).download()
        monkeypatch.setenv("ECALJ_SIG_MODE_SCRATCH", str(limits[1]))
        plain = call(form).download()
    finally:
        h.close()
    print(prec, form, relerr(whole, ref), relerr(plain, ref), flush=True)
    assert relerr(whole, ref) < TOLS[prec] and relerr(plain, ref) < TOLS[prec]
    assert (whole == parts).all()  # a k's modes and sums do not depend on its group
    assert (whole != plain).any()


def test_one_k_beyond_the_limit_takes_the_plain_form():
    """n = 2600, 21 frequencies in FP64: the planes of the modes would take 25 GB,
    the plain form's 2.3 GB."""
    import ctypes

    import ecalj_amd

    def free_bytes():
        a, b = ctypes.c_size_t(), ctypes.c_size_t()
        assert ecalj_amd.lib().hipMemGetInfo(ctypes.byref(a), ctypes.byref(b)) == 0  # (of the library's HIP runtime)
        return a.value

    ngb, nf = 2600, 20
    h = ecalj_amd.Handle(0, "f64")
    try:
        h.set_tuning(MODES)
        z, w, g, s = (h.array(n, t) for n, t in ((ngb, complex), (ngb * ngb * (nf + 1), complex), (nf + 1, float),
                                                 (1, complex)))
        for a in (z, w, g, s):
            a.zero()
        h.sync()
        before = free_bytes()
        h.sigc_dev(1, z, ngb, 1, 1, nf, w, g, s)
        h.sync()
        assert "sigc_modes" not in h.tuning_report()
        taken = before - free_bytes()
        assert s.download()[0] == 0.0
    finally:
        h.close()
    print("scratch", taken, flush=True)
    assert taken < 4 << 30


def test_capture_after_a_plain_warm_up(orc, monkeypatch):  # noqa: F811
    """No room for the modes (here: nothing may grow under capture, and the
    warm-up took the plain form): the call takes the plain form."""
    import ecalj_amd

    nk, ngb, nm, ntq, nf = 2, 140, 50, 7, 9
    data = [case(orc, 60 + k, ngb, nm, ntq, nf, "physical") for k in range(nk)]
    h = ecalj_amd.Handle(0, "f64")
    try:
        h.set_tuning(MODES)
        call = uniform(h, "f64", nk, ngb, nm, ntq, nf, data)
        monkeypatch.setenv("ECALJ_SIG_MODE_SCRATCH", "1000")
        plain = call("uniform").download()
        monkeypatch.delenv("ECALJ_SIG_MODE_SCRATCH")
        h.graph_begin()
        try:
            s = call("uniform")
        finally:
            gr = h.graph_end()
        for _ in range(2):
            gr.launch()
            h.sync()
            assert (s.download() == plain).all()
        gr.close()
    finally:
        h.close()


@pytest.mark.parametrize("prec,nf,nk", [("f64", 20, 3300), ("f32", 20, 3300), ("f64", 7, 4200)])
def test_more_k_than_one_grid_holds(orc, prec, nf, nk):  # noqa: F811
    """(k, frequency) and (k, group) pairs beyond 65535: several launches."""
    import ecalj_amd

    ngb, nm, ntq = 8, 1, 2
    four = [case(orc, 80 + k, ngb, nm, ntq, nf, "physical") for k in range(4)]
    h = ecalj_amd.Handle(0, prec)
    try:
        call = uniform(h, prec, nk, ngb, nm, ntq, nf, [four[k % 4] for k in range(nk)])
        plain = call("uniform").download()
        h.set_tuning(MODES)
        got = call("uniform").download()
    finally:
        h.close()
    print(prec, nf, nk, relerr(got, plain), flush=True)
    assert relerr(got, plain) < TOLS[prec]
