"""The Hilbert transform: bins around its rounds, outputs around its row tiles
and chunks, elements around a lane's four and a wave's 64, and the coefficient
table kept per mesh (two meshes in turn, meshes that differ in one point),
against the oracle.  The inputs are exact in 32 bits and the sums in 64: 1e-10
bar for both forms (the tables cancel z log((z-b)/(z-a)) + (b-a):
2^-53 (nu / bin width)^2 = 6e-12 for these meshes); the scaled rcxq is stored
in its own type (2^-24)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def mesh(nwhis, shift=0.0):
    e = 0.2 * (np.exp(0.05 * np.arange(nwhis + 1)) - 1.0)
    e[-1] += shift
    return e


def rel(a, b):
    return np.abs(a - b).max() / np.abs(b).max()


@pytest.mark.parametrize("prec,tol", [("f64", 1e-13), ("bf16x3", 2.0 ** -23)])
@pytest.mark.parametrize("nwhis,niw,shape", [(1, 1, (1, 1)), (7, 8, (3, 21)), (8, 9, (8, 8)), (9, 17, (17, 17)),
                                             (31, 20, (5, 13)), (40, 21, (17, 17)), (65, 24, (16, 16)),
                                             (66, 33, (2, 129))])
def test_dpsion_meshes(nwhis, niw, shape, prec, tol):
    import ecalj_amd
    import oracle as orc

    orc.build()
    rng = np.random.default_rng(nwhis)
    r = rng.standard_normal((*shape, nwhis + 1)) + 1j * rng.standard_normal((*shape, nwhis + 1))
    r = np.asfortranarray(r.astype(np.complex64).astype(np.complex128))
    nu = np.concatenate([[0.0], np.sort(rng.uniform(0.01, 2.0, niw - 1))])
    nu2 = nu.copy()
    nu2[-1] += 0.5
    h = ecalj_amd.Handle(0, prec)
    try:
        for fr, f in ((mesh(nwhis), nu), (mesh(nwhis, 0.01), nu), (mesh(nwhis), nu), (mesh(nwhis), nu2)):
            x, y = r.copy(order="F"), r.copy(order="F")
            g = h.dpsion_imag(x, fr, f)
            o = orc.dpsion_imag(y, fr, orc.imatt(f, fr))
            assert rel(g, o) < 1e-10
            assert rel(x[:, :, 1:], y[:, :, 1:]) < tol  # scaled in place
    finally:
        h.close()


# slices from 2 MB (up to 4 or 6 outputs) and from 5 MB (up to 8) take a thread per element; bins around its
# rounds of four; 33 outputs: one in the second chunk
@pytest.mark.parametrize("prec,tol", [("f64", 1e-13), ("bf16x3", 2.0 ** -23)])
@pytest.mark.parametrize("nwhis,niw,shape", [(1, 1, (700, 907)), (4, 4, (301, 500)), (5, 6, (500, 517)),
                                             (7, 8, (700, 907)), (10, 9, (700, 907)), (6, 33, (700, 907))])
def test_dpsion_few_outputs(nwhis, niw, shape, prec, tol):
    import ecalj_amd
    import oracle as orc

    orc.build()
    rng = np.random.default_rng(nwhis)
    r = (rng.standard_normal((*shape, nwhis + 1), np.float32) + 1j * rng.standard_normal((*shape, nwhis + 1), np.float32))
    r = np.asfortranarray(r.astype(np.complex128))
    fr, nu = mesh(nwhis), np.concatenate([[0.0], np.sort(rng.uniform(0.01, 2.0, niw - 1))])
    h = ecalj_amd.Handle(0, prec)
    try:
        x, y = r.copy(order="F"), r.copy(order="F")
        g = h.dpsion_imag(x, fr, nu)
        o = orc.dpsion_imag(y, fr, orc.imatt(nu, fr))
        assert rel(g, o) < 1e-10
        assert rel(x[:, :, 1:], y[:, :, 1:]) < tol
        if nwhis > niw:  # the real axis' own term
            w = np.linspace(0.0, 1.0, niw + 1)
            assert rel(h.dpsion_real(r, fr, w), orc.dpsion_real(r, fr, orc.rmatt(w, fr))) < 1e-9
    finally:
        h.close()
