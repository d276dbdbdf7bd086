"""The large-product FP64 kernel (gemm64.hip) through the inversion, the W
build and zmel: tile edges (128 rows, 64 columns, 8 k), K remainders, both
operand layouts, conjugations and the Gauss-Jordan epilogue, against numpy /
the oracle.  FP64 bars: rounding of n-long sums times the condition number
(well under 1e-10 for these inputs, the repository's FP64 bar)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def crand(rng, *sh):
    return np.asfortranarray(rng.standard_normal(sh) + 1j * rng.standard_normal(sh))


def rel(a, b):
    return np.abs(a - b).max() / np.abs(b).max()


@pytest.mark.parametrize("n,nb", [(129, 40), (200, 64), (321, 24), (384, 40), (385, 33)])
def test_inverse_batched(n, nb):
    import ecalj_amd

    rng = np.random.default_rng(n)
    a = np.stack([crand(rng, n, n) + 2.0 * np.sqrt(n) * np.eye(n) for _ in range(nb)], axis=2)
    h = ecalj_amd.Handle(0, "f64")
    try:
        d = h.to_dev(np.asfortranarray(a))
        h.zminv_dev(d, n, nbatch=nb)
        h.sync()
        g = d.download().reshape(n, n, nb, order="F")
    finally:
        h.close()
    for b in (0, nb // 2, nb - 1):
        assert rel(g[:, :, b], np.linalg.inv(a[:, :, b])) < 1e-11, (n, b)


@pytest.mark.parametrize("n,nw", [(130, 64), (200, 33), (257, 24)])
def test_w_build(n, nw):
    import ecalj_amd
    import oracle as orc

    orc.build()
    rng = np.random.default_rng(n)
    vc = rng.uniform(0.5, 10.0, n)
    q = np.asfortranarray(np.linalg.qr(crand(rng, n, n))[0])
    x = crand(rng, n, 60) * 0.02
    chi = np.stack([-(x @ x.conj().T) / (1.0 + i) for i in range(nw)], axis=2)
    h = ecalj_amd.Handle(0, "f64")
    try:
        h.set_coulomb(vc, q)
        g = h.wc_build(chi)
    finally:
        h.close()
    pick = [0, nw - 1]
    ref = orc.wc_build(np.asfortranarray(chi[:, :, pick]), np.sqrt(vc), q)
    assert rel(g[:, :, pick], ref) < 1e-11


# second contraction of zmel with N = 33 .. 200 columns and K = nv = 27 .. 65, to the E basis (A^H B) too
@pytest.mark.parametrize("nv,md,nm,nq,nb", [(27, 129, 3, 33, 40), (64, 130, 5, 65, 30), (65, 250, 2, 200, 16)])
def test_zmel(nv, md, nm, nq, nb):
    import ecalj_amd
    import oracle as orc

    orc.build()
    rng = np.random.default_rng(nv)
    ppb = np.asfortranarray(rng.standard_normal((nv, nv, md)))
    cm, cq = crand(rng, nv, nm, nb), crand(rng, nv, nq, nb)
    m2e = np.asfortranarray(np.linalg.qr(crand(rng, md, md))[0])
    h = ecalj_amd.Handle(0, "f64")
    try:
        h.set_ppb([nv], [md], ppb)
        h.set_coulomb(np.ones(md), m2e)
        for is_m, conj in ((True, True), (False, False), (True, False)):
            g = h.zmel(cm, cq, is_m_basis=is_m, zmelconjg=conj)
            for b in (0, nb - 1):
                ref = orc.zmel([nv], [md], [1.0], ppb, cm[:, :, b], cq[:, :, b], m2e=None if is_m else m2e, conjg=conj)
                assert rel(g[..., b], ref) < 1e-12
    finally:
        h.close()
