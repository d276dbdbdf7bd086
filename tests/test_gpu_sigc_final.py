"""The bf16x3 final product (sigfinal.hip) through Sigma_c: 16-column tile
edges of ntq, the largest ntq it takes and one more (the GEMM engine), rows
below, at and beyond a chunk; uniform and grouped k-points."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# one bf16x3 product per factor of czmelwc (2^-16 of each, no averaging assumed)
TOL = 2e-5


def crand(rng, *sh):
    return np.asfortranarray(rng.standard_normal(sh) + 1j * rng.standard_normal(sh))


@pytest.mark.parametrize("ngb,nms", [(5, [3]), (32, [16, 16]), (67, [61, 0, 5, 30])])
@pytest.mark.parametrize("ntq", [1, 16, 17, 33, 48, 49, 64, 65])
def test_final_product(ngb, nms, ntq):
    import ecalj_amd
    import oracle as orc

    orc.build()
    rng = np.random.default_rng(ngb + ntq)
    niw = 2
    zs = [crand(rng, ngb, nm, ntq) for nm in nms]
    gs = [np.asfortranarray(rng.standard_normal((niw + 1, nm, ntq))) for nm in nms]
    ws = [crand(rng, ngb, ngb, niw + 1) for _ in nms]
    ref = np.zeros((ntq, ntq), complex, order="F")
    for nm, z, g, w in zip(nms, zs, gs, ws):
        if nm:
            ref = orc.sigc_imag(z, w, g, ref)
    cat = lambda xs: np.concatenate([x.ravel(order="F") for x in xs])
    h = ecalj_amd.Handle(0, "bf16x3")
    try:
        h.set_tuning(1)
        dz, dg, dw = h.to_dev(cat(zs).astype(np.complex64)), h.to_dev(cat(gs)), h.to_dev(cat(ws))
        s = h.array((ntq, ntq))
        s.zero()
        h.sigc_grouped_dev(nms, dz, ngb, ntq, niw, dw, dg, s)
        out = [s.download()]
        if len(set(nms)) == 1:
            s.zero()
            h.sigc_dev(len(nms), dz, ngb, nms[0], ntq, niw, dw, dg, s)
            out.append(s.download())
    finally:
        h.close()
    for o in out:
        assert np.abs(o - ref).max() / np.abs(ref).max() < TOL, (ngb, nms, ntq)
