"""The bf16 planes of ppb that zmel keeps in the handle: rebuilt after every
set_ppb, per atom and through the rotated-atom map, complete for a call on
another stream, and the same results when a graph replays them."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# the bf16x3 bar of zmel (two products in a row, ~2^-16 each)
TOL = 1e-4


def crand(rng, *sh):
    return np.asfortranarray(rng.standard_normal(sh) + 1j * rng.standard_normal(sh))


def rel(a, b):
    return np.abs(a - b).max() / np.abs(b).max()


def test_planes_follow_set_ppb():
    import ecalj_amd
    import oracle as orc

    orc.build()
    rng = np.random.default_rng(2)
    h = ecalj_amd.Handle(0, "bf16x3")
    try:
        for nv, md in (([5, 33], [7, 20]), ([5, 33], [7, 20]), ([64], [130]), ([3, 9, 4], [1, 40, 6])):
            ppb = [rng.standard_normal((v, v, m)) for v, m in zip(nv, md)]
            flat = np.concatenate([p.ravel(order="F") for p in ppb])
            h.set_ppb(nv, md, flat)
            cm, cq = crand(rng, sum(nv), 3, 2), crand(rng, sum(nv), 40, 2)
            for _ in range(2):  # the planes built, then kept
                g = h.zmel(cm, cq, zmelconjg=True)
                for b in range(2):
                    ref = orc.zmel(nv, md, [1.0] * len(nv), flat, cm[:, :, b], cq[:, :, b], conjg=True)
                    assert rel(g[..., b], ref) < TOL, (nv, md, b)
        with pytest.raises(ecalj_amd.EcaljError):
            h.set_ppb([3, -1, 4], [1, 40, 6], np.zeros(3 * 3 + 40 + 16 * 6))
        assert np.array_equal(h.zmel(cm, cq, zmelconjg=True), g)  # refused: nothing changed
    finally:
        h.close()


def test_planes_in_a_graph():
    import ecalj_amd

    rng = np.random.default_rng(3)
    nv, md, nm, nq = 40, 50, 4, 60
    h = ecalj_amd.Handle(0, "bf16x3")
    try:
        h.set_ppb([nv], [md], rng.standard_normal((nv, nv, md)))
        cm, cq = h.to_dev(crand(rng, nv, nm)), h.to_dev(crand(rng, nv, nq))
        out = h.array((md, nm, nq), np.complex64)
        call = lambda: h.zmel_dev(cm, cq, out, nm=nm, nq=nq, ndima=nv, zmelconjg=True)
        call()
        want = out.download()
        h.graph_begin()
        try:
            call()
        finally:
            gr = h.graph_end()
        for _ in range(3):
            out.zero()
            gr.launch()
            h.sync()
            assert np.array_equal(out.download(), want)
        gr.close()
    finally:
        h.close()
