"""The bf16 planes of ppb that zmel keeps in the handle: rebuilt per atom after
every set_ppb, complete for a call on another stream, the same results when a
graph replays them, and split anew in a graph captured before they are built.
(The rotated-atom map: test_gpu_zmel_core.py.)"""
import ctypes

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


def test_capture_between_set_ppb_and_the_next_call():
    """Warmed up, then new ppb: the capture cannot build the planes it keeps, and
    each replay splits ppb; the eager call after it builds them."""
    import ecalj_amd

    rng = np.random.default_rng(4)
    nv, md, nm, nq = [40, 24], [50, 70], 4, 60
    flat = lambda: np.concatenate([rng.standard_normal((v, v, m)).ravel(order="F") for v, m in zip(nv, md)])
    h = ecalj_amd.Handle(0, "bf16x3")
    try:
        h.set_ppb(nv, md, flat())
        cm, cq = h.to_dev(crand(rng, sum(nv), nm)), h.to_dev(crand(rng, sum(nv), nq))
        out = h.array((sum(md), nm, nq), np.complex64)
        call = lambda: h.zmel_dev(cm, cq, out, nm=nm, nq=nq, ndima=sum(nv), zmelconjg=True)
        call()
        before = out.download()
        h.set_ppb(nv, md, flat())
        h.graph_begin()
        try:
            call()
        finally:
            gr = h.graph_end()
        got = []
        for _ in range(2):
            out.zero()
            gr.launch()
            h.sync()
            got.append(out.download())
        gr.close()
        call()
        want = out.download()
        assert not np.array_equal(want, before)
        assert np.array_equal(got[0], want) and np.array_equal(got[1], want)
    finally:
        h.close()


def test_planes_on_another_stream():
    import ecalj_amd

    rng = np.random.default_rng(5)
    nv, md, nm, nq = 200, 220, 3, 50
    h = ecalj_amd.Handle(0, "bf16x3")
    lib = ecalj_amd.lib()
    st = ctypes.c_void_p()
    try:
        ppb = rng.standard_normal((nv, nv, md))
        cm, cq = h.to_dev(crand(rng, nv, nm)), h.to_dev(crand(rng, nv, nq))
        out = h.array((md, nm, nq), np.complex64)
        call = lambda: h.zmel_dev(cm, cq, out, nm=nm, nq=nq, ndima=nv, zmelconjg=True)
        h.set_ppb([nv], [md], ppb)
        call()
        call()
        want = out.download()
        assert lib.hipStreamCreate(ctypes.byref(st)) == 0
        for _ in range(3):
            h.set_ppb([nv], [md], ppb)
            out.zero()
            h.sync()
            call()  # builds the planes on the handle's own stream
            h.sync()  # (the call's own scratch is of its stream)
            h.set_stream(st.value)
            out.zero()
            call()
            h.sync()
            assert np.array_equal(out.download(), want)
            h.set_stream(None)
    finally:
        h.close()
        if st.value:
            lib.hipStreamDestroy(st)
