"""The sizes of the Sigma_c mode form (ecalj_amd/csrc/moderule.hpp, compiled
here for the host with g++): the planes kept for the modes hold those of
physical weights, and the form is taken where it was measured faster."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

from ecalj_amd import synth

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("moderule") / "libmoderule.so")
    subprocess.run(["g++", "-O2", "-std=c++17", "-shared", "-fPIC", "-I", os.path.join(ROOT, "ecalj_amd", "csrc"),
                    os.path.join(ROOT, "tests", "host", "moderule_host.cpp"), "-o", so], check=True)
    return C.CDLL(so)


@pytest.fixture(scope="module")
def orc():
    import oracle

    oracle.build()
    return oracle


def pays(rule, form, n, nms, ntq, nf):
    nms = np.asarray(nms, np.int32)
    return rule.moderule_pays(int(form == "f64"), int(form == "bf16x3"), n, len(nms),
                              nms.ctypes.data_as(C.POINTER(C.c_int)), 1, ntq, nf + 1)


def rank(x, tol):
    """Steps of the pivoted Gram-Schmidt (sigmodes.hip) over the columns of x."""
    x = x / np.sqrt((x ** 2).sum(0))
    r = 0
    while r < len(x):
        r2 = (x ** 2).sum(0)
        j = r2.argmax()
        if not r2[j] > tol ** 2:
            break
        q = x[:, j] / np.sqrt(r2[j])
        x = x - q[:, None] * (q @ x)
        r += 1
    return max(r, 1)


@pytest.mark.parametrize("form", ["f64", "f32", "bf16x3"])
@pytest.mark.parametrize("nf", [7, 8, 10, 12, 16, 20, 23])
@pytest.mark.parametrize("nm,ntq", [(65, 8), (155, 18), (205, 30), (318, 36), (600, 34)])
def test_planes_hold_the_modes_of_physical_weights(rule, orc, form, nf, nm, ntq):
    t, w = np.polynomial.legendre.leggauss(nf)
    x, wx = 0.5 * (t + 1.0), 0.5 * w
    om = (1.0 - x) / x
    rng = np.random.default_rng(5)
    ek = np.concatenate([np.sort(rng.uniform(-12, 0, 5)), np.sort(rng.uniform(0.5, 60, nm - 5))]) / synth.RYDBERG_EV
    eq = np.sort(np.concatenate([rng.uniform(-11, 0, ntq // 2), rng.uniform(0.5, 12, ntq - ntq // 2)]))
    g = orc.wgtim(eq / synth.RYDBERG_EV, ek, 0.003, 1.0, x, wx, np.exp(-om ** 2)).reshape(nf + 1, -1, order="F")
    g = g / (1.0 + np.concatenate([[0.0], om]) ** 2)[:, None]  # times the norm of a W that decays
    bn, f64, bf3 = (128 if form == "bf16x3" else 64), int(form == "f64"), int(form == "bf16x3")
    cols = g.shape[1]
    tiles = -(-cols // bn)
    sorts = rule.moderule_sorts(tiles, bn)
    tp, total = -(-tiles // sorts), 0
    for t0 in range(0, tiles, tp):  # as sig_modes: sorted by the weight at the highest frequency, groups of whole tiles
        part = g[:, t0 * bn:min(cols, (t0 + tp) * bn)]
        part = part[:, np.argsort(np.abs(part[-1]))]
        gt = rule.moderule_group_tiles(-(-part.shape[1] // bn), sorts, f64, bf3, nf + 1)
        for c in range(0, part.shape[1], gt * bn):
            total += rank(part[:, c:c + gt * bn], 2.0 ** -51 if f64 else 2.0 ** -25)
    print(form, nf, cols, "modes", total, "planes", rule.moderule_planes(f64, nf + 1))
    assert total <= rule.moderule_planes(f64, nf + 1)


# (form, n, middle states per k, end states, frequencies - 1), us of the modes, us of the plain form (MI355X)
MEASURED = [
    ("f64", 300, [155] * 4, 10, 8, 2019, 1459), ("f64", 300, [205], 30, 12, 2270, 1712),
    ("f64", 600, [155] * 2, 10, 8, 2948, 2315), ("f64", 60, [605] * 4, 32, 20, 3152, 1869),
    ("f64", 300, [318], 36, 7, 3067, 2470), ("f64", 600, [159] * 8, 18, 16, 14400, 25450),
    ("f32", 300, [605], 32, 7, 2296, 1937), ("f32", 60, [605] * 8, 32, 8, 1397, 1098),
    ("f32", 300, [205] * 3, 20, 23, 1424, 3020), ("f32", 128, [305] * 8, 36, 20, 1685, 3114),
    ("bf16x3", 200, [605] * 4, 32, 8, 1073, 764), ("bf16x3", 450, [605], 32, 7, 1068, 752),
    ("bf16x3", 600, [65] * 8, 8, 16, 951, 752), ("bf16x3", 1200, [155], 18, 7, 849, 654),
    ("bf16x3", 600, [159] * 16, 18, 16, 3380, 5077), ("bf16x3", 1200, [318] * 12, 36, 20, 28500, 66570),
    ("bf16x3", 1080, [424, 158, 300, 250, 200, 350, 400, 180, 280], 16, 20, 10150, 20570),
]


@pytest.mark.parametrize("form,n,nms,ntq,nf,modes,plain", MEASURED)
def test_the_faster_form_is_taken(rule, form, n, nms, ntq, nf, modes, plain):
    assert bool(pays(rule, form, n, nms, ntq, nf)) == (modes < plain)


def test_edges(rule):
    assert not pays(rule, "bf16x3", 1200, [0, 0], 36, 20)          # no columns
    assert not pays(rule, "f64", 100, [3], 2, 20)                  # too little work to be measured
    assert pays(rule, "bf16x3", 1200, [0, 318, 0, 318], 36, 20)    # empty k between
    assert not pays(rule, "bf16x3", 600, [3000], 40, 20)           # eight sorts: more modes than planes
