"""Timed calls of the chi0 -> W -> Sigma_c path through its public entry points.

The cases are the pieces of one QSGW q-point as a driver calls them, on
device-resident data: zmel, the chi0 bins with their Hilbert transform, the W
build on the imaginary and the real axis, the Sigma_c contraction (uniform
and uneven band windows), the training step of the learned chi0 tail, and a
whole small q-point.  Sizes are those of the workloads of
``ecalj_amd.synth.CONFIGS`` (C1 .. C5) with the number of k-points cut to
what one call needs to fill the card; drawn cases spread over the ranges
between the smallest and the largest of them.

``prepare`` makes inputs from the seed alone, with the magnitudes the path
meets: cell-normalised zmel, screened W that decays with the frequency,
band energies in the ranges of ``ecalj_amd.synth``.  ``exact`` evaluates the
same quantities in complex128 with plain torch.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import ecalj_amd
from ecalj_amd import synth

RY = synth.RYDBERG_EV
OMEGA_CELL = 10.68 ** 3 / 4.0
C16, C8 = torch.complex128, torch.complex64


# ---------------------------------------------------------------- cases
def listed():
    return [
        # Sigma_c of a small (C1-like) cell: few hundred columns, launches count
        dict(name="sigma_small_bf16x3", kind="sigma", prec="bf16x3", ni=200, no=4, nu=60, ntq=8, nf=12, nk=8),
        # Sigma_c at the C2 shape, the mixed form
        dict(name="sigma_c2_bf16x3", kind="sigma", prec="bf16x3", ni=600, no=9, nu=150, ntq=18, nf=16, nk=16),
        # Sigma_c at the C3 shape, the mixed form: the largest share of the headline workload
        dict(name="sigma_c3_bf16x3", kind="sigma", prec="bf16x3", ni=1200, no=18, nu=300, ntq=36, nf=20, nk=12),
        # Sigma_c at the C2 shape in FP64, the form every result is judged by
        dict(name="sigma_c2_f64", kind="sigma", prec="f64", ni=600, no=9, nu=150, ntq=18, nf=16, nk=8),
        # Sigma_c over k-points with their own band windows (C4-like), grouped call
        dict(name="sigma_uneven_bf16x3", kind="uneven", prec="bf16x3", ni=1080, ntq=16, nf=20, nk=9, nm_lo=158,
             nm_hi=424, wseed=4),
        # zmel of chi0 (occupied x unoccupied, conjugated) at the C3 shape
        dict(name="zmel_chi0_c3_bf16x3", kind="zmel", prec="bf16x3", ni=1200, nb=320, nm=18, nq=300, nk=8, natom=1,
             conj=True, shared=False),
        # zmel of Sigma_c (middle x end states, end states shared by all k) at the C2 shape, FP64
        dict(name="zmel_sigma_c2_f64", kind="zmel", prec="f64", ni=600, nb=180, nm=159, nq=18, nk=16, natom=1,
             conj=False, shared=True),
        # chi0(i nu): histogram bins and Hilbert transform at the C2 shape
        dict(name="chi0_c2_bf16x3", kind="chi0", prec="bf16x3", ni=600, no=9, nu=150, nk=32, nf=16),
        # W_c on the imaginary axis at the C3 shape
        dict(name="w_imag_c3_bf16x3", kind="wbuild", prec="bf16x3", axis="imag", ni=1200, nw=21),
        # W_c on the real axis (pivoted inversion) at the C2 shape, FP64
        dict(name="w_real_c2_f64", kind="wbuild", prec="f64", axis="real", ni=600, nw=32),
        # a whole small q-point (the C1 shape): the latency of a full step
        dict(name="qpoint_c1_bf16x3", kind="qpoint", prec="bf16x3", nk=8, nb=100, no=4, nu=60, ni=200, nf=12),
        # one training step of the learned chi0 tail (forward, backward, Adam)
        dict(name="mlp_train", kind="mlp", batch=256, width=256, nin=21),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["sigma", "sigma", "uneven", "zmel", "chi0", "wbuild", "qpoint", "mlp"])
    prec = rng.choice(["bf16x3", "bf16x3", "f64", "f32"])
    if kind in ("sigma", "uneven"):
        ni, nf = _log(rng, 60, 1200), rng.choice([6, 10, 12, 16, 20])
        ntq = _log(rng, 3, 36)
        if prec != "bf16x3":
            ni = min(ni, 600)
        if kind == "uneven":
            lo = _log(rng, 20, 150)
            return dict(kind=kind, prec=prec, ni=ni, ntq=min(ntq, 16), nf=nf, nk=rng.randint(2, 6), nm_lo=lo,
                        nm_hi=2 * lo + rng.randint(0, 60), wseed=rng.randint(1, 1000))
        return dict(kind=kind, prec=prec, ni=ni, no=rng.randint(2, 18), nu=_log(rng, 20, 300), ntq=ntq, nf=nf,
                    nk=rng.randint(1, 8))
    if kind == "zmel":
        natom = rng.choice([1, 1, 2])
        nv, md = _log(rng, 12, 320 // natom), _log(rng, 30, 1200 // natom)
        return dict(kind=kind, prec=prec, ni=natom * md, nb=natom * nv, nm=rng.randint(2, 18), nq=_log(rng, 10, 300),
                    nk=rng.randint(1, 6), natom=natom, conj=rng.random() < 0.5, shared=rng.random() < 0.3)
    if kind == "chi0":
        return dict(kind=kind, prec=prec, ni=_log(rng, 40, 600), no=rng.randint(2, 9), nu=_log(rng, 13, 150),
                    nk=rng.randint(1, 16), nf=rng.choice([6, 10, 12, 16, 20]))
    if kind == "wbuild":
        axis = rng.choice(["imag", "real"])
        return dict(kind=kind, prec=prec, axis=axis, ni=_log(rng, 40, 1200 if axis == "imag" else 600),
                    nw=rng.randint(1, 21))
    if kind == "qpoint":
        no, nu = rng.randint(2, 4), rng.randint(5, 60)
        return dict(kind=kind, prec=prec, nk=rng.randint(2, 8), nb=no + nu + rng.randint(0, 36), no=no, nu=nu,
                    ni=_log(rng, 16, 200), nf=rng.choice([6, 10, 12]))
    return dict(kind="mlp", batch=_log(rng, 64, 2048), width=rng.choice([64, 128, 256]), nin=rng.randint(7, 33))


# ---------------------------------------------------------------- inputs
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 7919 + 17)


def _crand(g, *shape, dtype=C16):
    return torch.randn(*shape, generator=g, device="cuda", dtype=dtype) * math.sqrt(2.0)


def _store(prec):
    return (C16, np.complex128) if prec == "f64" else (C8, np.complex64)


class _Shared:
    """Array interface of a library buffer, which it keeps alive."""

    TYPES = {"complex128": "<c16", "complex64": "<c8", "float64": "<f8", "float32": "<f4"}

    def __init__(self, dev):
        self.dev = dev
        self.__cuda_array_interface__ = {"shape": tuple(reversed(dev.shape)), "typestr": self.TYPES[dev.dtype.name],
                                         "data": (dev.ptr, False), "version": 2, "strides": None}


def _tensor(dev):
    """The library buffer as a torch tensor (Fortran order: axes reversed), no copy."""
    return torch.as_tensor(_Shared(dev), device="cuda")


def _energies(rng, no, nu, nk):
    """Band energies (eV) of nk k-points, (no + nu) x nk: occupied in [-12, 0], unoccupied in [0.5, 60]."""
    e = [np.concatenate([np.sort(rng.uniform(-12.0, 0.0, no)), np.sort(rng.uniform(0.5, 60.0, nu))])
         for _ in range(nk)]
    return np.asfortranarray(np.stack(e, axis=1))


def _freqs(nf):
    t, w = np.polynomial.legendre.leggauss(nf)
    x, wx = 0.5 * (t + 1.0), 0.5 * w
    om = (1.0 - x) / x
    return x, wx, om, np.exp(-om ** 2)


def _screened(g, ni, nf, nk):
    """W_c(i nu) of nk k-points, (nk, nf+1, ni, ni): Hermitian, negative, decaying with nu."""
    _, _, om, _ = _freqs(nf)
    nu = np.concatenate([[0.0], om])
    a = _crand(g, ni, ni) / math.sqrt(2.0 * ni)
    c = 4.0 * torch.rand(ni, generator=g, device="cuda", dtype=torch.float64) ** 2 + 0.05
    w0 = 0.3 + 2.0 * torch.rand(ni, generator=g, device="cuda", dtype=torch.float64)
    ph = torch.rand(nk, ni, generator=g, device="cuda", dtype=torch.float64) * (2.0 * math.pi)
    ph = torch.polar(torch.ones_like(ph), ph)
    out = torch.empty(nk, nf + 1, ni, ni, device="cuda", dtype=C16)
    for v in range(nf + 1):
        d = c / (1.0 + (nu[v] / w0) ** 2)
        m = -((a * d) @ a.conj().T)
        m = 0.5 * (m + m.conj().T)
        for k in range(nk):
            # torch (J, I) row-major is Fortran W(I, J)
            out[k, v] = ph[k][None, :] * m * ph[k].conj()[:, None]
    return out


def _upload(h, a):
    return h.to_dev(np.ascontiguousarray(a, np.float64))


def _windows(case):
    if case["kind"] == "sigma":
        return [case["no"] + case["nu"]] * case["nk"]
    r = np.random.default_rng(case["wseed"])
    return [int(x) for x in r.integers(case["nm_lo"], case["nm_hi"] + 1, case["nk"])]


def _sigma_inputs(case, seed):
    g = _gen(seed)
    rng = np.random.default_rng(int(seed) + 5)
    ni, nf, nk, ntq = case["ni"], case["nf"], case["nk"], case["ntq"]
    nms = _windows(case)
    no = case.get("no", 16)
    w = _screened(g, ni, nf, nk)
    z = _crand(g, ni * ntq * sum(nms), dtype=_store(case["prec"])[0]) / math.sqrt(2.0 * ni * OMEGA_CELL)
    ekc = [_energies(rng, min(no, nm - 1), nm - min(no, nm - 1), 1)[:, 0] / RY for nm in nms]
    lo = rng.uniform(-11.0, 0.0, ntq // 2)
    hi = rng.uniform(0.5, 12.0, ntq - ntq // 2)
    omega = np.sort(np.concatenate([lo, hi])) / RY
    return nms, w, z, ekc, omega


def _wbuild_inputs(case, seed):
    """chi (nw, ni, ni) and the Coulomb basis: epsilon's eigenvalues between 1 and about 10."""
    g = _gen(seed)
    ni, nw = case["ni"], case["nw"]
    b = _crand(g, ni, ni) / math.sqrt(2.0 * ni)
    bb = -0.02 * (b @ b.conj().T)
    bb = 0.5 * (bb + bb.conj().T)
    x = torch.linspace(0.0, 2.0, nw, dtype=torch.float64, device="cuda")
    if case["axis"] == "imag":
        chi = bb[None] / (1.0 + x[:, None, None] ** 2)
    else:
        c = _crand(g, ni, ni) / math.sqrt(2.0 * ni)
        cc = 0.01 * (c @ c.conj().T)
        chi = bb[None] * (1.0 - 0.6 * x[:, None, None]) + 1j * cc[None] * (0.5 + x[:, None, None])
    q = torch.linalg.qr(_crand(g, ni, ni))[0]
    gv = synth.gvectors(ni)
    qg2 = (((np.array([0.1, 0.2, 0.3])[None, :] + gv) * (2.0 * math.pi / 10.68)) ** 2).sum(1)
    return chi.contiguous(), 4.0 * math.pi / qg2, q.contiguous()


def _zmel_inputs(case, seed):
    g = _gen(seed)
    na = case["natom"]
    nv, md = case["nb"] // na, case["ni"] // na
    ppb = torch.randn(na, md, nv, nv, generator=g, device="cuda", dtype=torch.float64)
    ppb *= na / math.sqrt(case["ni"] * OMEGA_CELL)
    cm = _crand(g, case["nk"], case["nm"], case["nb"]) / math.sqrt(2.0 * case["nb"])
    cq = _crand(g, 1 if case["shared"] else case["nk"], case["nq"], case["nb"]) / math.sqrt(2.0 * case["nb"])
    ph = np.exp(2j * math.pi * np.random.default_rng(int(seed) + 3).random(na))
    return ppb, cm, cq, ph


def _chi0_point(case, seed):
    """Energies and weights of a q-point without its eigenvectors (zmel is an input here)."""
    rng = np.random.default_rng(int(seed) + 11)
    cfg = synth.Config("case", nk=case["nk"], nb=case["no"] + case["nu"], no=case["no"], nu=case["nu"], ni=case["ni"],
                       nf=case["nf"], seed=1)
    e_k, e_kq = (_energies(rng, cfg.no, cfg.nu, cfg.nk) for _ in range(2))
    none = np.zeros(0)
    return synth.QPoint(cfg, e_k, e_kq, none, none, none, none, none, none, none, none, none,
                        np.full(cfg.nk, 1.0 / cfg.nk))


def _chi0_inputs(case, seed):
    qp = _chi0_point(case, seed)
    fr = synth.frhis(qp)
    ix = synth.x0kf_index(synth.pair_weights(qp, fr))
    z = _crand(_gen(seed), case["nk"], case["nu"], case["no"], case["ni"], dtype=_store(case["prec"])[0])
    z /= math.sqrt(2.0 * case["ni"] * OMEGA_CELL)
    return fr, ix, z


def _mlp_dims(case):
    return [case["nin"], case["width"], case["width"], case["nin"]]


def _mlp_inputs(case, seed):
    g = _gen(seed)
    dims = _mlp_dims(case)
    parts = []
    for i, o in zip(dims[:-1], dims[1:]):
        parts.append(torch.randn(o * i, generator=g, device="cuda") / math.sqrt(i))
        parts.append(0.05 * torch.randn(o, generator=g, device="cuda"))
    x = torch.randn(case["batch"], dims[0], generator=g, device="cuda")
    y = torch.randn(case["batch"], dims[-1], generator=g, device="cuda")
    p = torch.cat(parts)
    m = 1e-3 * torch.randn(p.numel(), generator=g, device="cuda")
    v = 1e-5 * (0.1 + torch.rand(p.numel(), generator=g, device="cuda"))
    return p, x, y, m, v


def _qpoint(case, seed):
    cfg = synth.Config("case", nk=case["nk"], nb=case["nb"], no=case["no"], nu=case["nu"], ni=case["ni"],
                       nf=case["nf"], seed=int(seed) + 1, alat=10.26)
    return synth.make_qpoint(cfg)


# ---------------------------------------------------------------- prepare / run
def prepare(case, seed):
    kind = case["kind"]
    prec = case.get("prec", "f32")
    if kind == "qpoint":
        from ecalj_amd.qsgw import QPointGPU

        q = QPointGPU(_qpoint(case, seed), prec)
        q.chi0()
        q.wbuild()
        q.make_wk()  # W_c of the internal k-points, a driver's input of Sigma_c
        return dict(case=case, q=q)
    h = ecalj_amd.Handle(0, prec)
    s = dict(case=case, h=h)
    st = _store(prec)[1]
    if kind in ("sigma", "uneven"):
        nms, w, z, ekc, omega = _sigma_inputs(case, seed)
        nk, nw1 = case["nk"], case["nf"] + 1
        x, wx, _, expa = _freqs(case["nf"])
        s.update(nms=nms, w=w, z=z, omega=_upload(h, np.tile(omega, nk)), ekc=_upload(h, np.concatenate(ekc)),
                 wk=_upload(h, np.full(nk, 1.0 / nk)), x=_upload(h, x), wx=_upload(h, wx), expa=_upload(h, expa),
                 wgt=h.array(nw1 * case["ntq"] * sum(nms), np.float64), zsec=h.array((case["ntq"], case["ntq"])))
    elif kind == "zmel":
        ppb, cm, cq, ph = _zmel_inputs(case, seed)
        na = case["natom"]
        h.set_ppb([case["nb"] // na] * na, [case["ni"] // na] * na, ppb.reshape(-1).cpu().numpy())
        s.update(cm=cm, cq=cq, ph=ph, out=h.array((case["ni"], case["nm"], case["nq"], case["nk"]), st))
    elif kind == "chi0":
        fr, ix, z = _chi0_inputs(case, seed)
        ni = case["ni"]
        _, _, om, _ = _freqs(case["nf"])
        s.update(fr=fr, ix=ix, z=z, nu=np.concatenate([[0.0], om]), rcxq=h.array((ni, ni, len(fr)), st),
                 chi=h.array((ni, ni, case["nf"] + 1)))
    elif kind == "wbuild":
        chi, vcoud, q = _wbuild_inputs(case, seed)
        h.set_coulomb(vcoud, q.T.cpu().numpy())  # Fortran zcousq(I, mu) = q[mu, I]
        s.update(chi=chi, wc=h.array((case["ni"], case["ni"], case["nw"])))
    else:
        p, x, y, m, v = _mlp_inputs(case, seed)
        s.update(p0=p, p=p.clone(), x=x, y=y, m0=m, m=m.clone(), v0=v, v=v.clone(), grad=torch.empty_like(p),
                 loss=torch.empty(1, device="cuda"))
    torch.cuda.synchronize()
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "qpoint":
        q = s["q"]
        q.step()
        return dict(chi=_tensor(q.chi), wc=_tensor(q.wc), zsec=_tensor(q.zsec))
    h = s["h"]
    if kind in ("sigma", "uneven"):
        nk, nw1, ntq, ni = case["nk"], case["nf"] + 1, case["ntq"], case["ni"]
        z, w = s["z"].data_ptr(), s["w"].data_ptr()
        tab = (s["x"], s["wx"], s["expa"])
        if kind == "sigma":
            nm = s["nms"][0]
            h.sigc_weights_dev(nk, case["nf"], nm, ntq, s["omega"], s["ekc"], 0.003, 1.0, s["wk"], *tab, s["wgt"])
            s["zsec"].zero()
            h.sigc_dev(nk, z, ni, nm, ntq, case["nf"], w, s["wgt"], s["zsec"])
        else:
            ofs = band = 0
            for k, nm in enumerate(s["nms"]):
                h.sigc_weights_dev(1, case["nf"], nm, ntq, s["omega"], s["ekc"].ptr + 8 * band, 0.003, 1.0,
                                   s["wk"].ptr + 8 * k, *tab, s["wgt"].ptr + 8 * ofs)
                ofs += nw1 * nm * ntq
                band += nm
            s["zsec"].zero()
            h.sigc_grouped_dev(s["nms"], z, ni, ntq, case["nf"], w, s["wgt"], s["zsec"])
        return _tensor(s["zsec"])
    if kind == "zmel":
        h.zmel_dev(s["cm"].data_ptr(), s["cq"].data_ptr(), s["out"], nm=case["nm"], nq=case["nq"], ndima=case["nb"],
                   nbatch=case["nk"], phase=s["ph"], zmelconjg=case["conj"], cphiq_stride=0 if case["shared"] else None)
        return _tensor(s["out"])
    if kind == "chi0":
        ni, nwhis, ix = case["ni"], len(s["fr"]) - 1, s["ix"]
        s["rcxq"].zero()
        h.x0gemm_batched_dev(s["rcxq"], ni, nwhis, case["nk"], ix.nkmin, ix.nkmax, s["z"].data_ptr(),
                             ni * case["no"] * case["nu"], ni, case["nu"], ix)
        h.dpsion_imag_dev(s["rcxq"], ni, ni, nwhis, s["fr"], s["nu"], s["chi"])
        return dict(rcxq=_tensor(s["rcxq"]), chi=_tensor(s["chi"]))
    if kind == "wbuild":
        f = h.wc_build_dev if case["axis"] == "imag" else h.wc_build_real_dev
        f(s["chi"].data_ptr(), s["wc"], case["ni"], case["nw"])
        return _tensor(s["wc"])
    dims, n = _mlp_dims(case), s["p"].numel()
    for a in ("p", "m", "v"):  # the same step on every pass
        h.memcpy_d2d(s[a].data_ptr(), s[a + "0"].data_ptr(), 4 * n)
    h.mlp_grad_dev(dims, s["p"].data_ptr(), s["x"].data_ptr(), s["y"].data_ptr(), case["batch"],
                   s["grad"].data_ptr(), s["loss"].data_ptr())
    h.mlp_adam_dev(n, s["p"].data_ptr(), s["grad"].data_ptr(), s["m"].data_ptr(), s["v"].data_ptr(), 3, 1e-3)
    return dict(grad=s["grad"], loss=s["loss"], p=s["p"], m=s["m"], v=s["v"])


# ---------------------------------------------------------------- work and tolerances
def work(case):
    kind = case["kind"]
    es = 16 if case.get("prec") == "f64" else 8
    if kind in ("sigma", "uneven"):
        cols = sum(_windows(case)) * case["ntq"]
        ni, nw1 = case["ni"], case["nf"] + 1
        # W is used through its upper triangle; one product of the Hermitian W with zmel per frequency
        return dict(bytes=8.0 * ni * ni * nw1 * case["nk"] + es * ni * cols,
                    flops=8.0 * ni * ni * nw1 * cols + 8.0 * ni * case["ntq"] * cols)
    if kind == "zmel":
        na, nb, ni = case["natom"], case["nb"], case["ni"]
        nm, nq, nk = case["nm"], case["nq"], case["nk"]
        small = min(nm * nk, nq * (1 if case["shared"] else nk))
        return dict(bytes=8.0 * nb * nb * ni / na ** 2 + 16.0 * nb * (nm + nq) * nk + es * ni * nm * nq * nk,
                    flops=4.0 * nb * nb * ni * small / na ** 2 + 8.0 * ni * nm * nq * nk * nb / na)
    if kind == "chi0":
        ni, pairs = case["ni"], case["no"] * case["nu"] * case["nk"]
        bins = _bins(case)
        return dict(bytes=es * ni * pairs + es * ni * ni * bins + 16.0 * ni * ni * (case["nf"] + 1),
                    flops=4.0 * ni * ni * pairs * 2.3 + 4.0 * ni * ni * bins * (case["nf"] + 1))
    if kind == "wbuild":
        ni, nw = case["ni"], case["nw"]
        return dict(bytes=32.0 * ni * ni * nw + 16.0 * ni * ni, flops=nw * 5 * 8.0 * ni ** 3)
    if kind == "qpoint":
        ni, nk, pairs = case["ni"], case["nk"], case["no"] * case["nu"] * case["nk"]
        nw1, ntq, nbt = case["nf"] + 1, 2 * case["no"], case["no"] + case["nu"]
        return dict(bytes=16.0 * ni * ni * nw1 * (nk + 2) + 8.0 * case["nb"] ** 2 * ni,
                    flops=8.0 * ni * ni * nw1 * nbt * ntq * nk + 8.0 * ni * ni * pairs + 40.0 * nw1 * ni ** 3)
    d, b = _mlp_dims(case), case["batch"]
    n = sum(i * o + o for i, o in zip(d[:-1], d[1:]))
    return dict(bytes=4.0 * (10 * n + 2 * b * case["nin"]), flops=6.0 * b * n)


def _bins(case):
    # bins of the mesh: bb (exp(aa i) - 1) up to about 73 eV (S/m_freq.f90:95-108)
    return int(math.log(1.0 + 0.03 * 2.9 / 1e-5 * 0.55) / 0.03)


def tolerance(case):
    """About four times the distance from the 64-bit result over the declared ranges (Sigma_c averages
    the roundings of many columns; a small one averages fewer)."""
    kind, prec = case["kind"], case.get("prec")
    if kind == "mlp":
        return {"rel": 3e-6}
    if kind in ("sigma", "uneven"):
        return {"rel": {"f64": 5e-14, "f32": 2e-6, "bf16x3": 5e-6}[prec]}
    if kind == "qpoint":
        return {"rel": {"f64": 1e-12, "f32": 1e-5, "bf16x3": 4e-5}[prec]}
    if kind == "wbuild":
        return {"rel": {"f64": 5e-13, "f32": 4e-6, "bf16x3": 2.5e-5}[prec]}
    return {"rel": {"f64": 1e-13, "f32": 2e-6, "bf16x3": 2.5e-5}[prec]}


# ---------------------------------------------------------------- 64-bit results
def _weights(omega, ekc, nf, wk):
    """Imaginary-axis weights (S/m_sxcf_gemm.f90:432-458), (ntq, nm, nf+1)."""
    x, wx, om, expa = (torch.as_tensor(a, device="cuda") for a in _freqs(nf))
    we = 0.5 * (torch.as_tensor(omega, device="cuda")[:, None] - torch.as_tensor(ekc, device="cuda")[None, :])
    sgn = torch.where(torch.signbit(we), -1.0, 1.0)
    sig2 = 2.0 * (0.5 * 0.003) ** 2
    omd2w = om ** 2 + we[..., None] ** 2
    r = omd2w / sig2
    series = sum((-1.0) ** j * r ** j / math.factorial(j + 1) for j in range(6)) / sig2
    cons = torch.where(r > 5e-3, (1.0 - torch.exp(-r)) / omd2w, series)
    wi = -we[..., None] * cons * wx / x ** 2 / math.pi
    aw = we.abs()
    w0 = we * (cons * expa * wx / x ** 2).sum(-1) / math.pi
    w0 = w0 + sgn * 0.5 * torch.exp(aw ** 2) * (torch.special.erfc(torch.sqrt(aw ** 2 + we ** 2 / sig2))
                                                - torch.special.erfc(aw))
    return wk * torch.cat([w0[..., None], wi], dim=-1)


def _sigma_exact(w, z, g, zsec):
    """zsec (m', m) += the contraction of one k: w (nw1, J, I), z (ntq, nm, ni), g (ntq, nm, nw1)."""
    ntq, nm, ni = z.shape
    zc = z.to(C16).reshape(ntq * nm, ni)
    cz = torch.zeros_like(zc)
    for v in range(w.shape[0]):
        u = torch.triu(w[v].T)  # W(I, J), I <= J: kept through its upper triangle
        full = u + torch.triu(w[v].T, 1).conj().T
        cz += (zc * g.reshape(ntq * nm, -1)[:, v, None]) @ full.conj()
    # czmelwc = sum W^H (g zmel): row form (g zmel)^T conj(W)
    a, b = cz.reshape(ntq, nm * ni), zc.reshape(ntq, nm * ni)
    zsec += (a.conj() @ b.T).T
    d = torch.diagonal(zsec)
    d.copy_(torch.complex(d.real, torch.clamp(d.imag, max=0.0)))
    return zsec


def _zmel_exact(case, ppb, cm, cq, ph):
    na, md = case["natom"], case["ni"] // case["natom"]
    nv, nk, nm, nq = case["nb"] // na, cm.shape[0], cm.shape[1], cq.shape[1]
    out = torch.zeros(nk, nq, nm, case["ni"], device="cuda", dtype=C16)
    for a in range(na):
        p = ppb[a].to(C16).reshape(md * nv, nv)  # (I, a-side), b-side contiguous
        for k in range(nk):
            q = cq[0 if case["shared"] else k][:, a * nv:(a + 1) * nv]
            t = (p @ q.T.contiguous()).reshape(md, nv, nq).permute(0, 2, 1).reshape(md * nq, nv)
            r = t @ cm[k][:, a * nv:(a + 1) * nv].conj().T.contiguous()
            out[k, :, :, a * md:(a + 1) * md] = complex(ph[a]) * r.reshape(md, nq, nm).permute(1, 2, 0)
    return out.conj().resolve_conj() if case["conj"] else out


def _hilbert(fr, nu):
    """imatt (S/dpsion5.f90:84-129 with hilbertmat, S/hilbertmat.f90:14-79) times -1/(R-L), (nu, bin)."""
    n = len(fr) - 1
    left, right = fr[:-1], fr[1:]
    c = 0.5 * (left + right)
    lo = np.concatenate([-right[::-1], [0.0], left])
    hi = np.concatenate([-left[::-1], [0.0], right])
    ce = np.concatenate([-c[::-1], [0.0], c])
    out = np.zeros((len(nu), n))

    def moments(z, a, b):
        da, db = z - a, z - b
        if abs(da) <= 1e-8 or abs(db) <= 1e-8:
            return 0.0, 0.0
        f = np.log(db / da)
        return z * f + (b - a), f

    for i, v in enumerate(nu):
        z = 1j * v + 1e-13j
        m = np.zeros(2 * n + 1, complex)
        for iw in range(-n, n + 1):
            if iw == 0:
                continue
            j = iw + n
            prev = lo[j] if iw == -n else (0.0 if iw == 1 else ce[j - 1])
            fm, fn = moments(z, lo[j], ce[j])
            m[j] += (fm - fn * prev) / (ce[j] - prev)
            if iw not in (-n, 1):
                m[j - 1] += (-fm + fn * ce[j]) / (ce[j] - prev)
            nxt = hi[j] if iw == n else (0.0 if iw == -1 else ce[j + 1])
            fm, fn = moments(z, ce[j], hi[j])
            m[j] += (-fm + fn * nxt) / (nxt - ce[j])
            if iw not in (n, -1):
                m[j + 1] += (fm - fn * ce[j]) / (nxt - ce[j])
        out[i] = np.real(m[n + 1:] - m[n - 1::-1]) / math.pi
    return -out / (right - left)


def _chi0_exact(ni, fr, ix, zk, nu):
    """rcxq (bin, J, I) and chi (nu, J, I); zk(k): (m, n, I) as stored."""
    nwhis = len(fr) - 1
    rc = torch.zeros(nwhis + 1, ni, ni, device="cuda", dtype=C16)
    nh = ix.iwend - ix.iwini + 1
    for k in range(len(ix.nkmin)):
        s = slice(int(ix.icounkmin[k]) - 1, int(ix.icounkmax[k]))
        z = zk(k).to(C16)
        pair = np.repeat(np.arange(s.start, s.stop), nh[s])
        first = int(ix.icouini[s.start]) - 1
        wt = ix.whwc[first:first + len(pair)]
        b = ix.iwini[pair] + np.arange(len(pair)) - np.repeat(ix.icouini[s] - 1 - first, nh[s])
        n, m = ix.itc[pair] - int(ix.nkmin[k]), ix.itpc[pair] - 1
        order = np.argsort(b, kind="stable")
        edges = np.searchsorted(b[order], np.arange(1, nwhis + 2))
        col = torch.as_tensor(m[order] * z.shape[1] + n[order], device="cuda")
        wt = torch.as_tensor(wt[order], device="cuda")
        zf = z.reshape(-1, ni)
        for iw in range(nwhis):
            e = slice(int(edges[iw]), int(edges[iw + 1]))
            if e.stop > e.start:
                x = zf[col[e]]
                rc[iw + 1] += (x * wt[e, None]).T @ x.conj()
    t = torch.as_tensor(_hilbert(fr, nu), device="cuda").to(C16)
    chi = (t @ rc[1:].reshape(nwhis, -1)).reshape(len(nu), ni, ni)
    return rc, chi


def _w_exact(chi, vcoud, zc, nspin=1):
    """W_c (nw, J, I) in the M basis; chi (nw, J, I); zc[mu, I] = zcousq(I, mu)."""
    v = torch.as_tensor(np.sqrt(vcoud), device="cuda")
    q = zc.T.contiguous()
    out = torch.empty_like(chi)
    eye = np.eye(len(vcoud))
    for i in range(chi.shape[0]):
        x = q.conj().T @ ((2.0 if nspin == 1 else 1.0) * chi[i].T) @ q
        eps = eye - (v[:, None] * x * v[None, :]).cpu().numpy()
        w = torch.as_tensor(np.linalg.inv(eps) - eye, device="cuda")
        out[i] = (q @ (v[:, None] * w * v[None, :]) @ q.conj().T).T
    return out


def exact(case, seed):
    kind = case["kind"]
    if kind in ("sigma", "uneven"):
        nms, w, z, ekc, omega = _sigma_inputs(case, seed)
        ntq, ni = case["ntq"], case["ni"]
        zsec = torch.zeros(ntq, ntq, device="cuda", dtype=C16)
        ofs = 0
        for k, nm in enumerate(nms):
            zk = z[ofs:ofs + ni * nm * ntq].reshape(ntq, nm, ni)
            ofs += ni * nm * ntq
            zsec = _sigma_exact(w[k], zk, _weights(omega, ekc[k], case["nf"], 1.0 / case["nk"]), zsec)
        return zsec
    if kind == "zmel":
        return _zmel_exact(case, *_zmel_inputs(case, seed))
    if kind == "chi0":
        fr, ix, z = _chi0_inputs(case, seed)
        nu = np.concatenate([[0.0], _freqs(case["nf"])[2]])
        rc, chi = _chi0_exact(case["ni"], fr, ix, lambda k: z[k], nu)
        return dict(rcxq=rc, chi=chi)
    if kind == "wbuild":
        return _w_exact(*_wbuild_inputs(case, seed))
    if kind == "qpoint":
        return _qpoint_exact(case, seed)
    p, x, y, m, v = (t.double() for t in _mlp_inputs(case, seed))
    p.requires_grad_(True)
    dims, o, hcur = _mlp_dims(case), 0, x
    for i, (a, b) in enumerate(zip(dims[:-1], dims[1:])):
        wt, bias = p[o:o + a * b].reshape(b, a), p[o + a * b:o + a * b + b]
        o += a * b + b
        hcur = hcur @ wt.T + bias
        if i < len(dims) - 2:
            hcur = torch.nn.functional.silu(hcur)
    loss = ((hcur - y) ** 2).mean()
    grad = torch.autograd.grad(loss, p)[0]
    m1, v1 = 0.9 * m + 0.1 * grad, 0.999 * v + 0.001 * grad ** 2
    step = (m1 / (1.0 - 0.9 ** 3)) / (torch.sqrt(v1 / (1.0 - 0.999 ** 3)) + 1e-8)
    return dict(grad=grad, loss=loss.detach().reshape(1), p=p.detach() - 1e-3 * step, m=m1, v=v1)


def _qpoint_exact(case, seed):
    qp = _qpoint(case, seed)
    cfg = qp.cfg
    t = lambda a: torch.as_tensor(np.ascontiguousarray(a), device="cuda")  # noqa: E731
    one = dict(natom=1, ni=cfg.ni, nb=cfg.nb, shared=False)
    ppb = t(np.ascontiguousarray(qp.ppb.T))[None]  # (1, I, a, b)
    ones = np.ones(1)
    fr = synth.frhis(qp)
    ix = synth.x0kf_index(synth.pair_weights(qp, fr))
    nu = np.concatenate([[0.0], _freqs(cfg.nf)[2]])
    no, nbt, ntq = cfg.no, cfg.nbt, cfg.nq

    def z_chi(k):
        return _zmel_exact(dict(one, conj=True), ppb, t(qp.c_k[:, :no, k].T)[None], t(qp.c_kq[:, no:, k].T)[None],
                           ones)[0]

    _, chi = _chi0_exact(cfg.ni, fr, ix, z_chi, nu)
    wc = _w_exact(chi, qp.vcoud, t(qp.zcousq.T))
    ph = t(synth.wc_phases(cfg))
    zsec = torch.zeros(ntq, ntq, device="cuda", dtype=C16)
    for k in range(cfg.nk):
        wk = ph[:, k][None, None, :] * wc * ph[:, k].conj()[None, :, None]
        z = _zmel_exact(dict(one, conj=False), ppb, t(qp.c_qmk[:, :, k].T)[None], t(qp.c_q[:, :ntq].T)[None], ones)[0]
        g = _weights(qp.e_q[:ntq] / RY, qp.e_qmk[:nbt, k] / RY, cfg.nf, float(qp.wk[k]))
        zsec = _sigma_exact(wk, z, g, zsec)
    return dict(chi=chi, wc=wc, zsec=zsec)
