"""W build in the bf16x3 form at sizes around the operand planes' chunks of 8,
slices of 32 and tiles of 128 (odd leading dimensions included: rows then start
at any 8 bytes), all basis options, against numpy in complex128.  Bar: four
transforms whose products each lose at most 3 * 2^-17 of sum |a||b| <= sqrt(n)
times the result's scale for a unitary factor, plus the complex64 storage of
chi_E and W_E, times cond(eps): 4 * 3 * 2^-17 * sqrt(131) = 1e-3 at worst, and a
tenth of it since the roundings are independent."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def h():
    import ecalj_amd

    hd = ecalj_amd.Handle(0, "bf16x3")
    yield hd
    hd.close()


@pytest.mark.parametrize("n", [1, 7, 8, 9, 31, 33, 64, 127, 129, 131])
@pytest.mark.parametrize("real", [False, True])
def test_wc_build_sizes(h, n, real):
    print("wc_build bf16x3", n, real, flush=True)
    rng = np.random.default_rng(n)
    vc = rng.uniform(0.5, 4.0, n)
    s = np.sqrt(vc)
    Q, _ = np.linalg.qr(rng.standard_normal((n, n)) + 1j * rng.standard_normal((n, n)))
    Q = np.asfortranarray(Q)
    chi = np.zeros((n, n, 2), complex, order="F")
    for v in range(2):
        x = (rng.standard_normal((n, max(1, n // 2))) + 1j * rng.standard_normal((n, max(1, n // 2)))) * 0.3 / np.sqrt(n)
        chi[:, :, v] = -(x @ x.conj().T) / (1 + v)
    h.set_coulomb(vc, Q)
    for xm in (True, False):
        for wm in (True, False):
            g = (h.wc_build_real if real else h.wc_build)(chi, nspin=2, is_x0_m_basis=xm, is_wc_m_basis=wm)
            for v in range(2):
                x = Q.conj().T @ chi[:, :, v] @ Q if xm else chi[:, :, v]
                eps = np.eye(n) - s[:, None] * x * s[None, :]
                w = s[:, None] * (np.linalg.inv(eps) - np.eye(n)) * s[None, :]
                w = Q @ w @ Q.conj().T if wm else w
                err = np.abs(g[:, :, v] - w).max() / np.abs(w).max()
                assert err < 1e-4 * np.linalg.cond(eps), (xm, wm, v, err)
