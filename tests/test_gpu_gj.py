"""The Gauss-Jordan inversion at the edges of its kernels: the in-register
inverse of a diagonal block (tiles of 16 rows and 16 or 32 columns, blocks of 64 and 128)
through the W build, and the pivoted panels (one row per thread up to 768 rows,
32 columns each, exchanges as a permutation) through zminv.  FP64 against
numpy: a backward-stable inverse is within n * cond * 2^-53 of it, below 1e-10
for the condition numbers here (asserted)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def h():
    import ecalj_amd

    hd = ecalj_amd.Handle(0, "f64")
    yield hd
    hd.close()


def crand(rng, *s):
    return rng.standard_normal(s) + 1j * rng.standard_normal(s)


@pytest.mark.parametrize("n", [1, 15, 16, 17, 31, 33, 63, 64, 65, 127, 128, 129, 145, 193, 257, 400, 401])
def test_in_order(h, n):
    print("in order", n, flush=True)
    rng = np.random.default_rng(n)
    vc = rng.uniform(0.5, 2.0, n)
    s = np.sqrt(vc)
    chi = np.zeros((n, n, 2), complex, order="F")
    ref = np.zeros_like(chi)
    for v in range(2):
        x = crand(rng, n, max(1, n // 3)) / np.sqrt(n)
        chi[:, :, v] = -x @ x.conj().T
        eps = np.eye(n) - s[:, None] * chi[:, :, v] * s[None, :]
        assert n * np.linalg.cond(eps) * 2.0 ** -53 < 1e-11
        ref[:, :, v] = s[:, None] * (np.linalg.inv(eps) - np.eye(n)) * s[None, :]
    h.set_coulomb(vc, np.eye(n, dtype=complex))
    g = h.wc_build(chi, nspin=2, is_x0_m_basis=False, is_wc_m_basis=False)
    assert np.abs(g - ref).max() < 1e-10 * np.abs(ref).max()


@pytest.mark.parametrize("ties", [False, True])
@pytest.mark.parametrize("n", [129, 161, 191, 256, 300, 400, 401, 769, 801, 897])
def test_pivoted(h, n, ties):
    print("pivoted", n, ties, flush=True)
    rng = np.random.default_rng(n)
    # many equal magnitudes (the first row wins), or rows of very different size
    a = rng.integers(-1, 2, (n, n)) + 1j * rng.integers(-1, 2, (n, n)) if ties else crand(rng, n, n)
    a = np.asfortranarray(a.astype(complex))
    if not ties:
        a[: n // 2] *= 1e-2
        a[0, 0] = 0.0
    assert n * np.linalg.cond(a) * 2.0 ** -53 < 1e-7
    tol = n * np.linalg.cond(a) * 2.0 ** -53 * 4
    g = h.zminv(a)
    ref = np.linalg.inv(a)
    assert np.abs(g - ref).max() < tol * np.abs(ref).max()


@pytest.mark.parametrize("scale", [1.0, 1e-120, 1e120, 1e-155])
def test_pivot_reciprocals(h, scale):
    """A diagonal matrix: every pivot's reciprocal alone (all other products are
    with 0 and 1) has the digits of the two divisions conj(d) / |d|^2, up to an
    odd last bit; at 1e-155 |d|^2 is subnormal and its divisions are exact."""
    from fractions import Fraction

    print("reciprocals", scale, flush=True)
    n = 769
    d = crand(np.random.default_rng(3), n) * scale
    got = np.diag(h.zminv(np.asfortranarray(np.diag(d))))
    same = np.zeros(n, bool)
    for a, b in ((d.real, d.imag), (d.imag, d.real)):  # |d|^2 with either square's rounding fused away
        m = np.array([float(Fraction(x) ** 2 + Fraction(float(y * y))) for x, y in zip(a, b)])
        same |= got == d.conj().real / m + 1j * (d.conj().imag / m)
    print("the divisions' digits:", same.mean(), flush=True)
    assert same.mean() > 0.99


@pytest.mark.parametrize("bad", [0.0, np.nan])
def test_singular_column(h, bad):
    import ecalj_amd

    print("singular", bad, flush=True)
    a = np.asfortranarray(crand(np.random.default_rng(1), 200, 200))
    a[:, 150] = bad
    with pytest.raises(ecalj_amd.EcaljError) as e:
        h.zminv(a)
    assert e.value.status == 2
    h.sync()
