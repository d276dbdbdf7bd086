"""x0gemm in the bf16x3 form at the edges of its 64 x 64 tiles and 32-entry
slices: square outputs with one set of sqrt(w) planes (no weight negative) and
with two (some negative), column windows, empty bins, against the FP64 oracle on
inputs exact in 32 bits.  Each product loses at most 3 * 2^-18 of |w z z'|, summed
over the entries: below 1e-4 of the largest element.  With one set of planes the
diagonal has no error beyond its FP32 sums (about K/32 * 6 roundings of 2^-24:
4e-6 for the 300 entries of a bin here), and the increment is Hermitian to the bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def h():
    import ecalj_amd

    hd = ecalj_amd.Handle(0, "bf16x3")
    yield hd
    hd.close()


@pytest.mark.parametrize("npr,ipr_col,npr_col", [(1, 1, 1), (5, 1, 5), (63, 1, 63), (64, 1, 64), (65, 1, 65),
                                                 (130, 1, 130), (193, 1, 193), (130, 7, 65), (65, 2, 64),
                                                 (70, 1, 3), (200, 100, 101)])
@pytest.mark.parametrize("sign", [1, -1])
def test_x0gemm_edges(h, npr, ipr_col, npr_col, sign):
    import oracle as orc

    orc.build()
    print("x0gemm", npr, ipr_col, npr_col, sign, flush=True)
    rng = np.random.default_rng(npr)
    nwhis, ns1, ns2, nq, npairs = 9, 1, 4, 6, 500
    z = rng.standard_normal((npr, ns2 - ns1 + 1, nq)) + 1j * rng.standard_normal((npr, ns2 - ns1 + 1, nq))
    z = np.asfortranarray(z.astype(np.complex64).astype(np.complex128))
    itc = rng.integers(1, ns2 + 1, npairs).astype(np.int32)
    itpc = rng.integers(1, nq + 1, npairs).astype(np.int32)
    iwini = rng.choice([1, 2, 2, 2, 2, 5, 8], npairs).astype(np.int32)  # bins 4 and 7 stay empty
    nhw = rng.integers(1, 3, npairs).astype(np.int32)
    iwend = (iwini + nhw - 1).astype(np.int32)
    icouini = np.concatenate([[1], 1 + np.cumsum(nhw)[:-1]]).astype(np.int32)
    whwc = rng.uniform(0.0, 1.0, int(nhw.sum()))
    whwc[0] = 0.0
    if sign < 0:
        whwc[::3] *= -1.0
    jpmc = np.ones(npairs, np.int32)
    r0 = np.zeros((npr, npr_col, nwhis + 1), complex, order="F")
    args = (npr, ipr_col, npr_col, nwhis, 1, ns1, ns2, z, 1, npairs, iwini, iwend, itc, itpc, jpmc, icouini, whwc)
    g = h.x0gemm(r0.copy(order="F"), *args)
    o = orc.x0gemm(r0.copy(order="F"), *args)
    assert np.abs(g - o).max() < 1e-4 * np.abs(o).max()
    assert np.all(g[:, :, np.abs(o).max(axis=(0, 1)) == 0.0] == 0.0)
    if ipr_col == 1 and npr == npr_col:
        i, j = np.triu_indices(npr, 1)
        assert np.array_equal(g[j, i], g[i, j].conj())
        if sign > 0:
            d = np.arange(npr)
            assert np.all(np.abs(g[d, d].real - o[d, d].real) <= 4e-6 * np.abs(o[d, d].real))
