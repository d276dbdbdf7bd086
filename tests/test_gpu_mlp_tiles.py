"""The training kernels of the learned tail at their tile edges: widths and
batches around 32-wide tiles and 16-deep chunks dealt to 8 waves, rows that
start unaligned, one layer; against the FP64 oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# FP32 sums of at most 1000 terms: 2^-24 sqrt(1000) = 1.9e-6 of the largest
# element, times the few layers that a rounding passes through
TOL = 2e-5


def relerr(a, b):
    return np.abs(a - b).max() / max(np.abs(b).max(), 1e-30)


@pytest.mark.parametrize("dims", [[1, 1], [16, 32, 16], [33, 65, 31], [21, 128, 64, 5], [32, 31]])
@pytest.mark.parametrize("B", [1, 31, 33, 129, 1000])
def test_grad_tiles(dims, B):
    import ecalj_amd
    import oracle as orc

    orc.build()
    rng = np.random.default_rng(B + len(dims))
    n = ecalj_amd.mlp_nparam(dims)
    p = (rng.standard_normal(n) * 0.3).astype(np.float32)
    x = rng.standard_normal((B, dims[0])).astype(np.float32)
    t = rng.standard_normal((B, dims[-1])).astype(np.float32)
    h = ecalj_amd.Handle(0, "f32")
    try:
        dp, dx, dt = h.to_dev(p), h.to_dev(x.T), h.to_dev(t.T)
        dg, dl, dy = h.array(n, np.float32), h.array(1, np.float32), h.array((dims[-1], B), np.float32)
        h.mlp_forward_dev(dims, dp, dx, B, dy)
        h.mlp_grad_dev(dims, dp, dx, dt, B, dg, dl)
        g, loss, y = dg.download(), dl.download()[0], dy.download().T
        h.mlp_grad_dev(dims, dp, dx, dt, B, dg)
        again = dg.download()
    finally:
        h.close()
    lo, go = orc.mlp_loss_grad(dims, *(a.astype(np.float64) for a in (p, x, t)))
    assert relerr(y, orc.mlp_forward(dims, p.astype(np.float64), x.astype(np.float64))) < TOL
    assert abs(loss - lo) / lo < TOL
    assert np.array_equal(g, again)
    o = 0
    for a, b in zip(dims[:-1], dims[1:]):
        for m in (a * b, b):
            assert relerr(g[o:o + m], go[o:o + m]) < TOL, (dims, B, o)
            o += m
