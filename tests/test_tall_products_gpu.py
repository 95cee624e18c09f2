"""Whitening at the sizes where its tall products change form: one row below and at the MFMA form's 4096, widths
k + 10 at 31, 32 and 33 (its narrowest) and at the edges of the 32, 64 and 128 tiles, and small partitions
whose products run in 16 x 16 tiles. The singular values of P_BC and the eigenvalues of M2 against the FP64
oracle from the same test matrices: the sketches are stored in FP32 (6e-8), and eigenvalues move by at most the
operator's perturbation, so 1e-5 of the largest leaves two decades."""
import numpy as np
import pytest

from oracle import core

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,k", [(300, 6), (1025, 54), (4095, 22), (4096, 21), (4096, 22), (4097, 23), (4200, 54), (4200, 55),
                                 (4300, 118), (4300, 119), (20000, 30)])
def test_whitening_spectra_at_tile_edges(mmsb, n, k):
    g = mmsb.generate(n, n, n, n, k, 1.0, min(0.9, 30.0 * k / n), 6.0 / n, seed=n + k)
    bl = {nm: core.Csr(g[nm][0], g[nm][1], g[nm][3], g[nm][4]) for nm in ("XA", "XB", "XC")}
    p = mmsb.Pipeline(mmsb.config(nx=n, na=n, nb=n, nc=n, ncom=k, alpha_0=1.0, oversample=10, power_iters=1, seed=5))
    try:
        p.set_graph(g)
        print(f"case n={n} k={k}", flush=True)
        p.whiten()
        sig, lam, muw = p.get("sigma"), p.get("lam_m2"), p.get("muw_a")
        W, mu = p.get("W"), p.get("mu_a")
    finally:
        p.close()
    ref = core.whiten(bl["XA"], bl["XB"], bl["XC"], core.WhitenConfig(k=k, alpha0=1.0, oversample=10, power_iters=1, seed=5))
    assert np.abs(sig - ref["sigma"]).max() <= 1e-5 * ref["sigma"][0]
    assert np.abs(lam - ref["lam_M2"]).max() <= 1e-5 * ref["lam_M2"][0]
    # the n x 1 by n x k product: W^T mu_A of the library's own W (FP32 values, FP64 sums)
    assert np.abs(muw - W.T @ mu).max() <= 1e-12 * (np.abs(W).T @ np.abs(mu)).max()


@pytest.mark.parametrize("n,k", [(400, 54), (400, 55), (700, 246), (700, 247), (900, 375), (900, 502), (1000, 503), (1300, 625),
                                 (1300, 760)])
def test_jacobi_at_the_edges_of_its_register_classes(mmsb, n, k):
    """r = k + 10 on both sides of the columns-per-lane classes (64, 256, 384, 512, 768 entries) and of the block widths
    (8 columns with V up to 634): U and V of P_BC's randomised SVD are orthonormal and diagonalise it, U^T P_BC V =
    diag(sigma), through the blocks in FP64. U and V are FP32 products of r terms: 1e-4 as in the other whitening
    tests."""
    g = mmsb.generate(n, n, n, n, min(k, 20), 1.0, 0.5, 0.2, seed=n + k)
    p = mmsb.Pipeline(mmsb.config(nx=n, na=n, nb=n, nc=n, ncom=k, alpha_0=1e-3, oversample=10, power_iters=0, seed=5,
                                  pinv_tol=1e-9))
    try:
        p.set_graph(g)
        print(f"case n={n} k={k}", flush=True)
        p.whiten()
        U, V, sig = p.get("U"), p.get("V"), p.get("sigma")
    finally:
        p.close()
    keep = sig > 1e-6 * sig[0]
    assert keep.sum() > k // 2
    for F in (U[:, keep], V[:, keep]):
        assert np.abs(F.T @ F - np.eye(F.shape[1])).max() <= 1e-4
    # sigma are the singular values of U^T P_BC V: P_BC V applied through the blocks
    bl = {nm: core.Csr(g[nm][0], g[nm][1], g[nm][3], g[nm][4]) for nm in ("XB", "XC")}
    PV = bl["XB"].T().mul(bl["XC"].mul(V)) / n
    assert np.abs(U.T @ PV - np.diag(sig))[np.ix_(keep, keep)].max() <= 1e-4 * sig[0]
