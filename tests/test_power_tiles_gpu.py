"""The power method's products at the edges of their 32 and 64 blocks, and of its 65536-row chunks, against the
oracle. Planted vectors (orthonormal directions plus noise), so that the orthonormalisation is well
conditioned: Phi returns rounded to FP32 (6e-8 of entries below 1), lambda is FP64 sums of n terms."""
import numpy as np
import pytest

from oracle import core

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,k", [(40, 1), (31, 31), (65, 33), (300, 64), (1025, 65), (6145, 70), (65537, 20), (131072, 5)])
@pytest.mark.parametrize("orth", [False, True])
def test_power_method_at_block_edges(mmsb, n, k, orth):
    rng = np.random.default_rng(n + k)
    V = np.linalg.qr(rng.standard_normal((k, k)))[0]
    base = np.sqrt(k) * V[np.arange(n) % k]
    ys = [(base + 0.2 * rng.standard_normal((n, k))).astype(np.float32).astype(np.float64) for _ in range(3)]
    mus = [y.mean(0) for y in ys]
    phi0 = np.linalg.qr(V.T + 0.2 * rng.standard_normal((k, k)))[0].astype(np.float32).astype(np.float64)
    cfg = mmsb.config(nx=n, na=n, nb=n, nc=n, ncom=k, alpha_0=0.8, oversample=0, minibatch=64)
    p = mmsb.Pipeline(cfg)
    try:
        p.set_yvectors(*ys, *mus)
        p.set_phi(phi0)
        print(f"case n={n} k={k} orth={orth}", flush=True)
        lam = p.power_method(2, orthogonalize=orth)
        phi = p.get("phi")
    finally:
        p.close()
    want, want_l = core.power_method(*ys, *mus, phi0, alpha0=0.8, iters=2, orthogonalize=orth)
    assert np.abs(phi - want).max() <= 1e-6
    assert np.abs(lam - want_l).max() <= 1e-9 * np.abs(want_l).max()
