"""CholeskyQR2 of Phi~ (the QR renormalisation) at the edges of the Cholesky forms: one column, the 16-row blocks, 64
lanes, the largest triangle kept in LDS (128) and the forms beyond, up to the block counts of the triangular inverse's
register classes (512 rows). One FP32 step from an orthonormal Phi keeps Phi~ well conditioned, so Phi carries the FP32
rounding of Phi~ and of the stored factor: a few 2^-24 per element, sqrt(k) of them in a norm; 1e-5 bounds both checks."""
import numpy as np
import pytest

from oracle import core

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [1, 2, 15, 16, 17, 31, 32, 33, 48, 63, 64, 65, 111, 112, 113, 127, 128, 129, 256, 257, 512, 513])
def test_qr_step(mmsb, k):
    n = max(64, k + 3)
    rng = np.random.default_rng(k)
    ys = [rng.standard_normal((n, k)) / np.sqrt(k) for _ in range(3)]
    mus = [0.2 * rng.standard_normal(k) for _ in range(3)]
    phi0 = core.init_phi(k, k)
    print(f"case k={k}", flush=True)
    p = mmsb.Pipeline(mmsb.config(nx=n, na=n, nb=n, nc=n, ncom=k, alpha_0=1.2, oversample=0, minibatch=n, learn_rate=1e-3,
                                  renorm_mode="qr", m2_scaling="gpu"))
    p.set_yvectors(*ys, *mus)
    p.set_phi(phi0)
    p.stgd(1, "fp32")
    phi = p.get("phi")
    ref, _ = core.stgd(*ys, *mus, phi0, alpha0=1.2, eta=1e-3, batch=n, epochs=1, steps=1, scaling="gpu", renorm_mode="qr")
    assert np.linalg.norm(phi - ref) / np.linalg.norm(ref) < 1e-5
    assert np.abs(phi.T @ phi - np.eye(k)).max() < 1e-5
    p.close()
