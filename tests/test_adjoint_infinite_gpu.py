"""The adjoint with one infinite entry of Phi, where every sum has infinities of one sign only: loss and gradient are
infinite as plain FP64 arithmetic over the k columns and nb rows gives them, at sizes that are and are not multiples
of the kernels' 32 and 64 blocks (columns and rows past the end take no part)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def reference(phi, ys, mus, c3, c1, c0, theta):
    A, B, C = (y @ phi for y in ys)
    a, b, c = (m @ phi for m in mus)
    nb = ys[0].shape[0]
    G = phi.T @ phi
    loss = 0.5 * theta * (G ** 3).sum()
    loss = loss - ((c3 * A * B * C + c1 * (A * B * c + A * b * C + a * B * C)).sum(0) / nb + c0 * a * b * c).sum()
    grad = 3 * theta * phi @ (G * G)
    for y, mu, (P, Q), (p, q) in ((ys[0], mus[0], (B, C), (b, c)), (ys[1], mus[1], (A, C), (a, c)), (ys[2], mus[2], (A, B), (a, b))):
        grad = grad - y.T @ (c3 * P * Q + c1 * (P * q + p * Q)) / nb - mu[:, None] * (c0 * p * q + c1 * (P * Q).mean(0))
    return loss, grad


@pytest.mark.parametrize("k,nb", [(1, 1), (6, 50), (32, 32), (32, 33), (33, 64), (64, 6144), (70, 6150)])
@pytest.mark.parametrize("dtype", ["float64", "float32"])
def test_infinite_entry(mmsb, dev, k, nb, dtype):
    print(f"case k={k} nb={nb} {dtype}", flush=True)
    rng = np.random.default_rng(k + nb)
    # positive Phi, negative vectors and means, positive coefficients: no infinities of different sign meet
    phi = rng.uniform(0.1, 1.0, (k, k))
    phi[k // 2, k - 1] = np.inf
    ys = [torch.from_numpy(-rng.uniform(0.1, 1.0, (nb, k))).to(getattr(torch, dtype)) for _ in range(3)]
    mus = [torch.from_numpy(-rng.uniform(0.1, 1.0, k)) for _ in range(3)]
    want_l, want = reference(torch.from_numpy(phi), [y.double() for y in ys], mus, 1.0, 1.0, 1.0, 0.7)
    assert torch.isposinf(want_l) and torch.isposinf(want).all()
    loss, grad = mmsb.stgd_grad(*[y.to(dev) for y in ys], *[m.to(dev) for m in mus], torch.from_numpy(phi).to(dev), (1.0, 1.0, 1.0), 0.7)
    assert torch.isposinf(loss).all()
    assert torch.isposinf(grad).all()
