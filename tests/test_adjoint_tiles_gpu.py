"""The adjoint's launch shapes at the edges of their 32 and 64 blocks: one element, one under, at and over a
block, the k at which the contraction changes its block, the size from which the products do, and row
slices of unequal length. FP64 and FP32 rows against the oracle's exact adjoint. Sums of at most 3 nb + k
terms in FP64: 1e-10 of the largest entry leaves three decades over their rounding."""
import numpy as np
import pytest

from oracle import core

SHAPES = [(1, 1), (1, 70), (5, 31), (31, 33), (32, 32), (33, 64), (64, 65), (65, 193), (100, 257), (256, 70), (257, 129),
          (70, 6144), (64, 12225)]


@pytest.mark.gpu
@pytest.mark.parametrize("k,nb", SHAPES)
@pytest.mark.parametrize("dtype", ["float64", "float32"])
def test_adjoint_at_block_edges(mmsb, dev, k, nb, dtype):
    import torch
    rng = np.random.default_rng(1000 * k + nb)
    ld = k + 3  # rows of a wider matrix
    ys = [torch.from_numpy(rng.standard_normal((nb, ld))).to(dev, getattr(torch, dtype))[:, :k] for _ in range(3)]
    mus = [0.3 * rng.standard_normal(k) for _ in range(3)]
    phi = rng.standard_normal((k, k)) / np.sqrt(k)
    t = lambda a: torch.from_numpy(a).to(dev)
    co = core.paper_coeffs(1.3)
    print(f"case k={k} nb={nb} {dtype}", flush=True)
    loss, grad = mmsb.stgd_grad(*ys, *[t(m) for m in mus], t(phi), co, 0.7)
    y64 = [y.double().cpu().numpy() for y in ys]
    want = core.tensor_grad(phi, *y64, *mus, co, 0.7)
    want_l = core.tensor_loss(phi, *y64, *mus, co, 0.7)
    assert np.abs(grad.cpu().numpy() - want).max() <= 1e-10 * np.abs(want).max()
    parts = np.abs(phi.T @ phi) ** 3
    assert abs(float(loss[0]) - want_l) <= 1e-10 * (abs(want_l) + parts.sum())


@pytest.mark.parametrize("k,nb,size", [(1, 1, 3584), (1, 1000000, 48009984), (10, 100, 55808), (100, 1024, 5565696),
                                       (100, 6504, 33549824), (256, 2216, 33546240), (500, 4000, 134049024),
                                       (1000, 70000, 3616096000), (2048, 512, 251854848)])
def test_published_workspace_size(mmsb, k, nb, size):
    """Callers hold buffers of mmsb_stgd_grad_workspace bytes and the fixed scratch of the allocation-free form
    bounds (k, nb) by it, so the size stays what it is."""
    assert mmsb.lib.mmsb_stgd_grad_workspace(k, nb) == size
