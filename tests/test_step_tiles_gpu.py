"""FP32 steps whose second phase takes 16 x 16 tiles (k <= 320) against the 32 x 32 tiles of a batch, which both add the
products in the same order: Phi and the log are equal bit for bit, over widths at the tiles' and the register rings'
edges and both sides of the limit, and minibatches whose rows are aligned, unaligned (odd logical size), ragged and of
one, two, three, four and many groups per wave. BF16 steps at the same sizes go along: their rings differ by the number
of groups too."""
import numpy as np
import pytest

from oracle import core

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [33, 64, 65, 129, 192, 256, 257, 320, 321])
@pytest.mark.parametrize("b,n", [(64, 130), (61, 200), (128, 128), (255, 700), (384, 800), (1024, 2100)])
@pytest.mark.parametrize("prec", ["fp32", "bf16"])
def test_step_tiles(mmsb, k, b, n, prec):
    print(f"case k={k} b={b} n={n} {prec}", flush=True)
    n = max(n, k)  # a partition holds at least k nodes
    rng = np.random.default_rng(k + b)
    ys = [rng.standard_normal((n, k)) for _ in range(3)]
    mus = [0.2 * rng.standard_normal(k) for _ in range(3)]
    phi = core.init_phi(k, k)

    def pipeline():
        p = mmsb.Pipeline(mmsb.config(nx=n, na=n, nb=n, nc=n, ncom=k, alpha_0=1.0, oversample=0, minibatch=b, learn_rate=1e-4,
                                      epochs=2, polish_epochs=0))
        p.set_yvectors(*ys, *mus)
        p.set_phi(phi)
        return p

    p, q = pipeline(), pipeline()
    B = mmsb.Batch([p], prec)
    B.run(2)
    B.close()
    q.stgd(-1, prec)
    assert np.isfinite(q.get("phi")).all()
    assert np.array_equal(p.get("phi"), q.get("phi")) and np.array_equal(p.get("frob"), q.get("frob"))
    p.close()
    q.close()
