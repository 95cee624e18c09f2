"""A context goes on after a run that diverged: mmsb_set_phi with good values makes its later runs those of a fresh
context, bit for bit, whichever kernels ran before and run now (one workgroup, 16 or 32 wide; phase kernels; a
batch). Nothing that a diverged run leaves behind in the padding of Phi's buffers is taken up again."""
import numpy as np
import pytest

from oracle import core

pytestmark = pytest.mark.gpu

N, B, SPE = 290, 100, 3   # an odd number of steps per epoch: Phi ends in the other of its two buffers


def pipeline(mmsb, k):
    rng = np.random.default_rng(k)
    ys = [rng.standard_normal((N, k)) for _ in range(3)]
    p = mmsb.Pipeline(mmsb.config(nx=N, na=N, nb=N, nc=N, ncom=k, alpha_0=1.3, oversample=0, minibatch=B, learn_rate=2e-3,
                                  epochs=3, polish_epochs=1, sgd_iter_min=0, sgd_iter_max=0))
    p.set_yvectors(*ys, *[0.2 * rng.standard_normal(k) for _ in range(3)])
    p.set_phi(core.init_phi(k, k))
    return p


def advance(mmsb, p, how, prec):
    if how == "stgd":
        p.stgd(-1, prec)
    elif how == "timed":
        p.stgd_timed(SPE, prec)
    else:
        b = mmsb.Batch([p], prec)
        b.run(1)
        b.close()


@pytest.mark.parametrize("k", [10, 20, 40])
@pytest.mark.parametrize("prec", ["fp32", "bf16"])
@pytest.mark.parametrize("diverge", ["stgd", "timed"])
@pytest.mark.parametrize("then", [("stgd", "stgd"), ("stgd", "timed"), ("stgd", "batch"), ("timed", "stgd", "timed"),
                                  ("batch", "stgd", "batch")])
def test_good_values_after_a_diverged_run(mmsb, k, prec, diverge, then):
    print(f"case k={k} {prec} {diverge} {then}", flush=True)
    p, q = pipeline(mmsb, k), pipeline(mmsb, k)
    p.set_learn_rate(1e30)
    for _ in range(2):  # both buffers of Phi
        advance(mmsb, p, diverge, prec)
    assert np.isnan(p.get("phi")).all()
    gone = p.get("frob").size
    p.set_learn_rate(2e-3)
    p.set_phi(core.init_phi(k, k))
    for how in then:
        advance(mmsb, p, how, prec)
        advance(mmsb, q, how, prec)
        assert np.isfinite(q.get("phi")).all()
        assert np.array_equal(p.get("phi"), q.get("phi"))
    assert np.array_equal(p.get("frob")[gone:], q.get("frob"))
    p.close()
    q.close()
