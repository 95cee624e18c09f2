"""Epochs that replay captured launches (from the third of a kind: precision, Phi parity and end test) and runs that a stop
request ends, on every path that takes them: more than 32 communities for the phase kernels, QR renormalisation and the
end test at any width, and the two one-workgroup kernels (FP32 up to 16 communities; up to 32). Results equal those of
direct, uninterrupted launches bit for bit, over even and odd numbers of steps per epoch."""
import threading

import numpy as np
import pytest

from oracle import core

pytestmark = pytest.mark.gpu

B = 64


def pipeline(mmsb, k, spe, **kw):
    n = B * spe
    rng = np.random.default_rng(k + spe)
    ys = [rng.standard_normal((n, k)) for _ in range(3)]
    base = dict(sgd_iter_min=0, sgd_iter_max=0, learn_rate=1e-3, polish_epochs=0)
    base.update(kw)
    p = mmsb.Pipeline(mmsb.config(nx=n, na=n, nb=n, nc=n, ncom=k, alpha_0=1.3, oversample=0, minibatch=B, **base))
    p.set_yvectors(*ys, *[0.2 * rng.standard_normal(k) for _ in range(3)])
    p.set_phi(core.init_phi(k, k))
    return p


def equal(p, q):
    phi = p.get("phi")
    assert np.isfinite(phi).all()
    assert np.array_equal(phi, q.get("phi")) and np.array_equal(p.get("frob"), q.get("frob"))


@pytest.mark.parametrize("spe", [16, 15])
@pytest.mark.parametrize("prec", ["fp32", "bf16"])
def test_replays_and_new_learning_rates(mmsb, spe, prec):
    """Eager work and host waits between the replays; a new rate drops the graphs, and later epochs capture again."""
    p, q = (pipeline(mmsb, 40, spe, use_graphs=g) for g in (1, 0))
    for epoch in range(18):
        for c in (p, q):
            if epoch in (8, 9):
                c.set_learn_rate(5e-4)
            c.stgd(spe, prec)
            c.eigen()
        equal(p, q)
    p.close()
    q.close()


@pytest.mark.parametrize("k", [5, 40, 130])
@pytest.mark.parametrize("spe", [4, 5])
@pytest.mark.parametrize("prec", ["fp32", "bf16"])
def test_replays_with_qr(mmsb, k, spe, prec):
    p, q = (pipeline(mmsb, k, spe, use_graphs=g, renorm_mode="qr") for g in (1, 0))
    for _ in range(7):
        for c in (p, q):
            c.stgd(spe, prec)
            c.eigen()
        equal(p, q)
        phi = p.get("phi")
        assert np.abs(phi.T @ phi - np.eye(k)).max() < 1e-5
    p.close()
    q.close()


@pytest.mark.parametrize("k", [12, 40])
@pytest.mark.parametrize("spe", [16, 15])
@pytest.mark.parametrize("prec", ["fp32", "bf16"])
@pytest.mark.parametrize("rule", ["thresh", "iter_max"])
@pytest.mark.parametrize("renorm", ["ns", "qr"])
def test_end_test_fires_in_a_replay(mmsb, k, spe, prec, rule, renorm):
    """The test fires at step 5 of the fifth epoch: the third or later of its kind at either parity. The context goes on
    from there."""
    last = 4 * spe + 5
    kw = dict(thresh=1e9, sgd_iter_min=last - 1) if rule == "thresh" else dict(thresh=0.0, sgd_iter_min=1, sgd_iter_max=last - 1)
    p = pipeline(mmsb, k, spe, epochs=7, renorm_mode=renorm, **kw)
    q = pipeline(mmsb, k, spe, use_graphs=0, renorm_mode=renorm)
    p.stgd(-1, prec)
    assert p.get("frob").size == last + 1
    q.stgd(last + 1, prec)
    equal(p, q)
    for c in (p, q):
        c.stgd(3, prec)
    equal(p, q)
    p.close()
    q.close()


@pytest.mark.parametrize("k", [10, 20, 40])
@pytest.mark.parametrize("spe", [16, 15])
@pytest.mark.parametrize("prec", ["fp32", "bf16"])
def test_stop_requests(mmsb, k, spe, prec):
    """Requested before the call: one epoch runs. Requested from another thread: the run ends at an epoch boundary. The
    context goes on from there."""
    p, q = (pipeline(mmsb, k, spe, epochs=50000, learn_rate=1e-5) for _ in range(2))
    p.request_stop()
    p.stgd(-1, prec)
    assert p.get("frob").size == spe
    timer = threading.Timer(0.05, p.request_stop)
    timer.start()
    p.stgd(-1, prec)
    timer.join()
    done = p.get("frob").size
    print(f"k={k} {prec}: stopped after {done // spe} epochs", flush=True)
    assert done % spe == 0 and 2 * spe <= done < 50001 * spe
    q.stgd(done, prec)
    equal(p, q)
    for c in (p, q):
        c.stgd(spe + 3, prec)
    equal(p, q)
    p.close()
    q.close()
