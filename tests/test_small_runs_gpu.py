"""Runs that fit one workgroup (k <= 32, padded minibatch <= 512) against the phase kernels, which the timed entry
point launches for every instance: Phi and the step log are equal bit for bit, over widths at the edges of the
products' pieces, full, ragged and one-row minibatches, both sides of the size limits, both Newton-Schulz
degrees, steps without renormalisation, heavy-tailed vectors that make the scale guard act, and runs longer
than one launch takes."""
import numpy as np
import pytest

from oracle import core

pytestmark = pytest.mark.gpu

SHAPES = [(1, 64, 130), (3, 1, 40), (8, 64, 64), (9, 65, 200), (10, 100, 1000), (15, 128, 129), (16, 192, 700), (17, 256, 1000),
          (24, 300, 2000), (25, 31, 95), (31, 448, 1500), (32, 500, 1777), (32, 512, 1024), (33, 512, 1500), (32, 513, 1500)]


def pipeline(mmsb, n, k, b, seed, heavy, **kw):
    rng = np.random.default_rng(seed)
    scale = rng.pareto(1.5, n)[:, None] + 0.5 if heavy else 1.0
    ys = [scale * rng.standard_normal((n, k)) for _ in range(3)]
    p = mmsb.Pipeline(mmsb.config(nx=n, na=n, nb=n, nc=n, ncom=k, alpha_0=1.3, oversample=0, minibatch=b, **kw))
    p.set_yvectors(*ys, *[0.2 * rng.standard_normal(k) for _ in range(3)])
    p.set_phi(core.init_phi(seed, k))
    return p


def same(mmsb, n, k, b, prec, runs, heavy=False, **kw):
    p, q = (pipeline(mmsb, n, k, b, n + k, heavy, **kw) for _ in range(2))
    try:
        for steps in runs:
            p.stgd(steps, prec)
            q.stgd_timed(steps, prec)
            assert np.array_equal(p.get("phi"), q.get("phi"), equal_nan=True)
        assert np.array_equal(p.get("frob"), q.get("frob"), equal_nan=True)
        assert np.isfinite(p.get("phi")).all()
    finally:
        p.close()
        q.close()


@pytest.mark.parametrize("k,b,n", SHAPES)
@pytest.mark.parametrize("prec", ["fp32", "bf16"])
def test_small_run_equals_phase_kernels(mmsb, k, b, n, prec):
    spe = -(-n // b)
    print(f"case k={k} b={b} n={n} {prec}", flush=True)
    same(mmsb, n, k, b, prec, (1, 2, spe, 2 * spe + 1), learn_rate=2e-3)


@pytest.mark.parametrize("prec", ["fp32", "bf16"])
@pytest.mark.parametrize("kw", [dict(ns_degree=5, ns_iters=1), dict(ns_degree=5, ns_iters=2), dict(ns_iters=1), dict(ns_iters=3),
                                dict(renorm_every=3), dict(renorm_every=0), dict(theta=0.3, m2_scaling="gpu")])
def test_small_run_settings(mmsb, prec, kw):
    same(mmsb, 900, 12, 128, prec, (3, 16), learn_rate=2e-3, **kw)


@pytest.mark.parametrize("prec", ["fp32", "bf16"])
def test_small_run_with_the_guard_acting(mmsb, prec):
    same(mmsb, 1000, 20, 100, prec, (10, 23), heavy=True, learn_rate=5e-2)


def test_small_run_longer_than_a_launch(mmsb):
    same(mmsb, 4099, 5, 1, "fp32", (4099, 4100), learn_rate=1e-4)


@pytest.mark.parametrize("first", [0, 3])
def test_joined_epochs_equal_single_ones(mmsb, first):
    """Mixed-precision epochs (the last one in FP32) as one call, from an epoch boundary and from inside an epoch."""
    n, k, b = 500, 10, 64
    p, q = (pipeline(mmsb, n, k, b, 5, False, epochs=6, polish_epochs=2, learn_rate=2e-3, sgd_iter_min=0, sgd_iter_max=0)
            for _ in range(2))
    p.stgd(first, "bf16")
    p.stgd(-1, "bf16")
    q.stgd_timed(first, "bf16")
    for e in range(6):
        q.stgd_timed(8, "bf16" if e < 4 else "fp32")
    assert np.array_equal(p.get("phi"), q.get("phi")) and np.array_equal(p.get("frob"), q.get("frob"))
    p.close()
    q.close()
