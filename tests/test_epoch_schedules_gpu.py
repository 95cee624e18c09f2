"""Epochs whose settings change every time are launched directly: with a new learning rate for each, a context that
may capture epochs takes no longer than one that may not (a capture for a single replay made it 1.35 times as long), and
gives the same results."""
import time

import numpy as np
import pytest

from oracle import core

pytestmark = pytest.mark.gpu


def test_learning_rate_schedule(mmsb):
    n, k, b = 4096, 40, 64  # 64 steps per epoch
    rng = np.random.default_rng(4)
    ys = [rng.standard_normal((n, k)) for _ in range(3)]
    mus = [0.1 * rng.standard_normal(k) for _ in range(3)]
    ps = []
    for graphs in (1, 0):
        p = mmsb.Pipeline(mmsb.config(nx=n, na=n, nb=n, nc=n, ncom=k, oversample=0, minibatch=b, learn_rate=1e-5,
                                      use_graphs=graphs))
        p.set_yvectors(*ys, *mus)
        p.set_phi(core.init_phi(3, k))
        ps.append(p)
    best = [1.0, 1.0]
    for epoch in range(30):
        for i, p in enumerate(ps):
            p.set_learn_rate(1e-4 / (epoch + 1))
            t = time.perf_counter()
            p.stgd(n // b, "fp32")
            if epoch >= 4:
                best[i] = min(best[i], time.perf_counter() - t)
    print(f"epoch {1e6 * best[0]:.0f} us with captures allowed, {1e6 * best[1]:.0f} without", flush=True)
    assert np.array_equal(ps[0].get("phi"), ps[1].get("phi")) and np.array_equal(ps[0].get("frob"), ps[1].get("frob"))
    assert best[0] < 1.15 * best[1]
    for p in ps:
        p.close()
