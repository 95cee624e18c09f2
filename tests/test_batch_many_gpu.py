"""Batch slots of more than 64 segments (the lookup compares 64 at a time) and of members that end at different
steps: every member's Phi and log equal, bit for bit, those of stepping it alone."""
import numpy as np
import pytest

from oracle import core

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("count", [63, 64, 65, 131])
@pytest.mark.parametrize("prec", ["fp32", "bf16"])
def test_batch_of_many_members_equals_single_runs(mmsb, count, prec):
    rng = np.random.default_rng(count)
    members = []
    for i in range(count):
        n, k, b = 60 + 7 * (i % 9), 3 + i % 5, 20 + 10 * (i % 3)
        ys = [rng.standard_normal((n, k)) for _ in range(3)]
        members.append((n, k, b, ys, [y.mean(0) for y in ys], core.init_phi(i, k)))

    def pipeline(n, k, b, ys, mus, phi):
        p = mmsb.Pipeline(mmsb.config(nx=n, na=n, nb=n, nc=n, ncom=k, alpha_0=1.0, oversample=0, minibatch=b, learn_rate=1e-3,
                                      epochs=2, polish_epochs=0))
        p.set_yvectors(*ys, *mus)
        p.set_phi(phi)
        return p

    batch = [pipeline(*m) for m in members]
    B = mmsb.Batch(batch, prec)
    B.run(2)
    B.close()
    for m, p in zip(members, batch):
        q = pipeline(*m)
        q.stgd(-1, prec)
        assert np.array_equal(p.get("phi"), q.get("phi")) and np.array_equal(p.get("frob"), q.get("frob"))
        q.close()
        p.close()
