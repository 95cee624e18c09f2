"""Runs of enough epochs that both Phi parities go from direct launches to captured epochs (odd and even steps per
epoch), with stored and with rebuilt neighbour vectors and under an end test that never fires: Phi and the log equal
those of direct launches throughout."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,b", [(700, 128), (1100, 64)])  # 6 and 18 steps; with b + 12: 5 and 15
@pytest.mark.parametrize("odd", [0, 12])
@pytest.mark.parametrize("mode", ["stored", "recompute"])
@pytest.mark.parametrize("prec,rule", [("fp32", 0), ("bf16", 0), ("bf16", 1)])
def test_many_epochs(mmsb, n, b, odd, mode, prec, rule):
    g = mmsb.generate(n, n, n, n, 40, 1.0, 0.5, 0.02, seed=1)
    out = []
    for graphs in (1, 0):
        p = mmsb.Pipeline(mmsb.config(nx=n, na=n, nb=n, nc=n, ncom=40, alpha_0=1.0, seed=2, minibatch=b + odd, epochs=9,
                                      learn_rate=1e-3, y_mode=mode, use_graphs=graphs, thresh=1e-30,
                                      sgd_iter_min=1 if rule else 0, sgd_iter_max=0))
        p.set_graph(g)
        p.whiten()
        p.stgd(-1, prec)
        p.stgd(-1, prec)
        out.append((p.get("phi"), p.get("frob")))
        p.close()
    assert out[0][1].size == 18 * -(-n // (b + odd)) and np.isfinite(out[0][0]).all()
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
