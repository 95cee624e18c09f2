"""Minibatch windows that hold the rows of several steps: runs that start inside an epoch, cross epochs and end at any
step, unaligned steps (odd minibatch), a window of the whole epoch, of part of it (k = 130, n = 20011: about 14000 rows)
and of the last ragged step alone -- Phi equal, bit for bit, to the form that keeps all neighbour vectors."""
import numpy as np
import pytest

from test_checkpointed_gpu import build_pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k,n,b,runs", [(12, 1000, 61, (1, 3, 17, 40)), (70, 1537, 128, (5, 13, 30)),
                                        (130, 20011, 1023, (7, 15, 21)), (130, 20011, 4096, (1, 9))])
@pytest.mark.parametrize("prec", ["fp32", "bf16"])
def test_runs_over_windows(mmsb, k, n, b, runs, prec):
    print(f"case k={k} n={n} b={b} {prec}", flush=True)
    res, win = build_pair(mmsb, n, k, b, epochs=2, p_in=min(0.5, 30.0 * k / n), p_out=10.0 / n)
    for steps in runs:
        for p in (res, win):
            p.stgd(steps, prec)
        assert np.array_equal(res.get("phi"), win.get("phi"))
    for p in (res, win):
        p.stgd(-1, prec)
    assert np.isfinite(win.get("phi")).all() and np.array_equal(res.get("phi"), win.get("phi"))
    res.close()
    win.close()
