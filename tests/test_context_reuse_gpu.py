"""Contexts that take over device blocks of closed ones: detections of graphs of two sizes in turn, from two threads at
once, while another context lives, give bit for bit what the first of each gave in a fresh process; the memory is given
back with the last context."""
import threading

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

SIZES = [(700, 6), (4099, 12)]


def detect(mmsb, g, n, k):
    p = mmsb.Pipeline(mmsb.config(nx=n, na=n, nb=n, nc=n, ncom=k, alpha_0=1.0, seed=1, minibatch=128, epochs=3,
                                  learn_rate=1e-3))
    p.set_graph(g)
    p.whiten()
    p.stgd(-1, "bf16")
    p.eigen()
    p.post()
    out = [p.get("phi"), p.get_f32("pin_x"), p.get_f32("pin_c")]
    p.close()
    return out


def test_blocks_of_closed_contexts(mmsb):
    graphs = [mmsb.generate(n, n, n, n, k, 1.0, min(0.9, 40 * k / n), 10 / n, seed=3) for n, k in SIZES]
    detect(mmsb, graphs[0], *SIZES[0])
    torch.cuda.synchronize()
    free0 = torch.cuda.mem_get_info()[0]
    first = [detect(mmsb, g, *s) for g, s in zip(graphs, SIZES)]
    keep = mmsb.Pipeline(mmsb.config(nx=100, na=100, nb=100, nc=100, ncom=3, seed=1))
    bad = []

    def work(order):
        for i in order:
            out = detect(mmsb, graphs[i], *SIZES[i])
            if not all(np.array_equal(a, b) for a, b in zip(out, first[i])):
                bad.append(i)

    threads = [threading.Thread(target=work, args=(o,)) for o in ([0, 1, 0, 1, 1], [1, 0, 0, 1, 0])]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    keep.close()
    assert not bad
    torch.cuda.synchronize()
    assert torch.cuda.mem_get_info()[0] >= free0 - (8 << 20)
