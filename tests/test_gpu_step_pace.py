"""GPU: several contexts of small grids stepped in turn by one thread, one step
a call, where the host's launches set the pace."""
import time

import numpy as np
import pytest

import oracle as O
import qvti
from cases import small_case

pytestmark = pytest.mark.gpu

NT = 640


def _run(n, graphs, contexts, read):
    """us a step, and every context's records and final state."""
    shot, model = small_case(*n, 4, NT, O.SRC_FZ, True)
    es = []
    for k in range(contexts):
        e = qvti.Engine(*n, shot["pml"], shot["dx"], shot["dy"], shot["dz"], shot["dt"], shot["f0"], shot["w0"],
                        vti=True)
        e.set_model_dict(model)
        e.set_graphs(graphs)
        e.begin(NT, shot["rik"] * np.float32(k + 1),
                [qvti.make_shot(O.SRC_FZ, (shot["sx"], shot["sy"], shot["sz"] + k % 3), shot["rx"], shot["ry"],
                                shot["rz"])])
        es.append(e)
    best, done = 1e9, 0
    for block in (40, 200, 200, 200):
        t0 = time.perf_counter()
        for it in range(block):
            for e in es:
                e.step(1)
            if read and it % 50 == 7:
                es[it % contexts].state()  # eager work and waits between the replays
        for e in es:
            e.sync()
        done += block
        best = min(best, (time.perf_counter() - t0) / block / contexts)
    assert done == NT
    out = [(e.finish()[0], e.state()) for e in es]
    for e in es:
        e.close()
    return best * 1e6, out


@pytest.mark.parametrize("n,contexts,read", [((18, 18, 20), 1, True), ((18, 18, 20), 3, True), ((20, 18, 16), 4, True),
                                             ((32, 32, 32), 8, False), ((50, 30, 32), 8, False)])
def test_contexts_stepped_in_turn_give_the_same_bits(n, contexts, read):
    """With several contexts in turn a step goes as a graph of its own, with one
    by direct launches: records and states equal those of direct launches
    (set_graphs(False)) in both, with readbacks between the replays too.  The
    times are printed only: the host's share differs between machines (32^3,
    eight contexts, direct / graph: 31 / 20 us and 23 / 19.5 us)."""
    direct, want = _run(n, False, contexts, read)
    us, got = _run(n, True, contexts, read)
    print("%dx%dx%d, %d contexts in turn: %.1f us a step by direct launches, %.1f now" % (*n, contexts, direct, us))
    for (r0, s0), (r1, s1) in zip(want, got):
        assert np.array_equal(r0, r1) and np.array_equal(s0, s1)
