"""GPU: runs advance by direct launches and by graphs of several steps; every
mix of the two - set by how the steps are requested, by the probe interval and
by qvti_set_graphs - must give the same bits, on every replay, with state
readbacks, checkpoints and other contexts' runs between the calls."""
import numpy as np
import pytest

import oracle as O
import qvti
from cases import rel_l2, small_case

pytestmark = pytest.mark.gpu

NT = 75


def _engine(shot, model, graphs=True, probe=50):
    e = qvti.Engine(shot["nx"], shot["ny"], shot["nz"], shot["pml"], shot["dx"], shot["dy"], shot["dz"], shot["dt"],
                    shot["f0"], shot["w0"], vti=True)
    e.set_model_dict(model)
    e.set_graphs(graphs)
    e.set_probe(probe)
    return e


def _shot(shot):
    return qvti.make_shot(shot["src_kind"], (shot["sx"], shot["sy"], shot["sz"]), shot["rx"], shot["ry"], shot["rz"])


@pytest.fixture(scope="module")
def case():
    shot, model = small_case(18, 18, 20, 4, NT, O.SRC_FZ, True)
    with _engine(shot, model, graphs=False) as e:
        rec = e.forward(NT, shot["rik"], _shot(shot))
        e.begin(NT, shot["rik"], [_shot(shot)])
        e.step(NT)
        e.finish()
        st = e.state()
    assert rel_l2(st, O.run(shot, model, "f64", state=True)["state"]) < 1e-5
    return shot, model, rec, st


@pytest.mark.parametrize("pattern,probe", [([75], 50), ([75], 0), ([75], 7), ([25, 25, 25], 50), ([10] * 7 + [5], 50),
                                           ([1] * 11 + [64], 50), ([9, 30, 1, 35], 20), ([20, 55], 10)])
def test_step_patterns_give_the_same_bits(case, pattern, probe):
    shot, model, rec, st = case
    with _engine(shot, model, probe=probe) as e, _engine(shot, model, probe=probe) as other:
        for rep in range(3):  # the context's buffers and graph start over with each run
            e.begin(NT, shot["rik"], [_shot(shot)])
            other.begin(NT, shot["rik"], [_shot(shot)])
            for n in pattern:
                e.step(n)
                other.step(min(n, 3))
                assert e.steps_done() <= NT
                e.state()
            assert np.array_equal(e.finish()[0], rec), (pattern, probe, rep)
            assert np.array_equal(e.state(), st), (pattern, probe, rep)


def test_runs_of_different_length_and_receivers_on_one_context(case):
    """Wavelet, receiver and record buffers are kept from run to run: a run
    after a longer one with more receivers, and after a shorter one with none."""
    shot, model, rec, _ = case
    rng = np.random.default_rng(3)
    with _engine(shot, model) as e:
        for nt, nrec in ((120, 40), (NT, None), (13, 0), (NT, None), (200, 3), (NT, None)):
            if nrec is None:
                assert np.array_equal(e.forward(NT, shot["rik"], _shot(shot)), rec)
            else:
                r = rng.integers(0, 18, (nrec, 3))
                got = e.forward(nt, np.ones(nt, np.float32),
                                qvti.make_shot(O.SRC_FX, (9, 9, 9), r[:, 0], r[:, 1], r[:, 2]))
                assert got.shape == (3, nt, nrec)


def test_checkpoint_between_graph_and_direct_steps(case):
    shot, model, rec, st = case
    for at in (10, 23, 40):
        with _engine(shot, model) as e:
            e.begin(NT, shot["rik"], [_shot(shot)])
            e.step(at)
            img = e.checkpoint()
        with _engine(shot, model) as e:
            e.begin(NT, shot["rik"], [_shot(shot)])
            e.restore(img)
            e.step(NT - at)
            assert np.array_equal(e.finish()[0], rec), at
            assert np.array_equal(e.state(), st), at
