"""GPU: edges of the strided tiles' widths and of the receivers' slice."""
import numpy as np
import pytest

import oracle as O
import qvti
from cases import rel_l2, small_case

pytestmark = pytest.mark.gpu


def _engine(shot, **kw):
    return qvti.Engine(shot["nx"], shot["ny"], shot["nz"], shot["pml"], shot["dx"], shot["dy"], shot["dz"],
                       shot["dt"], shot["f0"], shot["w0"], **kw)


# lengths whose widest tile is not all that 1024 threads hold (a multiple of 32
# pencils instead), and those that have that width only so; 72 cells a row leave
# a partial last tile of 32 and of 64 columns
@pytest.mark.parametrize("n", [96, 108, 162, 270, 288, 320, 324, 360, 384, 432, 450, 480, 500])
@pytest.mark.parametrize("axis", [0, 1])
def test_widest_tiles_give_the_same_bits(n, axis):
    dims = (n, 16, 72) if axis == 0 else (16, n, 72)
    shot, model = small_case(*dims, 4, 4, O.SRC_FX, True, seed=n)
    got = []
    for mode in (0, 2, 4, 20):
        with _engine(shot, vti=True) as e:
            e.set_autotune(mode)
            e.set_model_dict(model)
            e.begin(shot["nt"], shot["rik"], [qvti.make_shot(shot["src_kind"], (shot["sx"], shot["sy"], shot["sz"]),
                                                             shot["rx"], shot["ry"], shot["rz"])])
            e.step(shot["nt"])
            e.finish()
            got.append(e.state())
    assert np.isfinite(got[0]).all() and got[0].any()
    for st in got[1:]:
        assert np.array_equal(st, got[0])


@pytest.mark.parametrize("dims,axis", [((480, 16, 18), 0), ((16, 500, 18), 1)])
def test_widest_tiles_match_the_oracle(dims, axis):
    shot, model = small_case(*dims, 4, 6, O.SRC_FX, True, seed=axis)
    want = O.run(shot, model, "f64", state=True)["state"]
    with _engine(shot, vti=True) as e:
        e.set_autotune(4)
        e.set_model_dict(model)
        e.begin(shot["nt"], shot["rik"], [qvti.make_shot(shot["src_kind"], (shot["sx"], shot["sy"], shot["sz"]),
                                                         shot["rx"], shot["ry"], shot["rz"])])
        e.step(shot["nt"])
        e.finish()
        assert rel_l2(e.state(), want) < 1e-5


def test_more_receivers_than_threads():
    """The receivers of a step are taken by one slice of the inverse z pass: 7
    workgroups of 256 threads at 18x18x20 (51 rows each), so 6480 receivers take
    four rounds of the loop, 1793 two of which the second has one receiver; the
    records are the velocities that each step leaves behind, in both shots."""
    shot, model = small_case(18, 18, 20, 4, 5, O.SRC_FY, True)
    src = (shot["sx"], shot["sy"], shot["sz"])
    every = np.stack(np.meshgrid(np.arange(18), np.arange(18), np.arange(20), indexing="ij"), -1).reshape(-1, 3)
    order = np.random.default_rng(1).permutation(len(every))
    sets = [every[order].astype(np.int32), every[order[:1793]].astype(np.int32)]
    with _engine(shot, vti=True, max_shots=2) as e:
        e.set_model_dict(model)
        e.begin(shot["nt"], shot["rik"], [qvti.make_shot(O.SRC_FY, src, r[:, 0], r[:, 1], r[:, 2]) for r in sets])
        want = []
        for _ in range(shot["nt"]):
            e.step(1)
            want.append([e.state(k)[:3] for k in range(2)])
        rec = e.finish()
    for k, r in enumerate(sets):
        assert rec[k].shape == (3, shot["nt"], len(r))
        for t in range(shot["nt"]):
            assert np.array_equal(rec[k][:, t], want[t][k][:, r[:, 0], r[:, 1], r[:, 2]]), (k, t)
