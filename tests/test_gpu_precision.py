"""GPU: what the four-field stress family and its scaling leave of the FP32
accuracy, against the FP64 oracle."""
import numpy as np
import pytest

import oracle as O
import qvti
from cases import rel_l2, small_case

pytestmark = pytest.mark.gpu


def _engine(shot, **kw):
    return qvti.Engine(shot["nx"], shot["ny"], shot["nz"], shot["pml"], shot["dx"], shot["dy"], shot["dz"],
                       shot["dt"], shot["f0"], shot["w0"], **kw)


# wavelet about 95 Hz (small_case); the grid's f0 (which only shapes the C-PML)
# and the Q reference frequency far below it, at it, and f0 far above it
@pytest.mark.parametrize("f0,f_ref", [(0.5, 5.0), (0.5, 95.0), (30.0, 30.0), (95.0, 1.0), (400.0, 95.0)])
@pytest.mark.parametrize("kspace", [False, True])
def test_accuracy_does_not_depend_on_f0(f0, f_ref, kspace):
    """v shares a complex transform with w = alpha (v + kappa dv), which grows
    with the frequency of the wave: the rounding of v must stay that of plain
    FP32 for a wavelet of any band, within twice the FP32 oracle's own distance
    to FP64."""
    shot, model = small_case(48, 36, 40, 4, 24, O.SRC_FZ, True, seed=11)
    shot["f0"] = f0
    shot["w0"] = float(np.float32(2 * np.pi * f_ref))
    ks = dict(vref=4000.0) if kspace else None
    ref = O.run(shot, model, "f64", state=True, kspace=ks)["state"]
    floor = rel_l2(O.run(shot, model, "f32", state=True, kspace=ks)["state"], ref)
    with _engine(shot, vti=True) as e:
        e.set_model_dict(model)
        if kspace:
            e.set_kspace(ks["vref"])
        e.begin(shot["nt"], shot["rik"], [qvti.make_shot(shot["src_kind"], (shot["sx"], shot["sy"], shot["sz"]),
                                                         shot["rx"], shot["ry"], shot["rz"])])
        e.step(shot["nt"])
        e.finish()
        err = rel_l2(e.state(), ref)
    print("f0 %g, f_ref %g, k-space %d: state vs FP64 oracle %.2e, FP32 oracle %.2e" % (f0, f_ref, kspace, err, floor))
    assert err < 2 * floor
