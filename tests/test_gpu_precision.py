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


# The wave's axis (512 cells), the stress component that reads one moduli set
# along it, and the set's coefficients: P in pzz, D - 2 S in pxx, H in pxx
@pytest.mark.parametrize("axis,field,sets", [(2, 5, "P"), (2, 3, "D-2S"), (0, 3, "H")])
def test_q_coefficients_are_rounded_once(axis, field, sets):
    """The FP64 Q coefficients are rounded to FP32 and used as they are.

    In a model that varies from column to column only, a plane wave along the
    columns (put in through a checkpoint image, stresses at rest) gives each
    column of one stress update the value sum_j o_j p_j: its own four
    coefficients and four numbers common to all columns.  With the p_j fitted
    over the columns, the residual is the rounding of the update itself: four
    multiply-adds and the step, 2^-24 / sqrt(3) each, over 504 cells weighted
    with a sine, 4e-9 of the value.  The bound is 2.5 times that; one more
    rounding of a coefficient as large as the sum (low reference frequency and
    Q of 0.5 to 3: all four count) would add 2e-8 or more."""
    n = [24, 20, 24]
    n[axis] = 512
    pml, mode, pi = 4, 37, 3.1415926
    cols = [24, 20] if axis == 2 else [20, 24]
    rng = np.random.default_rng(7)
    draw = {"vp": (2000, 4000), "vs": (1000, 1400), "rho": (1500, 3000), "gp": (0.1, 0.4), "gs": (0.1, 0.4),
            "eps": (0.0, 0.2), "delta": (0.0, 0.1)}
    col = {k: rng.uniform(a, b, cols).astype(np.float32) for k, (a, b) in draw.items()}
    model = {k: np.ascontiguousarray(np.broadcast_to(np.expand_dims(a, axis), n)) for k, a in col.items()}
    shot = dict(nx=n[0], ny=n[1], nz=n[2], pml=pml, dx=10.0, dy=10.0, dz=10.0, dt=5e-4, f0=5.0,
                w0=float(np.float32(2 * np.pi * 5)))
    i = np.arange(512)
    N = int(np.prod(n))
    with _engine(shot, vti=True) as e:
        e.set_model_dict(model)
        e.begin(2, np.zeros(2, np.float32), [qvti.make_shot(O.SRC_EXPLOSIVE, (12, 10, 12), [], [], [])])
        img = np.frombuffer(bytes(e.checkpoint()), np.uint8).copy()
        slabs = [2 * pml * N // n[a] for a in range(3)]
        head = img.size - 4 * (9 * N + 8 * slabs[0] + 8 * slabs[1] + 7 * slabs[2])
        v = np.zeros([3] + n, np.float32)
        wave = np.expand_dims(np.cos(2 * np.pi * mode * i / 512), [a for a in range(3) if a != axis])
        v[axis] = wave.astype(np.float32)
        img[head:head + 12 * N] = v.view(np.uint8).reshape(-1)
        e.restore(img)
        e.step(1)
        e.finish()
        st = e.state()[field].astype(np.float64)
    # the coefficients (cuviscoelas_3D.cu:195-205) of A1 w, v, A3 v and w, up to powers of two
    c = {k: a.astype(np.float64) for k, a in col.items()}

    def coef(speed, g):
        cc = speed * np.cos(g * pi / 2)
        M = c["rho"] * cc * cc
        return np.stack([c["rho"] * cc * g * shot["w0"], M + M * g * g, c["rho"] * cc ** 3 * g / shot["w0"],
                         M * g * g]).astype(np.float32)

    c33, c44 = c["rho"] * c["vp"] ** 2, c["rho"] * c["vs"] ** 2
    vd = np.sqrt((np.sqrt((c33 - c44) * (c33 * (1 + 2 * c["delta"]) - c44)) + c44) / c["rho"])
    o = {"P": lambda: coef(c["vp"], c["gp"]), "H": lambda: coef(c["vp"] * np.sqrt(1 + 2 * c["eps"]), c["gp"]),
         "D-2S": lambda: coef(vd, c["gp"]) - 2 * coef(c["vs"], c["gs"])}[sets]()
    assert o.dtype == np.float32
    s = np.where((i >= pml) & (i < 512 - pml), np.sin(2 * np.pi * mode * (i + 0.5) / 512), 0.0)
    Y = np.tensordot(np.moveaxis(st, axis, 2), s, (2, 0))[:-1, :-1]  # (the last planes are not updated)
    inner = Y[pml:-pml, pml:-pml].ravel()
    X = np.stack([q[:-1, :-1][pml:-pml, pml:-pml].ravel().astype(np.float64) for q in o], 1) / inner[:, None]
    X /= np.abs(X).max(0)
    p = np.linalg.lstsq(X, np.ones(len(inner)), rcond=None)[0]
    rms = float(np.sqrt(np.mean((X @ p - 1) ** 2)))
    print("%s: residual rms %.2e over %d columns" % (sets, rms, len(inner)))
    assert rms < 1e-8


@pytest.mark.parametrize("media", [qvti.MEDIA_VISCO, qvti.MEDIA_DISPERSION, qvti.MEDIA_LOSSLESS, qvti.MEDIA_QCOMP])
def test_fluid_and_lossless_cells(media):
    """Cells without shear stiffness (vs = 0: a speed of zero has no low bits),
    without loss (gamma = 0), and with a negative gamma: the whole state within
    the bound of the other step cases."""
    shot, model = small_case(20, 18, 24, 4, 12, O.SRC_EXPLOSIVE, True, seed=5)
    model = {k: a.copy() for k, a in model.items()}
    model["vs"][:10] = 0
    model["gp"][:, :9] = 0
    model["gs"][:, :9] = 0
    model["gp"][:, :, :6] *= -1
    ref = O.run(shot, model, "f64", state=True, media=media)["state"]
    with _engine(shot, vti=True) as e:
        e.set_media(media)
        e.set_model_dict(model)
        e.begin(shot["nt"], shot["rik"], [qvti.make_shot(shot["src_kind"], (shot["sx"], shot["sy"], shot["sz"]),
                                                         shot["rx"], shot["ry"], shot["rz"])])
        e.step(shot["nt"])
        e.finish()
        st = e.state()
    assert np.isfinite(ref).all() and np.isfinite(st).all()
    assert rel_l2(st[:3], ref[:3]) < 1e-5 and rel_l2(st[3:], ref[3:]) < 1e-5
