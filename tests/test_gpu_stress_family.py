"""GPU: the four-field stress family {A1 w, v, A3 v, w}, w = alpha (v + kappa
dv), against the FP64 oracle, which evaluates the scheme's five terms per
moduli set.  kappa and alpha depend on the Q reference frequency and the
medium, and the stress update's tile (rows per workgroup) on the row length.

The bound is that of the other step cases (1e-5 relative L2): FP32 rounding
per step is about 1e-7 and the runs take at most 20 steps.
"""
import numpy as np
import pytest

import oracle as O
import qvti
from cases import rel_l2, small_case

pytestmark = pytest.mark.gpu

TOL = 1e-5

# row lengths of every tile shape (192, 256 and 512 threads; 1 to 10 rows),
# with row counts that leave a remainder; reference frequencies below, at and
# above the source's, so that w is dominated by dv, balanced, or close to v
CASES = [
    # nx, ny, nz, vti, media, w0 / (2 pi f0)
    (18, 30, 16, True, qvti.MEDIA_VISCO, 1.0),
    (16, 18, 64, False, qvti.MEDIA_VISCO, 0.05),
    (20, 18, 96, True, qvti.MEDIA_VISCO, 20.0),
    (18, 18, 128, True, qvti.MEDIA_QCOMP, 0.3),
    (18, 16, 150, False, qvti.MEDIA_DISPERSION, 1.0),
    (16, 18, 200, True, qvti.MEDIA_VISCO, 3.0),
    (16, 20, 256, False, qvti.MEDIA_LOSSLESS, 1.0),
    (18, 16, 324, True, qvti.MEDIA_QCOMP, 1.0),
    (16, 16, 400, True, qvti.MEDIA_VISCO, 0.5),
    (18, 16, 512, False, qvti.MEDIA_VISCO, 1.0),
]


@pytest.mark.parametrize("nx,ny,nz,vti,media,ratio", CASES)
def test_stress_family_matches_the_oracle(nx, ny, nz, vti, media, ratio):
    shot, model = small_case(nx, ny, nz, 4, 12 if nx * ny * nz > 50000 else 20, O.SRC_FX, vti, seed=nz)
    shot["w0"] = float(np.float32(shot["w0"] * ratio))
    ref = O.run(shot, model, "f64", state=True, media=media)
    with qvti.Engine(nx, ny, nz, shot["pml"], shot["dx"], shot["dy"], shot["dz"], shot["dt"], shot["f0"], shot["w0"],
                     vti=vti) as e:
        e.set_media(media)
        e.set_model_dict(model)
        e.begin(shot["nt"], shot["rik"], [qvti.make_shot(shot["src_kind"], (shot["sx"], shot["sy"], shot["sz"]),
                                                         shot["rx"], shot["ry"], shot["rz"])])
        e.step(shot["nt"])
        e.finish()
        st = e.state()
    errs = [rel_l2(st[k], ref["state"][k]) for k in range(9)]
    print("%dx%dx%d media %d w0 ratio %g: state vs FP64 oracle %.2e, per field max %.2e"
          % (nx, ny, nz, media, ratio, rel_l2(st, ref["state"]), max(errs)))
    assert rel_l2(st[:3], ref["state"][:3]) < TOL
    assert rel_l2(st[3:], ref["state"][3:]) < TOL


@pytest.mark.parametrize("scale", [0.05, 1.0, 20.0])
def test_field_scales_suit_slow_and_fast_media(scale):
    """v shares a complex transform with L |k| v; in a slow medium on a fine
    grid, and in a fast one on a coarse grid, its rounding must stay that of
    plain FP32: within twice the FP32 oracle's own distance to FP64."""
    shot, model = small_case(48, 36, 40, 4, 20, O.SRC_FX, True, seed=3)
    for k in ("dx", "dy", "dz"):
        shot[k] = float(np.float32(shot[k] * scale))
    shot["dt"] = float(np.float32(shot["dt"] * min(scale, 1.0)))
    model = dict(model, vp=model["vp"] * np.float32(scale), vs=model["vs"] * np.float32(scale))
    ref = O.run(shot, model, "f64", state=True)["state"]
    floor = rel_l2(O.run(shot, model, "f32", state=True)["state"], ref)
    with qvti.Engine(48, 36, 40, shot["pml"], shot["dx"], shot["dy"], shot["dz"], shot["dt"], shot["f0"], shot["w0"],
                     vti=True) as e:
        e.set_model_dict(model)
        e.begin(shot["nt"], shot["rik"], [qvti.make_shot(shot["src_kind"], (shot["sx"], shot["sy"], shot["sz"]),
                                                         shot["rx"], shot["ry"], shot["rz"])])
        e.step(shot["nt"])
        e.finish()
        err = rel_l2(e.state(), ref)
    print("scale %g: state vs FP64 oracle %.2e, FP32 oracle %.2e" % (scale, err, floor))
    assert err < 2 * floor


# strided lengths next to row lengths that leave a partial last tile at every
# tile width, and every pencil count per workgroup (8 to 64 columns)
STRIDED = [(16, 24, 18), (64, 18, 50), (18, 90, 30), (128, 16, 54), (20, 200, 18), (250, 16, 20), (16, 400, 36),
           (486, 18, 16), (18, 512, 30)]


@pytest.mark.parametrize("nx,ny,nz", STRIDED)
def test_strided_stress_derivatives_match_the_oracle(nx, ny, nz):
    """Shear sums and stored derivatives along x and y (two shots, so that the
    per-shot offsets count): within the bound at the narrowest tiles, and the
    same bits at every tile width and split."""
    shot, model = small_case(nx, ny, nz, 4, 8, O.SRC_EXPLOSIVE, True, seed=nx + ny)
    ref = O.run(shot, model, "f64", state=True)
    got = []
    for mode in (0, 2, 4, 16, 18, 20):
        with qvti.Engine(nx, ny, nz, shot["pml"], shot["dx"], shot["dy"], shot["dz"], shot["dt"], shot["f0"],
                         shot["w0"], vti=True, max_shots=2) as e:
            e.set_autotune(mode)
            e.set_model_dict(model)
            one = [qvti.make_shot(shot["src_kind"], (shot["sx"] + d, shot["sy"], shot["sz"]), shot["rx"], shot["ry"],
                                  shot["rz"]) for d in (1, 0)]
            e.begin(shot["nt"], shot["rik"], one)
            e.step(shot["nt"])
            e.finish()
            got.append(e.state(1))
    err = rel_l2(got[0], ref["state"])
    print("%dx%dx%d: state vs FP64 oracle %.2e" % (nx, ny, nz, err))
    assert err < TOL
    for st in got[1:]:
        assert np.array_equal(st, got[0])


@pytest.mark.parametrize("kind", [O.SRC_FX, O.SRC_FY, O.SRC_FZ, O.SRC_EXPLOSIVE])
def test_records_are_the_wavefield_after_the_source(kind):
    """Receivers are sampled before the stress update adds the source to its
    cell; the records must still be, bit for bit, the velocities that the
    step leaves behind - at the source cell, beside it, and for shots with
    more receivers than threads and with none."""
    shot, model = small_case(18, 18, 20, 4, 6, kind, True)
    src = (shot["sx"], shot["sy"], shot["sz"])
    near = [src, (src[0], src[1], src[2] + 1), (0, 0, 0), (17, 17, 19)]
    full = [(x, y, 7) for x in range(18) for y in range(18)] + near
    sets = [near, full, []]
    with qvti.Engine(18, 18, 20, shot["pml"], shot["dx"], shot["dy"], shot["dz"], shot["dt"], shot["f0"], shot["w0"],
                     vti=True, max_shots=3) as e:
        e.set_model_dict(model)
        rs = [np.array(r, np.int32).reshape(-1, 3) for r in sets]
        e.begin(shot["nt"], shot["rik"], [qvti.make_shot(kind, src, r[:, 0], r[:, 1], r[:, 2]) for r in rs])
        want = []
        for _ in range(shot["nt"]):
            e.step(1)
            want.append([e.state(k)[:3] for k in range(3)])
        rec = e.finish()
    for k, r in enumerate(rs):
        for t in range(shot["nt"]):
            assert np.array_equal(rec[k][:, t], want[t][k][:, r[:, 0], r[:, 1], r[:, 2]]), (k, t)


@pytest.mark.parametrize("nx,ny,nz,shots", [(96, 90, 512, 1), (128, 128, 128, 1), (64, 48, 96, 17), (160, 160, 64, 4)])
def test_streaming_variants_give_the_same_bits(nx, ny, nz, shots):
    """Grids beyond the Infinity Cache take non-temporal variants of the
    kernels (all of them, or the stress kernels only).  Shot 0 of the batch
    must equal the same shot run alone on a context of one shot, and every
    tile width must give the same bits (widths differ in which tiles are whole
    lines); the first case, one shot, is checked against the oracle."""
    shot, model = small_case(nx, ny, nz, 6, 3, O.SRC_FZ, True, seed=5)

    def run(n, mode):
        with qvti.Engine(nx, ny, nz, shot["pml"], shot["dx"], shot["dy"], shot["dz"], shot["dt"], shot["f0"],
                         shot["w0"], vti=True, max_shots=n) as e:
            e.set_autotune(mode)
            e.set_model_dict(model)
            e.begin(shot["nt"], shot["rik"],
                    [qvti.make_shot(shot["src_kind"], (shot["sx"] + k % 3, shot["sy"], shot["sz"]), shot["rx"],
                                    shot["ry"], shot["rz"]) for k in range(n)])
            e.step(shot["nt"])
            e.finish()
            return e.state(0)

    ref = run(1, 0)
    for mode in (0, 2, 4, 16):
        assert np.array_equal(run(shots, mode), ref), mode
    if (nx, ny, nz) == (96, 90, 512):
        want = O.run(shot, model, "f64", state=True)["state"]
        err = rel_l2(ref, want)
        print("%dx%dx%d: state vs FP64 oracle %.2e" % (nx, ny, nz, err))
        assert err < TOL
