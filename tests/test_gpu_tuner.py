"""GPU: what the tile tuner costs the first run of a context."""
import time

import numpy as np
import pytest

import qvti

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,nz", [(400, 400, 50), (500, 500, 32)])
def test_tuning_costs_less_than_a_short_run(nx, ny, nz):
    """Every tile candidate of the strided kernels is launched on the grid
    itself before the first run.  They take 0.6 to 0.8 of a step, six candidates
    each at these lengths: four launches for the first one and two for the
    others are 14 x 0.6 = 8.4 to 14 x 0.8 = 11.2 steps, four for each 14.4 to
    19.2.  The bound lies in the gap."""
    f = lambda v: np.full((nx, ny, nz), v, np.float32)  # noqa: E731
    model = dict(vp=f(3000), vs=f(1700), rho=f(2200), gp=f(0.005), gs=f(0.01))
    shot = qvti.make_shot(qvti.SRC_FZ, (nx // 2, ny // 2, nz // 2), [], [], [])
    rik = np.zeros(26, np.float32)
    ratio = []
    for rep in range(4):
        with qvti.Engine(nx, ny, nz, 8, 10.0, 10.0, 10.0, 5e-4, 20.0, 125.0) as e:
            e.set_model_dict(model)
            t = []
            for _ in range(2):  # the second one finds the tiles chosen
                t0 = time.perf_counter()
                e.begin(len(rik), rik, [shot])
                t.append(time.perf_counter() - t0)
            e.step(6)
            e.sync()
            t0 = time.perf_counter()
            e.step(20)
            e.sync()
            step = (time.perf_counter() - t0) / 20
        ratio.append((t[0] - t[1]) / step)
    print("%dx%dx%d: tuning takes %s steps of %.2f ms" % (nx, ny, nz, ["%.1f" % r for r in ratio], step * 1e3))
    assert min(ratio[1:]) < 13.0  # (the first context also loads the kernels)
