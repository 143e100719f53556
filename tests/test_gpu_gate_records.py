"""The gate reads positions from the grid's origin and velocities in float;
its reach covers their rounding.  A long domain far from the origin, fast
agents and pairs that nearly keep their distance: the same bits as the tiled
kernel, which evaluates every candidate."""
import numpy as np
import pytest

from crowddynamics_amd.stepper import Stepper
from tests.test_gpu_pair_queue import _agents

pytestmark = pytest.mark.gpu


@pytest.mark.filterwarnings('ignore')
@pytest.mark.parametrize('model', ['circular', 'three_circle'])
@pytest.mark.parametrize('precision', ['f64', 'f32'])
@pytest.mark.parametrize('length,offset,speed', [
    (30.0, 0.0, 1e-6),      # collisions later than any force looks
    (30.0, 1e7, 1.0),
    (1e5, -1e5, 1.0),       # a coordinate's float spacing is 2^-7 m
    (1e5, 0.0, 2000.0),
    (30.0, 0.0, 1e6),
])
def test_records_equal_every_candidate(model, precision, length, offset, speed):
    n = 600
    rng = np.random.default_rng(int(length + speed) % 1000)
    arr = _agents(model, n, 6.0, 7)
    shift = np.zeros((n, 2))
    shift[:, 0] = rng.integers(0, max(1, int(length / 30.0)), n // 20).repeat(20) * 30.0 + offset
    shift[:, 1] = offset
    for f in ('position', 'position_ls', 'position_rs'):
        if f in arr.dtype.names:
            arr[f] += shift
    # a common velocity and a small one of each agent's own
    arr['velocity'] = ((speed, 0.5 * speed) + speed * 1e-3 * arr['velocity']).astype(np.float32)
    out = []
    for kw in (dict(tile=(2, 2)), dict(lanes=4), dict(lanes=32)):
        st = Stepper(arr.copy(), cell_size=3.6, dt_min=1e-6, dt_max=1e-6, seed=3,
                     precision=precision, cell_capacity=150000, **kw)
        st.step(2)
        out.append(st.download(arr.copy()))
    for got in out[1:]:
        for f in ('position', 'velocity', 'force_prev'):
            assert np.array_equal(got[f], out[0][f]), f
