"""The gate reads positions from the grid's origin and velocities in float;
its reach covers their rounding.  A long domain far from the origin, fast
agents and pairs that nearly keep their distance: the same bits as the tiled
kernel, which evaluates every candidate."""
import numpy as np
import pytest

from crowddynamics_amd import _lib
from crowddynamics_amd.stepper import Stepper
from oracle import oracle as O
from tests.helpers import assert_vec_close
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


@pytest.mark.filterwarnings('ignore')
@pytest.mark.parametrize('model', ['circular', 'three_circle'])
@pytest.mark.parametrize('speed,closing,tau_0', [
    (1000.0, 1e-4, 1e5),   # a float holds these velocities to 3e-5 m/s
    (1000.0, 3e-3, 1e4),
    (30.0, 1e-5, 1e6),
    (1.5, 1e-6, 1e6),
])
def test_collisions_late_and_slow(model, speed, closing, tau_0):
    """Pairs that close in on each other far more slowly than they move: the
    three-circle pair has no latest time of collision, and with a large tau_0
    its force counts.  Against the oracle, and bit for bit against the tiled
    kernel."""
    m = 200  # pairs, 20 m apart
    rng = np.random.default_rng(int(speed))
    arr = _agents(model, 2 * m, 1.0, 3)
    at = 20.0 * np.stack([np.arange(m) // 15, np.arange(m) % 15], 1)
    a = rng.uniform(-np.pi, np.pi, m)
    d = np.stack([np.cos(a), np.sin(a)], 1)
    side = rng.uniform(-0.2, 0.2, m)[:, None] * d[:, ::-1] * (-1.0, 1.0)
    new = np.concatenate([at, at + rng.uniform(1.5, 3.0, m)[:, None] * d + side])
    arr['position'] = new
    if model == 'three_circle':
        off = 0.15 * np.stack([np.sin(arr['orientation']), -np.cos(arr['orientation'])], 1)
        arr['position_ls'], arr['position_rs'] = new - off, new + off
    common = speed * rng.uniform(0.7, 1.0, (m, 2)) * rng.choice([-1, 1], (m, 2)) * 0.7
    arr['velocity'] = np.concatenate([common + closing * d, common])
    arr['tau_0'] = tau_0
    want = arr.copy()
    O.agent_agent_block_list(want, 3.6)
    if model == 'three_circle':
        assert np.sum(want['force'].any(1)) > 0.9 * 2 * m
    out = []
    for kw in (dict(tile=(2, 2)), dict(lanes=2), dict(lanes=4), dict(lanes=32)):
        st = Stepper(arr.copy(), cell_size=3.6, dt_min=1e-6, dt_max=1e-6,
                     flags=_lib.CD_USE_AGENT_AGENT, bounds=(-5.0, -5.0, 305.0, 305.0), **kw)
        st.step(1)
        out.append(st.download(arr.copy()))
    for got in out:
        # one term an agent; the closing speed's rounding, 2^-53 speed,
        # enters it over a discriminant that is b^2 to within a hundredth
        tol = 1e3 * 2.0**-53 * speed / closing
        assert_vec_close(got['force_prev'], want['force'], 0.0, tol, 'force')
        assert np.array_equal(got['force_prev'], out[0]['force_prev'])
