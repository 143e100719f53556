"""The agent-parallel force kernel tests candidates with a gate and evaluates
those that pass from a queue; the tiled kernel evaluates every candidate.
Both must agree bit for bit: at every number of lanes, with cells holding
more agents than slots, crowds pressed together, agents at rest, queues that
fill several times and ones that stay empty, and shoulders anywhere."""
import numpy as np
import pytest

from crowddynamics_amd import core
from crowddynamics_amd.agents import empty_agents
from crowddynamics_amd.device import DeviceAgents, Workspace
from crowddynamics_amd.stepper import Stepper
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _agents(model, n, side, seed):
    rng = np.random.default_rng(seed)
    arr = empty_agents(n, model)
    arr['position'] = rng.uniform(0, side, (n, 2))
    arr['mass'] = rng.uniform(60, 100, n)
    arr['radius'] = rng.uniform(0.2, 0.3, n)
    arr['target_velocity'] = rng.uniform(0.8, 1.5, n)
    v = rng.normal(0, 1, (n, 2))
    v[rng.uniform(size=n) < 0.2] = 0.0          # pairs at rest
    v[rng.uniform(size=n) < 0.2] = (1.0, 0.25)  # pairs with one velocity
    arr['velocity'] = v.astype(np.float32)
    arr['target_direction'] = (1.0, 0.0)
    arr['inertia_rot'] = 4.0 * np.pi
    if model == 'three_circle':
        arr['orientation'] = rng.uniform(-np.pi, np.pi, n)
        arr['r_t'], arr['r_s'], arr['r_ts'] = 0.15, 0.1, 0.15
        arr['target_angular_velocity'] = 2 * np.pi
        # in the first step the shoulders are wherever the caller has them
        arr['position_ls'] = arr['position'] + rng.normal(0, 0.4, (n, 2))
        arr['position_rs'] = arr['position'] + rng.normal(0, 0.1, (n, 2))
    return arr


def _run(arr, steps=3, **kw):
    segs = np.array([[0, 0, 6, 0], [0, 0, 0, 6.0], [2, 1, 2, 4]])
    st = Stepper(arr.copy(), segments=segs, dt_min=0.001, dt_max=0.01, seed=3, **kw)
    st.step(steps)
    return st.download(arr.copy())


@pytest.mark.filterwarnings('ignore')
@pytest.mark.parametrize('model', ['circular', 'three_circle'])
@pytest.mark.parametrize('precision', ['f64', 'f32'])
@pytest.mark.parametrize('n,side,cell,slots', [
    (1, 1.0, 3.6, None),     # no candidate
    (2, 0.5, 0.6, None),
    (65, 40.0, 0.6, None),   # hardly any
    (400, 9.0, 3.6, None),   # long stencils, packed
    (300, 8.0, 3.6, 4),      # most cells overfull
    (700, 12.0, 0.9, 1),     # full and overfull cells side by side
])
def test_queue_equals_every_candidate(model, precision, n, side, cell, slots):
    arr = _agents(model, n, side, n)
    kw = dict(cell_size=cell, precision=precision, cell_slots=slots,
              bounds=(-4.0, -4.0, side + 4.0, side + 4.0))
    want = _run(arr, tile=(2, 2), **kw)
    for lanes in (2, 4, 16, 64):
        got = _run(arr, lanes=lanes, **kw)
        for f in ('position', 'velocity', 'force_prev'):
            assert np.array_equal(got[f], want[f]), (lanes, f)
        if model == 'three_circle':
            for f in ('orientation', 'angular_velocity', 'torque_prev'):
                assert np.array_equal(got[f], want[f]), (lanes, f)


@pytest.mark.filterwarnings('ignore')
@pytest.mark.parametrize('value', [np.nan, np.inf, 1e200])
def test_shoulders_that_are_not_finite(value):
    """A shoulder that is not finite gives its pairs in sight a NaN torque,
    also where their force is zero: the agents the oracle names, and the same
    from the queue as from every candidate."""
    n = 80
    arr = _agents('three_circle', n, 6.0, 5)
    off = 0.15 * np.stack([np.sin(arr['orientation']), -np.cos(arr['orientation'])], 1)
    arr['position_ls'], arr['position_rs'] = arr['position'] - off, arr['position'] + off
    arr['position_ls'][::13, 0] = value
    arr['position_rs'][5, 1] = value
    want = arr.copy()
    with np.errstate(all='ignore'):
        O.agent_agent_block_list(want, 3.6)
    for f in ('force', 'torque'):  # the exact sums hold terms below 2^62, a larger one is NaN
        want[f][~(np.abs(want[f]) < 2.0 ** 62)] = np.nan
    assert 0 < np.sum(np.isnan(want['torque'])) < n
    dev = DeviceAgents(arr.copy())
    core.agent_agent_block_list(dev, 3.6, Workspace(n, 64, 1, cell_slots=64))
    got = arr.copy()
    dev.download(got)
    assert np.array_equal(np.isnan(got['torque']), np.isnan(want['torque']))
    assert np.array_equal(np.isnan(got['force']), np.isnan(want['force']))
    kw = dict(cell_size=3.6, bounds=(-4.0, -4.0, 10.0, 10.0))
    every = _run(arr, 1, tile=(2, 2), **kw)
    for lanes in (2, 16):
        out = _run(arr, 1, lanes=lanes, **kw)
        for f in ('force_prev', 'torque_prev', 'orientation'):
            assert np.array_equal(out[f], every[f], equal_nan=True), (lanes, f)
