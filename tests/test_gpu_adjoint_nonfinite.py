"""An adjoint that is not finite reaches every agent in sight of its own, on a
collision course or not, and no other: a zero derivative times NaN is NaN.
The step after it, with finite adjoints, is as if it had not been."""
import numpy as np
import pytest
import torch

from crowddynamics_amd import examples as E
from crowddynamics_amd.adjoint import Rollout

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('lanes', [2, 16, 64])
@pytest.mark.parametrize('bad', [np.nan, np.inf])
def test_nonfinite_adjoint_reaches_those_in_sight(lanes, bad):
    rng = np.random.default_rng(8)
    n, cell = 120, 3.6
    arr = E._attributes(rng, n)
    arr['position'] = rng.uniform(0.0, 14.0, (n, 2))
    arr['velocity'] = rng.normal(0.0, 0.5, (n, 2))
    arr['target_direction'] = (1.0, 0.0)
    arr['target'] = 0
    R = Rollout(arr, steps=1, dt=0.005, cell_size=cell, lanes=lanes)
    R.agents.upload(arr)
    lam = {k: torch.as_tensor(rng.normal(0.0, 1.0, (n, 2)), device='cuda')
           for k in ('lam_x', 'lam_v', 'lam_g')}

    def step(first):
        for k in lam:
            R.adj[k].copy_(lam[k])
        R.adj['lam_g'][5] = first
        R.grad.zero_()
        R.adjoint_step(torch.zeros((n, 2), dtype=torch.float64, device='cuda'))
        return R.adj['lam_x'].cpu().numpy()

    clean = step(0.25)
    got = step(bad)
    x, r = arr['position'], arr['radius']
    near = np.hypot(*(x - x[5]).T) - r - r[5] < 3.0
    box = np.abs(np.trunc((x - x.min(0)) / cell) - np.trunc((x[5] - x.min(0)) / cell)).max(1) <= 1
    assert np.array_equal(np.isnan(got).any(1), near & box)
    assert np.array_equal(step(0.25), clean)
