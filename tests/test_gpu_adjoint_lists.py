"""The adjoint's pair lists: agents whose lists fill several times, cells
holding more agents than slots, and agents with nobody near, against torch
autograd of the dense step, at every number of lanes."""
import numpy as np
import pytest
import torch

from crowddynamics_amd import examples as E
from crowddynamics_amd.adjoint import Rollout, rollout_positions
from tests import dense_reference as D

pytestmark = pytest.mark.gpu

DT = 0.005


def _crowd(n, side, seed):
    rng = np.random.default_rng(seed)
    arr = E._attributes(rng, n)
    arr['position'] = rng.uniform(0.0, side, (n, 2))
    arr['position'][0] = (side + 30.0, side + 30.0)  # nobody near
    arr['velocity'] = rng.normal(0.0, 0.5, (n, 2))
    arr['force_prev'] = rng.normal(0.0, 50.0, (n, 2))
    arr['target_direction'] = (1.0, 0.0)
    arr['target'] = 0
    return arr


@pytest.mark.filterwarnings('ignore')
@pytest.mark.parametrize('n,side,cell', [
    (1, 1.0, 3.6),
    (2, 0.3, 0.6),     # one pair
    (150, 4.0, 3.6),   # each agent on course with dozens: lists fill again and again
    (400, 3.0, 3.6),   # more agents in a cell than its slots
    (90, 9.0, 3.6),
])
def test_step_equals_dense_autograd(n, side, cell):
    arr = _crowd(n, side, n)
    rng = np.random.default_rng(5)
    lam = {k: torch.as_tensor(rng.normal(0.0, 1.0, (n, 2))) for k in ('lam_x', 'lam_v', 'lam_g')}
    x, v, fp = (torch.as_tensor(np.array(arr[f])).requires_grad_(True)
                for f in ('position', 'velocity', 'force_prev'))
    p = [torch.full((n,), c, dtype=torch.float64).requires_grad_(True)
         for c in (3.0, 1.2e5, 4e4, 500.0)]
    p.append(torch.as_tensor(np.array(arr['target_velocity'])).requires_grad_(True))
    x1, v1, F = D.step(x, v, fp, D.constants(arr), DT, cell, *p)
    ((lam['lam_x'] * x1).sum() + (lam['lam_v'] * v1).sum() + (lam['lam_g'] * F).sum()).backward()
    want = {'lam_x': x.grad, 'lam_v': v.grad, 'lam_g': fp.grad}
    for lanes in (2, 4, 16, 64):
        R = Rollout(arr, steps=1, dt=DT, cell_size=cell, lanes=lanes,
                    bounds=(-1.0, -1.0, side + 31.0, side + 31.0))
        q = [t.detach() for t in p]
        R.set_parameters(*q)
        R.agents.upload(arr)
        R.set_parameters(*q)
        for k in lam:
            R.adj[k].copy_(lam[k])
        R.grad.zero_()
        R.adjoint_step(torch.zeros((n, 2), dtype=torch.float64, device='cuda'))
        # a pair's derivatives lose b^2 / (b^2 - a c), and the least
        # discriminant of n^2 random pairs is about b^2 / n^2; a few dozen
        # operations each
        tol = max(1e-11, 64 * 2.0**-53 * n * n)
        for k in want:
            err = float((R.adj[k].cpu() - want[k]).abs().max())
            assert err <= tol * float(want[k].abs().max()), (lanes, k, err)
        for c, t in enumerate(p):
            err = float((R.grad[:, c].cpu() - t.grad).abs().max())
            assert err <= 10 * tol * float(t.grad.abs().max()) + 1e-300, (lanes, c, err)


@pytest.mark.filterwarnings('ignore')
@pytest.mark.parametrize('n,side,lanes', [(150, 4.0, 2), (150, 4.0, 4), (150, 4.0, 16),
                                          (400, 5.0, 2), (400, 3.0, 4)])
def test_lists_that_fill_keep_the_bits(n, side, lanes):
    """Which agents share a wave, and so when a wave works its lists off, does
    not touch an agent's gradient: agents in index order, in cell order and in
    the order of every third step give the same bits."""
    arr = _crowd(n, side, n)
    gen = torch.Generator().manual_seed(n + lanes)
    w = torch.randn((5, n, 2), dtype=torch.float64, generator=gen).cuda()
    out = []
    for every in (0, 1, 3):
        R = Rollout(arr, steps=4, dt=DT, cell_size=3.6, lanes=lanes, order_every=every,
                    bounds=(-1.0, -1.0, side + 31.0, side + 31.0))
        p = [torch.full((n,), c, dtype=torch.float64, device='cuda').requires_grad_(True)
             for c in (3.0, 1.2e5, 4e4, 500.0)]
        p.append(torch.as_tensor(np.array(arr['target_velocity']), device='cuda')
                 .requires_grad_(True))
        out.append(torch.autograd.grad(rollout_positions(R, *p), p, w))
    for g in out[1:]:
        for a, b in zip(g, out[0]):
            assert torch.equal(a, b)
