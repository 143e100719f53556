"""The distance map at grid steps on either side of the range in which the
relaxation's own square root serves: a step of 2^k scales the map by 2^k."""
import numpy as np
import pytest

from crowddynamics_amd import field as F
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('k', [-480, -371, -370, -3, 0, 490, 491, 495])
def test_distance_map_scales(k):
    rng = np.random.default_rng(3)
    rows, cols = 40, 75
    phi = np.full((rows, cols), -1.0)
    phi[3:6, 2] = 1.0
    mask = rng.uniform(size=phi.shape) < 0.2
    mask &= phi < 0
    step = 2.0 ** k
    mg = F.meshgrid(step, 0.0, 0.0, step * (cols - 1.5), step * (rows - 1.5))
    assert mg.shape == phi.shape
    got = F.FieldBuilder(mg).distance_map(phi, mask).cpu().numpy() / step
    want = O.distance_map(phi, 1.0, mask)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    ok = ~np.isnan(want)
    # a rounding per node of the path from the target, on either side
    bound = 2.0 * (rows * cols) * np.finfo(float).eps * np.abs(want[ok]).max()
    assert np.abs(got[ok] - want[ok]).max() <= bound
