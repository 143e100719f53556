"""The distance map at the edges of its tiles (32 x 32 nodes) and on grids the
front must cross several times, and the nearest-direction fill, whose rings
must give the row-major first of equal distances."""
import numpy as np
import pytest
import torch

from crowddynamics_amd import field as F
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _grid(rows, cols, step=0.5):
    mg = F.meshgrid(step, 0.0, 0.0, step * (cols - 1) - 0.5 * step, step * (rows - 1) - 0.5 * step)
    assert mg.shape == (rows, cols)
    return mg


def _serpentine(rows, cols):
    """Masked walls with a gap at alternating ends: the longest path."""
    mask = np.zeros((rows, cols), dtype=bool)
    for k, r in enumerate(range(4, rows - 2, 5)):
        mask[r] = True
        mask[r, (slice(0, 2) if k % 2 else slice(cols - 2, cols))] = False
    return mask


@pytest.mark.parametrize('rows,cols,masked', [
    (2, 2, False), (2, 70, False), (31, 33, False), (32, 32, False), (33, 32, True),
    (65, 64, True), (97, 40, True), (64, 193, False),
])
def test_distance_map_tiles(rows, cols, masked):
    mg = _grid(rows, cols)
    phi = np.full((rows, cols), -1.0)
    phi[0, 0] = 1.0
    mask = _serpentine(rows, cols) if masked else None
    got = F.FieldBuilder(mg).distance_map(phi, mask).cpu().numpy()
    want = O.distance_map(phi, mg.step, mask)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    ok = ~np.isnan(want)
    # both reach the fixed point of the same update; a rounding per node of
    # the path from the target
    bound = 2.0 * (rows * cols) * np.finfo(float).eps * np.abs(want[ok]).max()
    assert np.abs(got[ok] - want[ok]).max() <= bound


@pytest.mark.parametrize('reach', [0, 1, 4, 9])
def test_fill_takes_the_first_of_the_nearest(reach):
    rng = np.random.default_rng(reach)
    rows, cols = 37, 41
    ex = rng.normal(size=(rows, cols))
    ey = rng.normal(size=(rows, cols))
    ex[rng.uniform(size=(rows, cols)) < 0.8] = np.nan
    ey[rng.uniform(size=(rows, cols)) < 0.3] = np.nan
    ex[10:22, 15:30] = np.nan  # a hole wider than a ring
    fill = rng.uniform(size=(rows, cols)) < 0.9
    fb = F.FieldBuilder(_grid(rows, cols))
    ox, oy = fb.fill_missing(torch.as_tensor(ex, device='cuda'), torch.as_tensor(ey, device='cuda'),
                             fill, reach)
    have = ~(np.isnan(ex) | np.isnan(ey))
    wx, wy = ex.copy(), ey.copy()
    for r, c in zip(*np.nonzero(fill & ~have)):
        r0, c0 = max(0, r - reach), max(0, c - reach)
        rr, cc = np.nonzero(have[r0:r + reach + 1, c0:c + reach + 1])
        if len(rr):
            k = np.argmin((rr + r0 - r) ** 2 + (cc + c0 - c) ** 2)
            wx[r, c], wy[r, c] = ex[rr[k] + r0, cc[k] + c0], ey[rr[k] + r0, cc[k] + c0]
    assert np.array_equal(ox.cpu().numpy(), wx, equal_nan=True)
    assert np.array_equal(oy.cpu().numpy(), wy, equal_nan=True)


@pytest.mark.parametrize('rows,cols,every,reach', [
    (37, 41, 0, 1024),   # no direction anywhere, squares far beyond the grid
    (37, 41, 13, 1024),  # few, whose distances tie
    (3, 300, 90, 200),
    (300, 3, 90, 200),
    (40, 60, 12, 5),     # nodes with none within reach beside ones with four
    (40, 60, 9, 8),
])
def test_fill_reaches_past_the_nearest_square(rows, cols, every, reach):
    ex = np.full((rows, cols), np.nan)
    if every:
        at = ex[every // 3::every, every // 3::every]
        at[...] = 1.0 + np.arange(at.size).reshape(at.shape)
        ex[0, -1] = -1.0
    fb = F.FieldBuilder(_grid(rows, cols))
    t = torch.as_tensor(ex, device='cuda')
    ox, oy = fb.fill_missing(t, 2.0 * t, np.ones((rows, cols), dtype=bool), reach)
    have = np.argwhere(~np.isnan(ex))  # row-major
    want = ex.copy()
    for r, c in np.argwhere(np.isnan(ex)):
        d = have - (r, c)
        near = (np.abs(d) <= reach).all(1)
        if near.any():
            k = np.flatnonzero(near)[np.argmin((d[near] ** 2).sum(1))]
            want[r, c] = ex[tuple(have[k])]
    assert np.array_equal(ox.cpu().numpy(), want, equal_nan=True)
    assert np.array_equal(oy.cpu().numpy(), 2.0 * want, equal_nan=True)
