"""Without a given number of lanes per agent the library chooses it by the
agents and their stencil: the same bits as four lanes on either side of every
line of the rule, for one scenario and for a batch."""
import numpy as np
import pytest

from crowddynamics_amd import examples as E
from crowddynamics_amd.ensemble import Ensemble
from crowddynamics_amd.stepper import Stepper

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('precision', ['f64', 'f32'])
@pytest.mark.parametrize('n,cell', [
    (1, 3.6), (40, 0.6),
    (2048, 0.6), (2049, 0.6),      # 32 lanes in one wave per SIMD, and one agent more
    (3072, 3.6), (3073, 3.6),      # long stencils: 64 lanes in one round, then 32
    (16384, 0.6), (16385, 3.6),
    (49153, 0.6),                  # two lanes
])
def test_default_equals_four_lanes(n, cell, precision):
    scn = E.room(n=n, seed=n, width=1.5 * np.sqrt(n), height=np.sqrt(n), nav_step=0.5) if n > 100 else E.hallway(n=n, width=20.0, height=8.0)
    out = []
    for lanes in (0, 4):
        st = Stepper(scn.agents.copy(), segments=scn.segments, cell_size=cell, dt_min=0.001,
                     dt_max=0.01, seed=1, bounds=scn.bounds, precision=precision, lanes=lanes)
        st.step(2)
        out.append(st.download(scn.agents.copy()))
    for f in ('position', 'velocity', 'force_prev'):
        assert np.array_equal(out[0][f], out[1][f]), f


def test_batch_default_equals_four_lanes():
    scns = [E.hallway(n=n, width=20.0, height=10.0, seed=n) for n in (1, 17, 160, 63)]
    out = []
    for lanes in (0, 4):
        ens = Ensemble([s for s in scns], lanes=lanes)
        ens.step(2)
        out.append(ens.agents['position'].clone())
    assert bool((out[0] == out[1]).all())
