"""Which parallel plans of one row per slice hold a walk table (GPU test).

Below 2400 wavefronts all do, with up to 8 lanes on a ray's cells (volumes of nx
+ ny up to 64 cells fewer: 1, 2 and 4 here); up to 8192 those of short rays (a harmonic mean of
nx and ny up to 32 cells) with more than 32 rows.  The plan's bytes show the
table (8 bytes per cell of every ray); the projection is the oracle's within
1e-5 of the maximum, as for the other FP forms, from zero and onto an output.
"""

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from ccpi.reconstruction import projectors as J
from geometries import PB, centred, oracle_geom
from test_gpu_par_fp_forms import _geom, _waves

pytestmark = pytest.mark.gpu


def _pb(nx, ny, nz, na, nh):
    ang = np.r_[0.0, np.pi / 2, np.linspace(0, np.pi, na, endpoint=False) + 0.01]
    return PB((nx, ny, nz), (1, 1, 1), ang, centred(nh, 1.0, 0.2), centred(nz, 1.0))


# geometry, wavefronts at least and below, whether a table is held
CASES = {
    "few_waves": (_pb(64, 64, 40, 60, 91), (1, 2400), True),
    "few_cells_one_lane": (_pb(20, 21, 40, 290, 31), (2050, 2400), True),
    "few_cells_two_lanes": (_pb(20, 20, 32, 250, 50), (1025, 2049), True),
    "few_cells_four_lanes": (_pb(25, 25, 36, 142, 25), (513, 1025), True),
    "short_33_rows": (_pb(32, 32, 33, 170, 70), (2400, 8192), True),
    "short_130_rows": (_pb(29, 35, 130, 90, 60), (2400, 8192), True),
    "short_long_side": (_pb(16, 700, 40, 90, 120), (2400, 8192), True),
    "short_32_rows": (_pb(31, 31, 32, 300, 80), (2400, 8192), False),
    "longer": (_pb(32, 33, 33, 170, 70), (2400, 8192), False),
    "many_waves": (_pb(31, 31, 70, 220, 80), (8192, 1 << 20), False),
}


@pytest.mark.parametrize("name", list(CASES))
def test_walk_table(name):
    g, waves, held = CASES[name]
    assert waves[0] <= _waves(g) < waves[1]
    J.plan_cache_clear()
    print(f"\nparallel FP {name} {g.shape} {g.sino_shape} {_waves(g)} waves", flush=True)
    rng = np.random.default_rng(53)
    x = rng.random(g.shape).astype(np.float32)
    y0 = rng.random(g.sino_shape).astype(np.float32)
    X = torch.from_numpy(x).cuda()
    y = J.forward_project(_geom(g), X).cpu().numpy()
    # at least 4 cells per ray on average; the other tables are far smaller
    assert (J.plan_cache_bytes() > 4 * 8 * len(g.angles) * len(g.h_pix)) == held
    yo = oracle_geom(g).fp(x)
    scale = np.abs(yo).max()
    assert scale > 0 and np.abs(y - yo).max() < 1e-5 * scale
    ya = J.forward_project(_geom(g), X, torch.from_numpy(y0).cuda()).cpu().numpy()
    assert np.abs(ya - oracle_geom(g).fp(x, y0.copy())).max() < 1e-5 * scale
    J.plan_cache_clear()
