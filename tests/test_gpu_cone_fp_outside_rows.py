"""Rows of the cone FP that never meet the volume (GPU test).

A wavefront's walk limits come from a table per 64 rows: the least walk
parameter until which all of its rows are inside, and the largest at which one
leaves the volume's z range.  Waves that have left before their ray's first
segment add nothing and still scale what the output holds (y = (y + A x)
d_conv).  The detectors are several times taller than the volumes: waves that
never enter below, above or on both sides of the source, ones with a few rows
inside, and a last wave of one row.  The sums are the oracle's bit for bit, from
zero and onto an output.
"""

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from geometries import CB, centred, oracle_geom
from test_gpu_bp_paths import _geom

pytestmark = pytest.mark.gpu

A = np.linspace(0, 2 * np.pi, 11, endpoint=False) + 0.07


def _cb(nz, nv, pitch, shift=0.0, source_z=0.0):
    return CB((14, 9, nz), (1, 1, 1), A, centred(21, 1.1, 0.2), centred(nv, pitch, shift), 40.0,
              80.0, source_z=source_z)


CASES = {
    "two_slices_447": _cb(2, 447, 0.7, shift=0.2),
    "all_above": _cb(4, 193, 0.9, shift=-120.0),
    "all_below": _cb(4, 257, 0.9, shift=150.0),
    "few_inside_321": _cb(6, 321, 1.3, shift=0.4, source_z=1.1),
    "source_at_the_bottom": _cb(8, 130, 1.5, shift=0.3, source_z=-4.0),
    "source_at_the_top": _cb(8, 129, 1.5, shift=0.3, source_z=4.0),
}


@pytest.mark.parametrize("name", list(CASES))
def test_outside_rows_equal_the_oracle(name):
    from ccpi.reconstruction.projectors import forward_project
    g = CASES[name]
    print(f"\ncone FP {name} {g.shape} {g.sino_shape}", flush=True)
    rng = np.random.default_rng(47)
    x = rng.random(g.shape).astype(np.float32)
    y0 = rng.random(g.sino_shape).astype(np.float32)
    og, X = oracle_geom(g), torch.from_numpy(x).cuda()
    y = forward_project(_geom(g), X).cpu().numpy()
    assert np.array_equal(y, og.fp(x))
    assert float((y == 0).mean()) > 0.3
    acc = forward_project(_geom(g), X, torch.from_numpy(y0).cuda()).cpu().numpy()
    assert np.array_equal(acc, og.fp(x, y0.copy()))
