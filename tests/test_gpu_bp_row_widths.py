"""Rows per lane of the phased cone backprojector (GPU test).

The phased form gives a lane as many detector rows (1, 2, 3, 4, 6, 8, 12 or
16, at most the layout's) as cover the detector in one block of 64 lanes, in
as many lane phases as keep a round's lanes on distinct slices.  The cases
take the last row count of each width and the first of the next, a source
below the volume's middle (both row-set forms in one block), and a nearer
source with more phases.  Against the oracle's b2D at 1e-5 of the maximum
and by the adjoint identity, as the other BP path tests.
"""

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from geometries import CB, centred, oracle_geom
from test_gpu_bp_paths import _geom, _rel

pytestmark = pytest.mark.gpu

A10 = np.linspace(0, 2 * np.pi, 10, endpoint=False) + 0.05
ROWS = [63, 64, 65, 128, 129, 192, 193, 256, 257, 384, 385, 513]


@pytest.mark.parametrize("near", [False, True])
@pytest.mark.parametrize("rows", ROWS)
def test_phased_row_widths(rows, near):
    from ccpi.reconstruction import _lib
    from ccpi.reconstruction.projectors import backward_project, forward_project
    import ctypes as C
    pitch = 0.25 if near else 0.4
    sod = 24.0 if near else 40.0
    nz = max(4, int(rows * pitch * 0.45))
    g = CB((12, 10, nz), (1, 1, 1), A10, centred(18, 1.6), centred(rows, pitch, 0.1 * pitch), sod,
           2 * sod, source_z=0.013 - 0.2 * nz if near else 0.03)
    G = _geom(g)
    out = [C.c_int() for _ in range(4)]
    _lib.check(_lib.lib().ccpi_cone_bp_layout(C.byref(G.c_struct()), *[C.byref(q) for q in out]))
    assert out[1].value == 1
    og = oracle_geom(g)
    rng = np.random.default_rng(rows)
    print(f"\nphased BP rows={rows} near={near} layout={[q.value for q in out]}", flush=True)
    x = rng.random(g.shape).astype(np.float32)
    s = rng.random(g.sino_shape).astype(np.float32)
    y = forward_project(G, torch.from_numpy(x).cuda()).cpu().numpy()
    b = backward_project(G, torch.from_numpy(s).cuda()).cpu().numpy()
    assert _rel(b, og.bp(s)) < 1e-5
    lhs = float(np.vdot(y.astype(np.float64), s))
    rhs = float(np.vdot(x.astype(np.float64), b))
    assert abs(lhs - rhs) < 1e-5 * abs(lhs)
