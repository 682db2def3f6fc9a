"""SIRT and MLEM with the cone BP's input scaled where it is formed (GPU
test).

The residual (SIRT) and the ratio (MLEM) go straight into the BP's scaled,
padded rows: rows shorter than a workgroup (several rays at a time), longer
than one, odd, and one that fills its padding.  Five iterations against the
oracle at 1e-4 of the maximum, as the other SIRT and MLEM tests.
"""

import numpy as np
import pytest

torch = pytest.importorskip("torch")

import oracle
from geometries import CB, centred, ellipsoid_phantom, oracle_geom
from test_gpu_bp_paths import _geom, _rel

pytestmark = pytest.mark.gpu

A = np.linspace(0, 2 * np.pi, 17, endpoint=False) + 0.1


@pytest.mark.parametrize("rows,pitch", [(7, 3.0), (64, 1.4), (75, 1.0), (300, 1.0), (128, 0.4)])
def test_sirt_mlem_scaled_rows(rows, pitch):
    from ccpi.reconstruction.projectors import mlem, sirt
    nz = max(4, int(rows * pitch * 0.45))
    g = CB((14, 12, nz), (1, 1, 1), A, centred(23, 1.5), centred(rows, pitch, 0.25 * pitch), 40.0,
           80.0)
    og = oracle_geom(g)
    b = og.fp(ellipsoid_phantom(g.shape, g.vsize, g.origin, 4, seed=rows))
    print(f"\nscaled rows {rows}", flush=True)
    xs = sirt(_geom(g), torch.from_numpy(b).cuda(), 5)
    assert _rel(xs.cpu().numpy(), oracle.sirt(og, b, 5)) < 1e-4
    xm = mlem(_geom(g), torch.from_numpy(b).cuda(), 5)
    assert _rel(xm.cpu().numpy(), oracle.mlem(og, b, 5)) < 1e-4
