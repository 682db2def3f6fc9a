"""Every row and ray split of the cone forward projector against the oracle
(GPU test).

The FP takes a ray's rows in wavefronts of 64 (workgroups of 1 to 4 of
them), its segments 8 at a time, the ones inside the volume by a path without
clamps or range checks, and its rays in tiles of up to 64 angles x 8 columns
per XCD; volumes of 4 GiB and more keep column indices instead of byte
offsets in the ray table.  The sizes below meet the edges of these: 64 and 65
rows, a wavefront with rows on both sides of the source, 257 rows (two
workgroups), one angle, 65 angles (two tiles), 9 columns, rays of fewer than
8 segments, a volume lower than its shadow (rows that leave through the
faces: the floor form), a source near the volume's top.

Weights and summation order are the oracle's, so the results are equal bit
for bit; the FP64-accumulation option is checked through MLEM in
test_gpu_accum_fp64.py.
"""

import numpy as np
import pytest

torch = pytest.importorskip("torch")

import oracle
from geometries import CB, centred

pytestmark = pytest.mark.gpu


def _cb(shape, na, nh, nv, vox=1.0, sod=60.0, source_z=0.0, pitch=1.1, vshift=0.0):
    ang = np.linspace(0, 2 * np.pi, na, endpoint=False) + 0.05
    return CB(shape, (vox, vox, vox), ang, centred(nh, pitch), centred(nv, pitch, vshift), sod,
              2 * sod, source_z=source_z)


CASES = {
    "rows64": _cb((20, 18, 24), 7, 30, 64),
    "rows65_mixed_wave": _cb((20, 18, 24), 7, 30, 65, vshift=0.3),
    "rows100_mixed_wave": _cb((24, 24, 40), 5, 40, 100),
    "rows257_two_blocks": _cb((16, 16, 100), 3, 24, 257, pitch=0.7, vshift=0.2),
    "one_angle": _cb((32, 32, 32), 1, 50, 70),
    "angles65": _cb((12, 12, 12), 65, 9, 20),
    "short_rays": _cb((3, 4, 10), 9, 8, 16),
    "low_volume": _cb((30, 30, 9), 6, 44, 130, sod=40.0),
    "source_near_top": _cb((20, 20, 20), 6, 30, 66, source_z=9.3, vshift=-0.4),
}


def _check(g, x):
    from ccpi.reconstruction.projectors import Geometry, forward_project
    G = Geometry(g.angles, g.h_pix, g.v_pix, g.origin, g.vsize, g.shape, cone=True,
                 source=g.source, detector_x=g.det_x)
    og = oracle.Geometry(g.angles, g.h_pix, g.v_pix, g.origin, g.vsize, g.shape, cone=True,
                         source=g.source, det_x=g.det_x)
    y = forward_project(G, torch.from_numpy(x).cuda()).cpu().numpy()
    yo = og.fp(x)
    assert float(np.abs(yo).max()) > 0
    assert np.array_equal(y, yo)


@pytest.mark.parametrize("name", list(CASES))
def test_fp_paths_equal_the_oracle(name):
    g = CASES[name]
    print(f"\ncone FP {name} {g.shape} {g.sino_shape}", flush=True)
    _check(g, np.random.default_rng(31).random(g.shape).astype(np.float32))


def test_fp_volume_past_4_gib():
    g = _cb((1025, 1024, 1024), 2, 12, 70, vox=0.05)
    print(f"\ncone FP {g.shape}", flush=True)
    x = np.random.default_rng(32).random(g.shape, dtype=np.float32)
    _check(g, x)
