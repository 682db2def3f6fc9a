"""Turned rows of tiles of the parallel FP's shared walk (GPU test).

Four column blocks of 64, and multiples of eight, are turned from row of tiles
to row of tiles (32 angles each): every ray has to be projected, once, with a
last block that is full or holds one ray and a last row of one angle; three
and five blocks are not turned.  Against the oracle's f2D at 1e-5 of the
maximum, the summation-order tolerance of the other FP tests; the residual
after one CGLS iteration, whose step needs ||A d||^2 over every ray, at 1e-4 of
the data's maximum (1e-5 each of the step, A d and A^T b, and the data's
cancellation).
"""

import numpy as np
import pytest

torch = pytest.importorskip("torch")

import oracle
from geometries import PB, centred

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nh", [192, 193, 256, 257, 449, 512, 513, 1000])
def test_every_ray_once(nh):
    from ccpi.reconstruction.projectors import Geometry, cgls, forward_project
    na = 129
    ang = np.deg2rad(np.linspace(0, 180, na, endpoint=False) + 0.4)
    g = PB((36, 40, 18), (1.0, 1.0, 1.0), ang, centred(nh, 0.4, 0.13), centred(18, 1.0))
    # the shared walk takes 2400 wavefronts and more (18 rows: 8 lanes a ray)
    assert na * (-(-nh // 64) * 64) * 8 // 64 >= 2400
    G = Geometry(g.angles, g.h_pix, g.v_pix, g.origin, g.vsize, g.shape)
    og = oracle.Geometry(g.angles, g.h_pix, g.v_pix, g.origin, g.vsize, g.shape)
    rng = np.random.default_rng(nh)
    x = rng.random(g.shape).astype(np.float32)
    y0 = rng.random(g.sino_shape).astype(np.float32)
    print(f"\nparallel FP, {nh} columns", flush=True)
    want = og.fp(x, y0.copy())
    y = forward_project(G, torch.from_numpy(x).cuda(), torch.from_numpy(y0).cuda())
    assert np.abs(y.cpu().numpy() - want).max() < 1e-5 * np.abs(want).max()
    b = og.fp(x)
    d = og.bp(b).astype(np.float64)
    ad = og.fp(d.astype(np.float32)).astype(np.float64)
    r1 = b - ad * ((d ** 2).sum() / (ad ** 2).sum())
    _, r, _ = cgls(G, torch.from_numpy(b).cuda(), 1)
    assert np.abs(r.cpu().numpy() - r1).max() < 1e-4 * np.abs(b).max()
