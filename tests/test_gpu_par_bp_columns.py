"""The tiled parallel-beam backprojector's two-column form (GPU test).

On evenly spaced columns, at angles where a voxel's shadow is under two
columns wide, the tiled BP weighs the two columns after the shadow's start
without a loop.  The cases lie about that rule's lines: pixels whose widest
shadow is just under, at and over two columns; columns that are not even (by
1e-3 and by 5e-8 of a pixel); lines within 1e-7 to 1e-3 of an axis; a
detector that starts or ends inside the volume's shadow; rows of inactive
lanes (ragged tiles); and voxels that are not square.  Against the oracle's
b2D at 1e-5 of the maximum, as the other BP tests.
"""

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from geometries import PB, centred, oracle_geom

pytestmark = pytest.mark.gpu

V1 = (1.0, 1.0, 1.0)


def _turn(n, start=0.0):
    return np.deg2rad(np.linspace(0, 360, n, endpoint=False) + start)


def _uneven(n, pitch, by):
    h = centred(n, pitch, 0.2)
    return h + by * pitch * np.random.default_rng(5).uniform(-1, 1, n)


NEAR = np.array([0.0, 0.5, 1.0, 1.5])[:, None] * np.pi + \
    np.array([-1e-3, -1e-5, -3e-7, -1.3e-7, -1e-7, 1e-7, 1.3e-7, 3e-7, 1e-5, 1e-3])[None, :]
CASES = {
    "under_two": PB((33, 35, 16), V1, _turn(72, 0.0), centred(70, np.sqrt(2) / 1.985, 0.1),
                    centred(16, 1.0)),
    "two": PB((33, 35, 16), V1, _turn(72, 0.0), centred(70, np.sqrt(0.5), 0.1),
              centred(16, 1.0)),
    "over_two": PB((33, 35, 9), V1, _turn(72, 0.0), centred(72, 0.69, 0.1), centred(9, 1.0)),
    "uneven": PB((34, 30, 8), V1, _turn(50, 0.3), _uneven(50, 1.0, 1e-3), centred(8, 1.0)),
    "nearly_even": PB((34, 30, 8), V1, _turn(50, 0.3), _uneven(50, 1.0, 5e-8), centred(8, 1.0)),
    "near_axes": PB((34, 37, 12), V1, NEAR.ravel(), centred(56, 1.0, 0.37), centred(12, 1.0)),
    "starts_inside": PB((40, 40, 16), V1, _turn(60, 0.1), np.arange(30) - 7.3, centred(16, 1.0)),
    "ends_inside": PB((40, 40, 16), V1, _turn(60, 0.1), np.arange(30) - 25.6, centred(16, 1.0)),
    "ragged": PB((17, 49, 13), V1, _turn(45, 0.2), centred(58, 1.0, -0.3), centred(13, 1.0)),
    "finest_16": PB((17, 18, 12), V1, _turn(20, 0.3), centred(570, 0.0453, 0.01),
                    centred(12, 1.0)),
    "finest_8": PB((17, 18, 8), V1, _turn(14, 0.3), centred(1160, 0.0223, 0.01),
                   centred(8, 1.0)),
    "not_square": PB((24, 40, 16), (1.3, 0.6, 1.0), _turn(60, 0.4), centred(46, 0.9, 0.1),
                     centred(16, 1.0)),
}


@pytest.mark.parametrize("name", list(CASES))
def test_two_column_form(name):
    from ccpi.reconstruction.projectors import Geometry, backward_project
    g = CASES[name]
    G = Geometry(g.angles, g.h_pix, g.v_pix, g.origin, g.vsize, g.shape)
    s = np.random.default_rng(43).random(g.sino_shape).astype(np.float32)
    print(f"\ntiled parallel BP columns {name}", flush=True)
    want = oracle_geom(g).bp(s)
    b = backward_project(G, torch.from_numpy(s).cuda()).cpu().numpy()
    assert np.abs(b - want).max() < 1e-5 * np.abs(want).max()
