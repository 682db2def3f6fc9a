"""The centre search's sequential sum at its edges (GPU test).

The device adds the terms of a candidate in chunks of 2048, four at a time:
term counts of every remainder by 4, below, at and above one and two chunks.
The chosen centre on rows of noise is the oracle's, bit for bit.
"""

import numpy as np
import pytest

torch = pytest.importorskip("torch")

import oracle
from test_gpu_centre import _device_centre

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("na,nh", [(7, 9), (5, 13), (13, 10), (46, 44), (64, 32), (23, 89),
                                   (41, 50), (63, 65), (45, 91), (64, 64), (17, 241)])
def test_find_centre_term_counts(na, nh):
    from ccpi.reconstruction import instruments as ins
    ang = np.linspace(0, 360, na, endpoint=False).astype(np.float32)
    setup = ins.xtek_setup((na, nh, 4), ang, 1, -500.0, 500.0, 1.0, 1.0, 60.0)
    g = setup.geometry
    og = oracle.Geometry(g.angles, g.h_pixels, g.v_pixels, g.origin, g.voxel_size, g.shape,
                         cone=True, source=g.source, det_x=g.detector_x)
    y = np.random.default_rng(na * nh).random(g.sino_shape).astype(np.float32)
    print(f"\nfind_centre {na} x {nh} = {na * nh} terms", flush=True)
    want, _ = oracle.find_centre(og, y, 2)
    got, _ = _device_centre(og, y, 2)
    assert got == want
