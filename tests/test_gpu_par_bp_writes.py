"""What the tiled parallel-beam backprojector writes, slice count by slice
count (GPU test).

A lane of the tiled BP writes its 8 or 16 slices in groups of four where the
group has its detector rows, else one by one; the cases reach every remainder
of a group and of a lane's slices, detectors with fewer rows and with more
rows than slices, and both launches: few angles on a volume of many tiles
(one group, written straight into the volume, added to what it holds or over
zeros) and more angles on few tiles (groups, added up by a second kernel).
The volume starts one float into its allocation, so that no group is 16-byte
aligned, and the floats on both sides of it stay as they were.  Against the
oracle's b2D at 1e-5 of the maximum, the summation-order tolerance of the
other BP tests.
"""

import numpy as np
import pytest

torch = pytest.importorskip("torch")

import oracle
from geometries import PB, centred

pytestmark = pytest.mark.gpu

V1 = (1.0, 1.0, 1.0)


@pytest.mark.parametrize("rows", [-2, 0, 3])
@pytest.mark.parametrize("nz", list(range(1, 21)) + [31, 32, 35])
def test_slices_of_every_count(nz, rows):
    from ccpi.reconstruction.projectors import Geometry, backward_project
    nv = max(1, nz + rows)
    for nx, ny, na in ((19, 35, 3), (17, 15, 41)):
        ang = np.deg2rad(np.linspace(0, 180, na, endpoint=False) + 0.7)
        g = PB((nx, ny, nz), V1, ang, centred(49, 1.0, 0.3), centred(nv, 1.0))
        G = Geometry(g.angles, g.h_pix, g.v_pix, g.origin, g.vsize, g.shape)
        og = oracle.Geometry(g.angles, g.h_pix, g.v_pix, g.origin, g.vsize, g.shape)
        rng = np.random.default_rng(100 * nz + nv)
        s = rng.random(g.sino_shape).astype(np.float32)
        print(f"\ntiled parallel BP writes {g.shape} nv {nv} na {na}", flush=True)
        for x0 in (np.zeros(g.shape, np.float32), rng.random(g.shape).astype(np.float32)):
            buf = torch.full((x0.size + 9,), -7.0, device="cuda")
            out = buf[1:1 + x0.size].view(g.shape)
            out.copy_(torch.from_numpy(x0))
            backward_project(G, torch.from_numpy(s).cuda(), out)
            want = og.bp(s, x0.copy())
            got = out.cpu().numpy()
            assert np.abs(got - want).max() <= 1e-5 * np.abs(want).max()
            assert (buf[:1].cpu() == -7.0).all() and (buf[1 + x0.size:].cpu() == -7.0).all()
