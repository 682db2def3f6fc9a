"""The batched CGLS's forward-projection items at their edges (GPU test).

One workgroup of the batched FP takes 64 rays of an angle, its first
wavefront walking them for four others with 1 to 8 lanes of four detector
rows per ray; problems whose rows do not go one to one with the slices keep
a wavefront per block of rays.  One batch holds each number of lanes per
ray (1 row to 40, the last in two row blocks), fewer than four slices, more
slices than rows and more rows than slices, detectors of 63, 64, 65 and 130
columns, 33 and 65 angles (one more than a tile), axis-aligned lines and a
problem of two rows per slice.  Each problem's iterates and gradient norms
are those of the one-problem CGLS, within the summation order of the step
lengths (1e-5 of the maximum, 1e-6 of the norm, as in the other batched
tests), in every order of the batch.
"""

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from geometries import PB, centred

pytestmark = pytest.mark.gpu

V1 = (1.0, 1.0, 1.0)


def _turn(n, start=0.0):
    return np.deg2rad(np.linspace(0, 180, n, endpoint=False) + start)


CASES = [
    PB((20, 24, 1), V1, _turn(33), centred(63, 0.6, 0.1), centred(1, 1.0)),
    PB((44, 45, 2), V1, _turn(65, 0.3), centred(64, 1.0, 0.3), centred(2, 1.0)),
    PB((45, 44, 7), V1, _turn(30), centred(65, 1.0), centred(7, 1.0)),
    PB((30, 31, 13), V1, _turn(36, 0.2), centred(45, 1.0, -0.2), centred(13, 1.0)),
    PB((90, 91, 17), V1, _turn(40), centred(130, 1.0, 0.21), centred(17, 1.0)),
    PB((32, 32, 40), V1, _turn(32), centred(47, 1.0), centred(40, 1.0)),
    PB((24, 20, 3), V1, _turn(28, 0.4), centred(33, 1.0), centred(20, 1.0)),
    PB((24, 20, 12), V1, _turn(28), centred(33, 1.0), centred(6, 1.0)),
    PB((20, 20, 6), V1, _turn(24), centred(30, 1.0, 0.3), centred(12, 0.5)),
]


@pytest.mark.parametrize("order", ["given", "reversed", "alone"])
def test_batched_fp_items(order):
    from ccpi.reconstruction.projectors import Geometry, cgls, cgls_batched, forward_project
    rng = np.random.default_rng(37)
    geoms = [Geometry(c.angles, c.h_pix, c.v_pix, c.origin, c.vsize, c.shape) for c in CASES]
    bs = [forward_project(G, torch.from_numpy(rng.random(c.shape).astype(np.float32)).cuda())
          for G, c in zip(geoms, CASES)]
    index = list(range(len(CASES)))
    if order == "reversed":
        index.reverse()
    print(f"\nbatched FP items, {order}", flush=True)
    if order == "alone":
        got = [[v[0] for v in cgls_batched([geoms[i]], [bs[i]], 3)] for i in index]
    else:
        got = list(zip(*cgls_batched([geoms[i] for i in index], [bs[i] for i in index], 3)))
    for i, (x, r, n) in zip(index, got):
        xp, rp, npl = cgls(geoms[i], bs[i], 3)
        scale = float(xp.abs().max())
        assert scale > 0
        assert float((x - xp).abs().max()) < 1e-5 * scale, i
        assert float((r - rp).abs().max()) < 1e-5 * float(bs[i].abs().max()), i
        assert np.allclose(n, npl, rtol=1e-6), i
