"""Launches of 2^32 threads and more (GPU test).

HIP takes fewer than 2^32 threads along one grid dimension.  The cases are
projections whose workgroups times threads pass that, at the smallest data
that get there.  The rays of one angle do not depend on the other angles, so
the first, middle and last angles have to equal, bit for bit, the projection
of a geometry of those angles alone; the problems of a batch are checked
against the one-problem CGLS, within the tolerances of the other batched tests.
"""

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from ccpi.reconstruction import projectors as J
from geometries import centred

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _memory_back():
    yield
    J.plan_cache_clear()
    torch.cuda.empty_cache()


def _check(geom, x):
    y = J.forward_project(geom(slice(None)), x)
    na = y.shape[0]
    for part in (slice(0, 3), slice(na // 2, na // 2 + 3), slice(na - 3, na)):
        want = J.forward_project(geom(part), x)
        assert float(want.abs().max()) > 0
        assert torch.equal(y[part], want)
    # no angle was left out
    assert bool((y.reshape(na, -1).amax(1) > 0).all())


def test_cone_fp_of_2_32_pixels():
    na, nh, nv = 257, 2048, 8192
    ang = np.linspace(0, 2 * np.pi, na, endpoint=False) + 0.05
    h, v = centred(nh, 0.01, 0.002), centred(nv, 0.005)
    print(f"\ncone FP {na} x {nh} x {nv}", flush=True)

    def geom(part):
        return J.Geometry(ang[part], h, v, (-4, -4, -8), (1, 1, 1), (8, 8, 16), cone=True,
                          source=(-40.0, 0.0, 0.0), detector_x=40.0)
    x = torch.rand(8, 8, 16, generator=torch.Generator().manual_seed(3)).cuda() + 0.1
    _check(geom, x)


def test_parallel_fp_of_2_32_threads():
    # 64 rays a workgroup of 576 threads: two columns fill it least
    na, nh, nv = 7_460_001, 2, 33
    ang = np.linspace(0, np.pi, na, endpoint=False) + 0.01
    h, v = centred(nh, 1.0, 0.1), centred(nv, 1.0)
    print(f"\nparallel FP {na} x {nh} x {nv}", flush=True)

    def geom(part):
        return J.Geometry(ang[part], h, v, (-1, -1, -nv / 2), (1, 1, 1), (2, 2, nv))
    _check(geom, torch.rand(2, 2, nv, generator=torch.Generator().manual_seed(4)).cuda() + 0.1)


def test_batch_of_2_32_fp_threads():
    # 64 rays and 32 rows a workgroup of 320 threads; the two-columns problems
    # of 33 rows fill them least
    na, nh, nv, count = 105_001, 2, 33, 64
    print(f"\nbatched CGLS {count} x {na} x {nh} x {nv}", flush=True)
    geoms, bs = [], []
    for q in range(count):
        ang = np.linspace(0, np.pi, na, endpoint=False) + 0.001 * (q + 1)
        geoms.append(J.Geometry(ang, centred(nh, 1.0, 0.1), centred(nv, 1.0),
                                (-1, -1, -nv / 2), (1, 1, 1), (2, 2, nv)))
        x = torch.rand(2, 2, nv, generator=torch.Generator().manual_seed(q)).cuda() + 0.1
        bs.append(J.forward_project(geoms[-1], x))
    xs, rs, norms = J.cgls_batched(geoms, bs, 1)
    for q in (0, 31, count - 1):
        x, r, n = J.cgls(geoms[q], bs[q], 1)
        assert float(x.abs().max()) > 0
        assert float((xs[q] - x).abs().max()) < 1e-5 * float(x.abs().max())
        assert float((rs[q] - r).abs().max()) < 1e-5 * float(bs[q].abs().max())
        assert np.allclose(norms[q], n, rtol=1e-6)
