"""Launches of 2^32 threads and more (GPU test).

HIP takes fewer than 2^32 threads along one grid dimension.  The cases are
projections whose workgroups times threads pass that, at the smallest data
that get there.  The rays of one angle do not depend on the other angles, so
the first, middle and last angles have to equal, bit for bit, the projection
of a geometry of those angles alone.
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
