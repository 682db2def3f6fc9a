"""Parallel-beam CGLS with the step lengths summed in the updates (GPU test).

Problems of fewer than 2^20 voxels and pixels sum the norm partials in the
update kernels; the others, and the regularised form, in kernels of one
workgroup.  With lambda = 0 the regularised form is the plain one bit for
bit, so it is the other route: sizes of one workgroup's work, odd ones, just
below and at the limit, in one call, and as a session of single steps.
"""

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from geometries import PB, centred

pytestmark = pytest.mark.gpu

V1 = (1.0, 1.0, 1.0)


def _case(nx, ny, nz, na, nh, nv):
    return PB((nx, ny, nz), V1, np.linspace(0, np.pi, na, endpoint=False) + 0.01,
              centred(nh, 1.0, 0.21), centred(nv, 1.0))


CASES = {"tiny": _case(5, 4, 2, 7, 9, 2), "odd": _case(33, 61, 5, 40, 71, 5),
         "below": _case(128, 127, 64, 20, 181, 64), "at": _case(128, 128, 64, 20, 181, 64),
         "pixels_at": _case(24, 24, 64, 128, 128, 64)}


@pytest.mark.parametrize("name", list(CASES))
def test_sum_updates_same_bits(name):
    from ccpi.reconstruction.projectors import (CglsSession, Geometry, TIKHONOV, cgls, cgls_reg)
    c = CASES[name]
    G = Geometry(c.angles, c.h_pix, c.v_pix, c.origin, c.vsize, c.shape)
    rng = np.random.default_rng(47)
    b = torch.from_numpy(rng.random(c.sino_shape).astype(np.float32)).cuda()
    print(f"\nCGLS sums in updates {name}", flush=True)
    x, r, n = cgls(G, b, 4)
    xr, rr, nr = cgls_reg(G, b, 4, TIKHONOV, 0.0)
    assert torch.equal(x, xr) and torch.equal(r, rr) and np.array_equal(n, nr)
    xs = torch.zeros_like(x)
    s = CglsSession(G, b.clone(), xs, 4)
    for _ in range(4):
        s.iterate(1)
    assert np.array_equal(s.norms(), n) and torch.equal(xs, x)
    s.close()
    x0, _, n0 = cgls(G, torch.zeros_like(b), 2)
    assert torch.count_nonzero(x0) == 0 and np.all(n0 == 0)
