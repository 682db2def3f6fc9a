"""The parallel FP on volumes past 2 and 3.5 GiB (GPU test).

The shared walk gathers by 32-bit byte offsets up to 3.5 GiB, past 2 GiB with
the top bit set; larger volumes have the walk table below 8192 wavefronts and
every lane's own walk from there on, and in a batch the latter.  Few angles and
columns keep the rays few; the volumes hold numbers to their last voxel.
Against the oracle at 1e-5 of the maximum, as the other FP forms; the batch
against the one-problem CGLS within the tolerances of the other batched tests.
"""

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from ccpi.reconstruction import projectors as J
from geometries import PB, centred, oracle_geom
from test_gpu_par_fp_forms import _geom, _waves

pytestmark = pytest.mark.gpu

GIB = 1 << 30
V1 = (1.0, 1.0, 1.0)


def _pb(nz, na, nh):
    ang = np.deg2rad(np.linspace(0, 180, na, endpoint=False) + 33.0)
    return PB((1025, 1024, nz), V1, ang, centred(nh, 3.7, 0.31), centred(nz, 1.0))


# volume bytes and wavefronts of each form
CASES = {
    "shared_past_2_gib": (_pb(520, 3, 400), (2 * GIB, 3.5 * GIB), (2400, 8192)),
    "table_past_3.5_gib": (_pb(900, 2, 380), (3.5 * GIB, 4 * GIB), (2400, 8192)),
    "lanes_past_3.5_gib": (_pb(900, 6, 380), (3.5 * GIB, 4 * GIB), (8192, 1 << 20)),
}


def _volume(g):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(5)
    return torch.rand(g.shape, generator=gen, device="cuda")


@pytest.fixture(autouse=True)
def _memory_back():
    J.plan_cache_clear()
    yield
    J.plan_cache_clear()
    torch.cuda.empty_cache()


@pytest.mark.parametrize("name", list(CASES))
def test_fp_of_large_volumes(name):
    g, size, waves = CASES[name]
    assert size[0] < 4 * np.prod(g.shape) <= size[1] and waves[0] <= _waves(g) < waves[1]
    print(f"\nparallel FP {name} {g.shape} {g.sino_shape}", flush=True)
    x = _volume(g)
    y = J.forward_project(_geom(g), x).cpu().numpy()
    # rays of some 1200 cells, 8 bytes each in a walk table; no other table of
    # these plans is near a megabyte
    cells = 8 * len(g.angles) * len(g.h_pix) * 500
    assert (J.plan_cache_bytes() > cells) == name.startswith("table")
    yo = oracle_geom(g).fp(x.cpu().numpy())
    scale = np.abs(yo).max()
    assert scale > 0 and np.abs(y - yo).max() < 1e-5 * scale


@pytest.mark.parametrize("name", ["shared_past_2_gib", "lanes_past_3.5_gib"])
def test_batched_fp_of_large_volumes(name):
    g, _, _ = CASES[name]
    print(f"\nbatched CGLS {name} {g.shape} {g.sino_shape}", flush=True)
    G = _geom(g)
    b = J.forward_project(G, _volume(g))
    x, r, n = J.cgls(G, b, 1)
    xs, rs, norms = J.cgls_batched([G], [b], 1)
    scale = float(x.abs().max())
    assert scale > 0
    assert float((xs[0] - x).abs().max()) < 1e-5 * scale
    assert float((rs[0] - r).abs().max()) < 1e-5 * float(b.abs().max())
    assert np.allclose(norms[0], n, rtol=1e-6)
