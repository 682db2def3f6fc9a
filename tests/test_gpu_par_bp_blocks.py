"""The tiled parallel-beam backprojector's staging at its edges (GPU test).

The tiled BP stages blocks of up to four angles in two LDS buffers, finds
the tiles' detector spans 256 angles at a time and, where a wavefront's
footprints are at most two columns, weighs them without a loop.  The cases
reach: more than 256 angles in one group and in several, with a last block
that is not full; pixels so fine that a block is one angle and every
footprint long; pixels wider than the voxels; a detector narrower than the
volume's shadow (empty spans); axis-aligned lines; one slice; more rows than
slices and more slices than rows; a sinogram whose memory is not 16-byte
aligned.  Against the oracle's b2D at 1e-5 of the maximum, the
summation-order tolerance of the other BP tests, into zeros and into a
non-zero volume; and in one batched call together, whose first gradient
norm is that of the oracle's BP.
"""

import numpy as np
import pytest

torch = pytest.importorskip("torch")

import oracle
from geometries import PB, centred

pytestmark = pytest.mark.gpu


def _turn(n, start=0.0):
    return np.deg2rad(np.linspace(0, 180, n, endpoint=False) + start)


V1 = (1.0, 1.0, 1.0)
CASES = {
    "angles_613": PB((33, 17, 16), V1, _turn(613), centred(51, 1.0, 0.3), centred(16, 1.0)),
    "angles_257_groups": PB((16, 16, 3), V1, _turn(2057, 0.01), centred(23, 1.0), centred(3, 1.0)),
    "fine_pixels": PB((19, 18, 9), V1, _turn(31), centred(420, 0.0666, 0.1), centred(9, 1.0)),
    "wide_pixels": PB((47, 48, 16), V1, _turn(30, 0.5), centred(32, 2.3, 0.4), centred(16, 1.0)),
    "narrow_detector": PB((64, 64, 8), V1, _turn(45), centred(12, 1.0, 0.2), centred(8, 1.0)),
    "axes": PB((34, 20, 12), V1, np.deg2rad(np.r_[0.0, 90.0, 180.0, 270.0, 45.0, 135.0, 225.0]),
               centred(50, 1.0, 0.25), centred(12, 1.0)),
    "one_slice": PB((40, 40, 1), V1, _turn(60), centred(57, 1.0, 0.31), centred(1, 1.0)),
    "more_rows": PB((18, 30, 6), V1, _turn(50, 1.0), centred(36, 1.0), centred(20, 1.0)),
    "more_slices": PB((18, 30, 21), V1, _turn(50, 1.0), centred(36, 1.0), centred(10, 1.0)),
}


def _geoms(g):
    from ccpi.reconstruction.projectors import Geometry
    return (Geometry(g.angles, g.h_pix, g.v_pix, g.origin, g.vsize, g.shape),
            oracle.Geometry(g.angles, g.h_pix, g.v_pix, g.origin, g.vsize, g.shape))


def _rel(a, b):
    return float(np.abs(a - b).max() / max(np.abs(b).max(), 1e-30))


@pytest.mark.parametrize("name", list(CASES))
def test_tiled_bp_blocks(name):
    from ccpi.reconstruction.projectors import backward_project
    g = CASES[name]
    G, og = _geoms(g)
    rng = np.random.default_rng(29)
    s = rng.random(g.sino_shape).astype(np.float32)
    x0 = rng.random(g.shape).astype(np.float32)
    print(f"\ntiled parallel BP blocks {name} {g.shape}", flush=True)
    # one float into its allocation: 4-byte aligned rows
    buf = torch.zeros(s.size + 1, device="cuda")
    off = buf[1:].view(g.sino_shape)
    off.copy_(torch.from_numpy(s))
    want = og.bp(s)
    b = backward_project(G, torch.from_numpy(s).cuda())
    assert _rel(b.cpu().numpy(), want) < 1e-5
    assert torch.equal(backward_project(G, off), b)
    b2 = backward_project(G, torch.from_numpy(s).cuda(), torch.from_numpy(x0).cuda())
    assert _rel(b2.cpu().numpy(), og.bp(s, x0.copy())) < 1e-5


def test_batched_items_share_lds():
    from ccpi.reconstruction.projectors import cgls, cgls_batched
    rng = np.random.default_rng(31)
    names = [n for n in CASES if n != "angles_257_groups"]
    geoms = [_geoms(CASES[n])[0] for n in names]
    bs = [torch.from_numpy(rng.random(CASES[n].sino_shape).astype(np.float32)).cuda()
          for n in names]
    print("\nbatched tiled BP items", flush=True)
    xs, _, norms = cgls_batched(geoms, bs, 2)
    for n, G, b, x, nb in zip(names, geoms, bs, xs, norms):
        x1, _, n1 = cgls(G, b.clone(), 2)
        # the sums of the projectors are the one-problem path's; the norms'
        # orders differ
        assert _rel(x.cpu().numpy(), x1.cpu().numpy()) < 1e-5, n
        assert np.allclose(nb, n1, rtol=1e-5), n
