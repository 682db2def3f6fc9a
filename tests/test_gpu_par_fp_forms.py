"""Every form of the parallel forward projector against the oracle (GPU test).

One row per slice: launches of few wavefronts read the plan's walk table,
with 1 to 8 lanes per ray's cells; the others share one wavefront's
walk of 64 rays, with 1 or 2 rays per lane and, below 4 slices, single
reads.  Other row maps walk in every lane.  The sizes meet the edges: rays
of fewer than 8 cells, ray counts off 64 and the angle tile (32), axis-
parallel and diagonal lines, 1 to 5 slices, a last lane of fewer than 4
rows, rows past the volume, several row blocks, fewer rows than slices.

Tolerance 1e-5 of the maximum, as in test_gpu_parity (summation order).  A
cell's value is only ever added where its ray crosses it: a volume with one
infinite voxel gives infinite sums on exactly the oracle's rays.  All forms
add in the walk's order: ccpi_pb_f2D_noalloc, which has no
table, equals ccpi_pb_f2D bit for bit (test_zz_no_alloc).
"""

import numpy as np
import pytest

torch = pytest.importorskip("torch")

import oracle
from geometries import PB, centred

pytestmark = pytest.mark.gpu


def _pb(shape, na, nh, nv, shift=0.31, pitch=1.0, vsize=(1.0, 1.0, 1.0), start=0.0):
    ang = np.deg2rad(np.r_[0.0, 45.0, 90.0, 135.0, np.linspace(start, 180 + start, na,
                                                              endpoint=False)])
    return PB(shape, vsize, ang, centred(nh, pitch, shift), centred(nv, 1.0))


TABLE = {
    "t_one_slice": _pb((64, 64, 1), 30, 91, 1),
    "t_short_rays": _pb((3, 2, 6), 5, 7, 6),
    "t_three_slices": _pb((20, 33, 3), 9, 41, 3),
    "t_ragged_rows": _pb((37, 21, 22), 20, 56, 22),
    "t_many_lanes": _pb((24, 24, 70), 16, 40, 70),
    "t_half_pixels": _pb((40, 40, 9), 60, 120, 9, pitch=0.5),
}
SHARED = {
    "s_one_slice": _pb((300, 300, 1), 400, 425, 1),
    "s_two_slices": _pb((200, 180, 2), 620, 283, 2),
    "s_three_slices_lr1": _pb((128, 128, 3), 900, 190, 3),
    "s_five_slices": _pb((150, 130, 5), 350, 233, 5),
    "s_sixteen": _pb((128, 128, 16), 221, 182, 16),
    "s_odd_29": _pb((100, 127, 29), 130, 190, 29),
    "s_row_blocks_70": _pb((64, 64, 70), 67, 91, 70),
    "s_thin": _pb((600, 4, 12), 90, 640, 12),
}
OTHER = {
    "rows_past_volume": PB((90, 90, 6), (1, 1, 1), np.deg2rad(np.linspace(0, 180, 700)),
                           centred(130, 1.0, 0.3), np.arange(8) - 2.5),
    "fewer_rows": PB((90, 90, 9), (1, 1, 1), np.deg2rad(np.linspace(0, 180, 900)),
                     centred(130, 1.0, 0.3), np.arange(5) - 4.0),
    "two_rows_per_slice": PB((60, 60, 5), (1, 1, 2), np.deg2rad(np.linspace(0, 180, 300)),
                             centred(90, 1.0, 0.3), centred(10, 1.0)),
}
CASES = TABLE | SHARED | OTHER


def _geom(g):
    from ccpi.reconstruction.projectors import Geometry
    return Geometry(g.angles, g.h_pix, g.v_pix, g.origin, g.vsize, g.shape)


def _waves(g):
    nv = len(g.v_pix)
    lr = 1
    while lr < 16 and 4 * lr < nv:
        lr *= 2
    return len(g.angles) * len(g.h_pix) * -(-nv // (4 * lr)) * lr // 64


def test_cases_reach_both_forms():
    assert all(_waves(g) < 2400 for g in TABLE.values())
    assert all(_waves(g) >= 2400 for g in SHARED.values())


@pytest.mark.parametrize("name", list(CASES))
def test_fp_forms_parity_and_accumulation(name):
    from ccpi.reconstruction.projectors import forward_project
    g = CASES[name]
    print(f"\nparallel FP {name} {g.shape} {g.sino_shape} {_waves(g)} waves", flush=True)
    og = oracle.Geometry(g.angles, g.h_pix, g.v_pix, g.origin, g.vsize, g.shape)
    rng = np.random.default_rng(41)
    x = rng.random(g.shape).astype(np.float32)
    y0 = rng.random(g.sino_shape).astype(np.float32)
    yo = og.fp(x)
    scale = np.abs(yo).max()
    y = forward_project(_geom(g), torch.from_numpy(x).cuda()).cpu().numpy()
    assert np.abs(y - yo).max() < 1e-5 * scale
    ya = forward_project(_geom(g), torch.from_numpy(x).cuda(), torch.from_numpy(y0).cuda())
    assert np.abs(ya.cpu().numpy() - og.fp(x, y0.copy())).max() < 1e-5 * scale
    xi = x.copy()
    xi[tuple(q // 2 for q in g.shape)] = np.inf
    yi = forward_project(_geom(g), torch.from_numpy(xi).cuda()).cpu().numpy()
    assert np.array_equal(np.isposinf(yi), np.isposinf(og.fp(xi)))
    assert not np.isnan(yi[~np.isnan(og.fp(xi))]).any()
