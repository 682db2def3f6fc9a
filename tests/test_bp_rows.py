"""Rows per lane and rounds that the cone BP runs with (CPU test:
ccpi_cone_bp_rows is a host computation and touches no device).

The layout of test_bp_layout.py is the most rows that a lane takes; the phased
form takes fewer, in more rounds, where 64 lanes of fewer rows cover the
detector.  The pair that runs has to keep the lanes of a round on distinct
slices as the layout's does, and the kernel instance that a geometry reaches
follows from it.
"""

import ctypes as C

import numpy as np
import pytest

from bp_cases import CASES, bp_path
from ccpi.reconstruction import _lib
from geometries import CB, centred
from test_bp_layout import _geom, _layout, _max_rows_per_slice

A10 = np.linspace(0, 2 * np.pi, 10, endpoint=False) + 0.05


def row_geometry(rows, near):
    """The scans of test_gpu_bp_row_widths.py."""
    pitch = 0.25 if near else 0.4
    sod = 24.0 if near else 40.0
    nz = max(4, int(rows * pitch * 0.45))
    return CB((12, 10, nz), (1, 1, 1), A10, centred(18, 1.6), centred(rows, pitch, 0.1 * pitch),
              sod, 2 * sod, source_z=0.013 - 0.2 * nz if near else 0.03)


# (rows, near source) -> rows per lane, rounds: the last row count of each
# width and the first of the next
WIDTHS = {
    (63, False): (1, 7), (64, False): (1, 7), (65, False): (2, 4), (128, False): (2, 4),
    (129, False): (3, 3), (192, False): (3, 3), (193, False): (4, 2), (256, False): (4, 2),
    (257, False): (6, 2), (384, False): (6, 2), (385, False): (8, 1), (512, False): (8, 1),
    (513, False): (12, 1), (64, True): (1, 13), (128, True): (2, 7), (192, True): (3, 5),
    (256, True): (4, 4), (384, True): (6, 3), (385, True): (8, 2), (513, True): (12, 2),
    (769, True): (16, 1),
}
# the ones that run with other rows than their layout's
NARROWED = {"phased_s8_small": (1, 7), "phased_s8_offz": (1, 7), "phased_s8_2ph": (6, 3)}


def bp_rows(g):
    out = [C.c_int(), C.c_int()]
    _lib.check(_lib.lib().ccpi_cone_bp_rows(C.byref(_geom(g).c_struct()),
                                            *[C.byref(q) for q in out]))
    return tuple(q.value for q in out)


def _distinct(g, rows, rounds, phased):
    dense = np.linspace(0, 2 * np.pi, 3600, endpoint=False)
    worst = max(_max_rows_per_slice(g, g.angles), _max_rows_per_slice(g, dense))
    return rounds * rows >= worst or (phased and rounds == 64)


@pytest.mark.parametrize("name", list(CASES))
def test_rows_of_the_path_cases(name):
    g, path = CASES[name]
    stride, phased, phases = bp_path(g)
    rows, rounds = bp_rows(g)
    assert (rows, rounds) == NARROWED.get(name, (path[0], path[2]))
    assert rows <= stride and rounds >= phases
    assert _distinct(g, rows, rounds, phased)


@pytest.mark.parametrize("rows,near", list(WIDTHS))
def test_rows_follow_the_detector(rows, near):
    g = row_geometry(rows, near)
    stride, phased, _, bound = _layout(g)
    lane, rounds = bp_rows(g)
    assert phased == 1 and (lane, rounds) == WIDTHS[rows, near]
    # the least width that covers the detector in one block, or the layout's
    assert lane == min([stride] + [s for s in (1, 2, 3, 4, 6, 8, 12) if 64 * s >= rows])
    assert rounds == min(64, -(-bound // lane))
    assert _distinct(g, lane, rounds, True)


def test_rows_query_rejects():
    from ccpi.reconstruction.projectors import Geometry
    from geometries import pb_small
    g = pb_small()
    G = Geometry(g.angles, g.h_pix, g.v_pix, g.origin, g.vsize, g.shape)
    out = [C.c_int(), C.c_int()]
    L = _lib.lib()
    assert L.ccpi_cone_bp_rows(C.byref(G.c_struct()), *[C.byref(q) for q in out]) == -1
    cone = _geom(CASES["s1"][0]).c_struct()
    assert L.ccpi_cone_bp_rows(C.byref(cone), None, C.byref(out[1])) == -1
