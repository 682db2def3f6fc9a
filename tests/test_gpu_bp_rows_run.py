"""FP64 accumulation at every width of the phased cone BP (GPU test).

Each case names the rows per lane and rounds that its geometry runs with and
asks the library for them, so a geometry that reaches another kernel instance
fails.  Two MLEM iterations are no further from the FP64 oracle (L2, relative)
than the float oracle is plus 1e-5, as in test_gpu_accum_fp64_paths.py; the
float instances have the same geometries in test_gpu_bp_row_widths.py.
"""

import numpy as np
import pytest

torch = pytest.importorskip("torch")

import oracle
from bp_cases import CASES
from geometries import oracle_geom
from test_bp_rows import WIDTHS, bp_rows, row_geometry
from test_gpu_bp_paths import _geom

pytestmark = pytest.mark.gpu

RUN = {f"rows{r}{'_near' if near else ''}": (row_geometry(r, near), WIDTHS[r, near])
       for r, near in [(64, False), (65, False), (192, True), (193, False), (384, False),
                       (385, False), (385, True), (513, True)]}
RUN["rows1000"] = (CASES["phased_s16_2ph"][0], (16, 2))


@pytest.mark.parametrize("name", list(RUN))
def test_mlem_fp64_at_each_width(name):
    from ccpi.reconstruction.projectors import mlem
    g, want = RUN[name]
    assert bp_rows(g) == want
    og = oracle_geom(g)
    b = np.random.default_rng(43).random(g.sino_shape).astype(np.float32) + 0.1
    print(f"\nphased BP, FP64 sums, {name}: {want[0]} rows per lane, {want[1]} rounds", flush=True)
    x64 = oracle.mlem(og, b.astype(np.float64), 2, dtype=np.float64)
    x32 = oracle.mlem(og, b, 2).astype(np.float64)
    xa = mlem(_geom(g), torch.from_numpy(b).cuda(), 2, accum_fp64=True).cpu().numpy()
    nrm = np.linalg.norm(x64)
    assert nrm > 0
    assert np.linalg.norm(xa.astype(np.float64) - x64) / nrm <= \
        np.linalg.norm(x32 - x64) / nrm + 1e-5
