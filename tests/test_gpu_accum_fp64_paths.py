"""FP64 accumulation on the cone BP's paths (GPU test).

The FP64-accumulation BP folds each row's set into LDS addresses of 8-byte
cells where every row is in one set, for 1 to 4 rows per lane, with blocks
under, across and above the source row, padded rows and edge rows; columns
whose sets overlap take the general path, and the phased form its own.  Two
MLEM iterations of each are no further from the FP64 oracle (L2, relative)
than the float oracle is plus 1e-5, the bound of the full-size cases.
"""

import numpy as np
import pytest

torch = pytest.importorskip("torch")

import oracle
from bp_cases import CASES
from geometries import oracle_geom
from test_gpu_bp_paths import _geom

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", ["s1", "s2_blocks", "s3", "s4", "phased_s8_main",
                                  "phased_s8_offz", "phased_s8_2ph"])
def test_mlem_fp64_paths(name):
    from ccpi.reconstruction.projectors import mlem
    g, _ = CASES[name]
    og = oracle_geom(g)
    b = np.random.default_rng(19).random(g.sino_shape).astype(np.float32) + 0.1
    print(f"\nFP64 accumulation {name}", flush=True)
    x64 = oracle.mlem(og, b.astype(np.float64), 2, dtype=np.float64)
    x32 = oracle.mlem(og, b, 2).astype(np.float64)
    xa = mlem(_geom(g), torch.from_numpy(b).cuda(), 2, accum_fp64=True).cpu().numpy()
    nrm = np.linalg.norm(x64)
    assert np.linalg.norm(xa.astype(np.float64) - x64) / nrm <= \
        np.linalg.norm(x32 - x64) / nrm + 1e-5
