"""Device memory that solver calls leave held (GPU test).

One workspace stays after any number of calls in turn, at most four after
overlapping ones, and none of more than 2 GiB.  The order in which they go and
the second try of a refused allocation are checked on the CPU
(test_host_rules.py).
"""

import threading

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from ccpi.reconstruction import projectors as J
from geometries import centred

pytestmark = pytest.mark.gpu

A = np.linspace(0, np.pi, 24, endpoint=False) + 0.02


def _geom(n, nz, na=24):
    nh = int(1.42 * n)
    return J.Geometry(A[:na], centred(nh, 1.0), centred(nz, 1.0), (-n / 2, -n / 2, -nz / 2),
                      (1, 1, 1), (n, n, nz))


def _workspace(g):
    """Bytes of a CGLS workspace: three volumes and two sinograms (nothing
    else of it comes near a volume)."""
    return 4 * (3 * int(np.prod(g.shape)) + 2 * int(np.prod(g.sino_shape)))


def _overlapping(g, bs, calls):
    start = threading.Barrier(len(bs))

    def work(b):
        with torch.cuda.stream(torch.cuda.Stream()):
            start.wait()
            for _ in range(calls):
                J.cgls(g, b, 3)

    torch.cuda.synchronize()
    ts = [threading.Thread(target=work, args=(b,)) for b in bs]
    for t in ts:
        t.start()
    for t in ts:
        t.join()


@pytest.fixture
def held():
    """Device memory taken since the start, outside torch.  What the runtime
    allocates once (code, queues, their scratch) is there before."""
    g = _geom(64, 16)
    b = torch.ones(g.sino_shape, device="cuda")
    J.cgls(g, b, 1)
    _overlapping(g, [b] * 8, 2)
    J.plan_cache_clear()
    torch.cuda.empty_cache()
    torch.cuda.synchronize()
    free0, own0 = torch.cuda.mem_get_info()[0], torch.cuda.memory_reserved()
    yield lambda: (free0 - torch.cuda.mem_get_info()[0]
                   - (torch.cuda.memory_reserved() - own0))
    J.plan_cache_clear()
    torch.cuda.empty_cache()


def test_calls_in_turn_hold_one_workspace(held):
    g = _geom(256, 64)
    b = torch.ones(g.sino_shape, device="cuda")
    w = _workspace(g)
    J.cgls(g, b, 1)
    once = held()
    for _ in range(6):
        J.cgls(g, b, 1)
    print(f"\nworkspace {w}, held {once} and {held()}", flush=True)
    assert 0.9 * w < once < 1.5 * w
    assert held() - once < w // 4
    J.plan_cache_clear()
    assert held() < w // 4


def test_overlapping_calls_leave_at_most_four(held):
    g = _geom(256, 64)
    bs = [torch.ones(g.sino_shape, device="cuda") for _ in range(8)]
    J.cgls(g, bs[0], 1)
    once = held()    # one workspace, its buffers in whole pages, and the plan
    _overlapping(g, bs, 4)
    print(f"\none workspace {once}, held {held()}", flush=True)
    assert held() <= 4 * once


def test_a_workspace_past_2_gib_goes_back(held):
    g = _geom(1024, 200, na=4)
    b = torch.ones(g.sino_shape, device="cuda")
    assert _workspace(g) > 2 << 30
    J.cgls(g, b, 1)
    print(f"\nworkspace {_workspace(g)}, held {held()}", flush=True)
    assert held() < 100 << 20
