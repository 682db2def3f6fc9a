"""Solver workspaces kept between calls (GPU test).

A solver call leaves its workspace for the next call of the device.  Calls
of different geometries, solvers and sizes in turn (buffers larger than
needed, dirty, or missing parts) give bit for bit what each gives first
after plan_cache_clear, which frees plans and workspaces; so do host threads
with streams of their own; and the memory that stays is bounded and comes
back.
"""

import threading

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from geometries import CB, PB, centred

pytestmark = pytest.mark.gpu

V1 = (1.0, 1.0, 1.0)
A = np.linspace(0, np.pi, 24, endpoint=False) + 0.02
CASES = [
    PB((40, 40, 16), V1, A, centred(57, 1.0, 0.3), centred(16, 1.0)),
    CB((20, 22, 12), V1, 2 * A, centred(40, 1.4), centred(30, 1.4), 60.0, 120.0),
    PB((18, 20, 3), V1, A, centred(29, 1.0), centred(6, 0.5)),
    CB((12, 10, 30), V1, 2 * A, centred(18, 1.6), centred(128, 0.4, 0.04), 40.0, 80.0),
    PB((64, 48, 7), V1, A, centred(81, 1.0), centred(7, 1.0)),
]


def _geom(g):
    from ccpi.reconstruction.projectors import Geometry
    if not g.cone:
        return Geometry(g.angles, g.h_pix, g.v_pix, g.origin, g.vsize, g.shape)
    return Geometry(g.angles, g.h_pix, g.v_pix, g.origin, g.vsize, g.shape, cone=True,
                    source=g.source, detector_x=g.det_x)


def _calls():
    from ccpi.reconstruction import projectors as J
    geoms = [_geom(c) for c in CASES]
    rng = np.random.default_rng(41)
    bs = [torch.from_numpy(rng.random(c.sino_shape).astype(np.float32)).cuda() for c in CASES]
    calls = []
    for G, b in zip(geoms, bs):
        calls.append(lambda G=G, b=b: J.cgls(G, b, 3))
        calls.append(lambda G=G, b=b: J.mlem(G, b, 2))
        calls.append(lambda G=G, b=b: J.cgls_reg(G, b, 2, J.TV, 1e-3))
        calls.append(lambda G=G, b=b: J.sirt(G, b, 2))
    pick = [0, 2, 4]
    calls.append(lambda: J.cgls_batched([geoms[i] for i in pick], [bs[i] for i in pick], 2))
    return calls


def _flat(r):
    out = []
    for v in (r if isinstance(r, (tuple, list)) else [r]):
        if isinstance(v, (tuple, list)):
            out += _flat(v)
        else:
            out.append(v.cpu().numpy() if torch.is_tensor(v) else np.asarray(v))
    return out


def _same(a, b):
    return len(a) == len(b) and all(np.array_equal(p, q) for p, q in zip(a, b))


def test_calls_in_turn_and_threads():
    from ccpi.reconstruction import projectors as J
    calls = _calls()
    print("\nworkspaces", flush=True)
    want = []
    for f in calls:
        J.plan_cache_clear()
        want.append(_flat(f()))
    order = list(range(len(calls)))
    for seq in (order, order[::-1], order[::3] + order[1::3] + order[2::3]):
        for i in seq:
            assert _same(_flat(calls[i]()), want[i]), i
    bad = []

    def work(seq):
        with torch.cuda.stream(torch.cuda.Stream()):
            for i in seq:
                r = calls[i]()
                torch.cuda.current_stream().synchronize()
                if not _same(_flat(r), want[i]):
                    bad.append(i)

    torch.cuda.synchronize()
    ts = [threading.Thread(target=work, args=(order[k::4] + order[(k + 1) % 4::4],))
          for k in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad


def test_kept_memory_comes_back():
    from ccpi.reconstruction import projectors as J
    g = PB((256, 256, 64), V1, A, centred(364, 1.0), centred(64, 1.0))
    G = _geom(g)
    b = torch.ones(g.sino_shape, device="cuda")
    J.cgls(G, b, 1)
    J.plan_cache_clear()
    torch.cuda.synchronize()
    free0 = torch.cuda.mem_get_info()[0]
    need = 3 * 4 * 256 * 256 * 64
    for _ in range(6):
        J.cgls(G, b, 1)
    held = free0 - torch.cuda.mem_get_info()[0]
    assert held < 8 * need      # one workspace and a plan, not six
    J.plan_cache_clear()
    assert free0 - torch.cuda.mem_get_info()[0] < need // 4
