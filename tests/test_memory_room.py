"""The Python layer's allocations give the library's kept workspaces back
before they fail (CPU test; the device and the library are stand-ins)."""

import pytest

torch = pytest.importorskip("torch")

from ccpi.reconstruction import projectors as J


class _Library:
    def __init__(self):
        self.cleared = 0

    def ccpi_workspaces_clear(self):
        self.cleared += 1

    def __getattr__(self, name):   # entry points that are never reached
        return None


@pytest.fixture
def library(monkeypatch):
    L = _Library()
    monkeypatch.setattr(J, "lib", lambda: L)
    return L


def _full(monkeypatch, name, until):
    """torch.<name> with no room until ``until()``."""
    real = getattr(torch, name)

    def alloc(*a, **k):
        if not until():
            raise torch.cuda.OutOfMemoryError("no room")
        return real(*a, **k)
    monkeypatch.setattr(torch, name, alloc)


def _geom():
    return J.Geometry([0.1, 0.2], [-0.5, 0.5], [0.5], (-1, -1, 0), (1, 1, 1), (2, 2, 1))


@pytest.mark.parametrize("call", ["forward_project", "backward_project", "cgls", "sirt", "mlem"])
def test_an_output_is_tried_again(monkeypatch, library, call):
    g = _geom()
    _full(monkeypatch, "empty" if call == "mlem" else "zeros", lambda: library.cleared > 0)
    arg = torch.ones(g.shape if call == "forward_project" else g.sino_shape)
    # past the allocation: the CPU tensor is refused as ever
    with pytest.raises(TypeError):
        getattr(J, call)(g, arg, *([2] if call in ("cgls", "sirt", "mlem") else []))
    assert library.cleared == 1


def test_no_room_at_all_is_the_error_it_was(monkeypatch, library):
    _full(monkeypatch, "zeros", lambda: False)
    with pytest.raises(torch.cuda.OutOfMemoryError):
        J.forward_project(_geom(), torch.ones(2, 2, 1))
    assert library.cleared == 1


def test_nothing_is_given_back_while_there_is_room(library):
    with pytest.raises(TypeError):
        J.forward_project(_geom(), torch.ones(2, 2, 1))
    assert library.cleared == 0
