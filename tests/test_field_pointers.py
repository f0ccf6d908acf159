"""MeshData.pointers: an address keeps its container alive. A mesh and its containers refer to
each other, so the collector frees them at a time of its own; a view made from a bare address
would then read freed device memory."""
import ctypes as C
import gc
import weakref

import parthenon_amd as pa


class Library:
    """Stands for the library: a field's data at one address, no coarse buffer, no fluxes."""

    memory = C.c_double(0.0)

    def pth_field_pointers(self, handle, field, data, coarse, flux):
        data._obj.contents = self.memory
        return 0


class Mesh:
    def __init__(self):
        self.data = {"base": pa.MeshData(self, "base", None)}


def test_address_keeps_the_mesh(monkeypatch):
    monkeypatch.setattr(pa, "lib", lambda: Library())
    mesh = Mesh()
    gone = weakref.ref(mesh)
    data, coarse, flux = mesh.data["base"].pointers("u")
    assert data == C.addressof(Library.memory) and coarse is None and flux is None
    view = {"data": (data, False)}
    del mesh, data
    gc.collect()
    assert gone() is not None  # the view still names its memory
    view.clear()
    gc.collect()
    assert gone() is None
