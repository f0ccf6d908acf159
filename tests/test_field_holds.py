"""Views over MeshData.pointers. The addresses keep no mesh alive (torch never drops the tuple that
it reads them from, so nothing that they kept would be freed); the memory that they name stays
readable past the end of the mesh, or a remesh, until the next mesh is finalized or changes."""
import ctypes as C
import gc
import weakref

import numpy as np
import pytest

import parthenon_amd as pa
from parthenon_amd.burgers import DeviceBurgersDriver, make_burgers_mesh


class Library:
    """Stands for the library: a field's data, its holds and a remesh, in the order of the calls."""

    memory = C.c_double(0.0)

    def __init__(self):
        self.calls, self.modified = [], 0

    def pth_field_pointers(self, handle, field, data, coarse, flux):
        data._obj.contents = self.memory
        return 0

    def pth_field_hold(self, handle, field):
        self.calls.append("hold " + field.decode())
        return 1

    def pth_field_release(self, hold):
        self.calls.append("release")

    def pth_mesh_adapt(self, handle, modified):
        self.calls.append("adapt")
        modified._obj.value = self.modified
        return 0

    def pth_mesh_finalize(self, handle):
        self.calls.append("finalize")
        return 0

    def pth_mesh_destroy(self, handle):
        self.calls.append("destroy")


@pytest.fixture
def library(monkeypatch):
    library = Library()
    monkeypatch.setattr(pa, "lib", lambda: library)
    monkeypatch.setattr(pa, "_LIB", library)
    monkeypatch.setattr(pa.Mesh, "_shapes", lambda self: None)
    yield library
    pa._Kept.replace(())


def mesh_of(library, cells=4):
    m = object.__new__(pa.Mesh)
    m._h, m.fields, m.multilevel = 1, {"u": (1, 0), "v": (1, 0)}, False
    m.nblocks, m.ent = 1, (cells, cells, cells)
    m._data = {"base": pa.MeshData(m, "base", None)}
    return m


def test_addresses_keep_no_mesh_but_its_memory(library):
    m = mesh_of(library)
    gone = weakref.ref(m)
    data, coarse, flux = m._data["base"].pointers("u")
    assert data == C.addressof(Library.memory) and coarse is None and flux is None
    view = {"data": (data, False)}
    del m, data
    gc.collect()
    # the mesh is destroyed, the memory that was given out (not the other field's) is held
    assert gone() is None and library.calls == ["hold u", "destroy"]
    pa.Mesh.finalize(mesh_of(library))
    assert library.calls[2:4] == ["release", "finalize"]  # before the new mesh takes memory
    assert view


def test_a_remesh_holds_the_old_memory_until_the_next(library):
    m = mesh_of(library)
    m._data["base"].pointers("u")
    m.adapt()
    assert library.calls == ["hold u", "adapt", "release"]  # the mesh is as it was
    library.modified = 1
    m.adapt()
    assert library.calls[3:] == ["hold u", "adapt"]
    m.adapt()
    assert library.calls[5:] == ["hold u", "adapt", "release"]
    m._data.clear()


def test_held_memory_is_bounded(library, monkeypatch):
    monkeypatch.setattr(pa._Kept, "LIMIT", 8 * 4 ** 3 * 2)
    for n in range(4):
        m = mesh_of(library, 4)
        m._data["base"].pointers("u")
        del m
        gc.collect()
        assert len(pa._Kept.holds) == min(n + 1, 2)
    m = mesh_of(library, 6)  # larger than the limit by itself
    m._data["base"].pointers("u")
    del m
    gc.collect()
    assert not pa._Kept.holds and library.calls.count("release") == 5


class View:
    """A field's memory for torch."""

    def __init__(self, md, field):
        self.__cuda_array_interface__ = dict(data=(md.pointers(field)[0], False),
                                             shape=md.mesh.field_shape(field), typestr="<f8",
                                             version=3)


@pytest.mark.gpu
def test_meshes_that_torch_looked_at_are_freed():
    # 96 MB a mesh: every mesh's memory but the last one's views is back before the next
    print("case views are freed", flush=True)
    import torch
    used = []
    for _ in range(4):
        m = pa.Mesh((64,) * 3, (16,) * 3, 4)
        m.add_field("q", 8)
        m.finalize()
        t = torch.as_tensor(View(m.mesh_data("base"), "q"), device="cuda")
        t.fill_(1.0)
        del m, t
        gc.collect()
        torch.cuda.synchronize()
        free, total = pa.device_memory()
        used.append(total - free)
    assert used[3] - used[1] < 8 << 20, used


@pytest.mark.gpu
def test_view_of_a_mesh_that_is_gone():
    print("case view after the mesh", flush=True)
    import torch
    m = pa.Mesh((32,) * 3, (16,) * 3, 4)
    m.add_field("q", 2)
    m.finalize()
    md = m.mesh_data("base")
    values = np.random.default_rng(1).random(m.field_shape("q"))
    md.upload("q", values)
    view = torch.as_tensor(View(md, "q"), device="cuda")
    gone = weakref.ref(m)
    del m, md
    gc.collect()
    assert gone() is None
    other = torch.full((view.numel(),), 7.0, dtype=torch.float64, device="cuda")
    assert other.data_ptr() != view.data_ptr() and np.array_equal(view.cpu().numpy(), values)


@pytest.mark.gpu
def test_view_from_before_a_remesh():
    print("case view over a remesh", flush=True)
    import torch
    crit = [dict(field="U", comp=3, method="derivative_order_1", refine_tol=1e-6,
                 derefine_tol=0.0)]
    m = make_burgers_mesh((16, 16, 16), (8, 8, 8), 4, 1,
                          adaptive=dict(numlevel=2, derefine_count=10, criteria=crit))
    d = DeviceBurgersDriver(m)
    d.initialize("sinusoid", seed=2)
    before = torch.as_tensor(View(d.base, "U"), device="cuda")
    where = before.data_ptr()
    d.cycles(1)
    values = d.base.download("U")
    pa.Refinement.Tag(d.base)
    assert m.nblocks == 8 and m.adapt() and m.nblocks == 64
    after = torch.as_tensor(View(d.base, "U"), device="cuda")
    # new memory for the field; the old one, which new tensors do not get, is as it was
    assert after.data_ptr() != where and np.array_equal(after.cpu().numpy(), d.base.download("U"))
    other = torch.full((before.numel(),), 7.0, dtype=torch.float64, device="cuda")
    assert other.data_ptr() != where and np.array_equal(before.cpu().numpy(), values)
