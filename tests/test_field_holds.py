"""MeshData.pointers across a remesh: the memory that somebody's address names is held before the
mesh changes and released with the last address; nothing is held where nobody has one."""
import ctypes as C
import gc

import numpy as np
import pytest

import parthenon_amd as pa
from parthenon_amd.burgers import DeviceBurgersDriver, make_burgers_mesh


class Library:
    """Stands for the library: a field's data, its holds and a remesh, in the order of the calls."""

    memory = C.c_double(0.0)

    def __init__(self):
        self.calls = []

    def pth_field_pointers(self, handle, field, data, coarse, flux):
        data._obj.contents = flux._obj.contents = self.memory
        return 0

    def pth_field_hold(self, handle, field):
        self.calls.append("hold " + field.decode())
        return 1

    def pth_field_release(self, hold):
        self.calls.append("release")

    def pth_mesh_adapt(self, handle, modified):
        self.calls.append("adapt")
        return 0


def test_addresses_hold_their_memory_over_a_remesh(monkeypatch):
    library = Library()
    monkeypatch.setattr(pa, "lib", lambda: library)
    monkeypatch.setattr(pa, "_LIB", library)
    mesh = object.__new__(pa.Mesh)
    mesh._h = None
    md = pa.MeshData(mesh, "base", None)
    mesh._data = {"base": md}
    md.pointers("u")
    mesh.adapt()
    assert library.calls == ["adapt"]  # the addresses are gone: nothing to hold
    data, coarse, flux = md.pointers("u")
    mesh.adapt()
    mesh.adapt()
    assert library.calls[1:] == ["hold u", "adapt", "adapt"]
    del data
    gc.collect()
    assert library.calls[-1] == "adapt"  # the flux address names the same memory
    del flux
    gc.collect()
    assert library.calls[-1] == "release"


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

    class View:
        def __init__(self):
            self.__cuda_array_interface__ = dict(
                data=(d.base.pointers("U")[0], False), shape=m.field_shape("U"), typestr="<f8",
                version=3)

    before = torch.as_tensor(View(), device="cuda")
    where = before.data_ptr()
    d.cycles(1)
    values = d.base.download("U")
    pa.Refinement.Tag(d.base)
    assert m.nblocks == 8 and m.adapt() and m.nblocks == 64
    after = torch.as_tensor(View(), device="cuda")
    # new memory for the field; the old one, which new tensors do not get, is as it was
    assert after.data_ptr() != where and np.array_equal(after.cpu().numpy(), d.base.download("U"))
    other = torch.full((before.numel(),), 7.0, dtype=torch.float64, device="cuda")
    assert np.array_equal(before.cpu().numpy(), values)
    assert other.data_ptr() != where
    del before, after, other
    gc.collect()
