"""The HIP runtime's last error, which all libraries of a process share and which stays until it is
read: an error that other code left behind is neither reported by the framework's launches nor
taken from its owner, and what the framework does and destroys leaves none behind."""
import ctypes as C
import gc

import numpy as np
import pytest

import parthenon_amd as pa
from parthenon_amd import gmg
from parthenon_amd.burgers import BurgersDriver, DeviceBurgersDriver, make_burgers_mesh

pytestmark = pytest.mark.gpu

BOX = [((-0.1, 0.1, -0.1, 0.1, -0.1, 0.1), 1)]


def runtime():
    pa.lib()
    with open("/proc/self/maps") as f:
        path = next(line.split()[-1] for line in f if "libamdhip64.so" in line)
    return C.CDLL(path)


def exchange(form):
    m = pa.Mesh((24, 24, 24), (8, 8, 8), 2, refine_boxes=BOX)
    m.add_field("q", 2)
    m.finalize()
    md = m.mesh_data("base")
    md.upload("q", np.ones(m.field_shape("q")))
    return m, lambda: form(md), lambda: md.download("q")


def device_run(use_graph, block, scalars, boxes=()):
    m = make_burgers_mesh((3 * block,) * 3, (block,) * 3, 4, scalars, refine_boxes=boxes)
    d = DeviceBurgersDriver(m, use_graph=use_graph)
    d.initialize("sinusoid", seed=1)
    return d, lambda: d.cycles(2), lambda: d.base.download("U")


def task_run():
    m = make_burgers_mesh((24, 24, 24), (8, 8, 8), 4, 1, refine_boxes=BOX)
    d = BurgersDriver(m)
    d.initialize("sinusoid", seed=1)
    return d, d.cycle, lambda: d.base.download("U")


def remesh():
    crit = [dict(field="U", comp=3, method="derivative_order_1", refine_tol=1e-6,
                 derefine_tol=0.0)]
    m = make_burgers_mesh((24, 24, 24), (8, 8, 8), 4, 1,
                          adaptive=dict(numlevel=2, derefine_count=10, criteria=crit))
    d = DeviceBurgersDriver(m)
    d.initialize("sinusoid", seed=1)
    return d, lambda: d.adaptive_cycles(2), lambda: d.base.download("U")


def mesh_solve(boxes, precision):
    m = pa.Mesh((16, 16, 16), (8, 8, 8), 2, periodic=(0, 0, 0), bcs=("fixed_face",) * 6,
                refine_boxes=boxes)
    m.add_field("u", 1)
    m.add_field("rhs", 1)
    m.finalize()
    md = m.mesh_data("base")
    md.upload("rhs", np.ones(m.field_shape("rhs")))
    s = gmg.MeshMGSolver(m, "u", "rhs", gmg.MeshMGParams(max_iters=6, precision=precision))

    def run():
        gmg.set_to_zero(md, "u")
        s.setup(md)
        s.solve(md)
    return s, run, lambda: md.download("u")


def array_solve(precision):
    s = gmg.MGSolver(32, precision)

    def run():
        s.set_rhs_blobs(3)
        s.reset()
        s.solve()
    return s, run, s.solution


def served():
    s = gmg.Server("mixed", keep_solutions=True)
    r = s.submit(32, 5)
    return s, lambda: s.run(realtime=False), lambda: s.solution(r)


CASES = {
    "exchange-fused": lambda: exchange(pa.exchange_fused),
    "exchange-tasks": lambda: exchange(pa.exchange),
    "run-eager": lambda: device_run(False, 16, 4),
    "run-graph": lambda: device_run(True, 8, 2),
    "run-graph-other-shape": lambda: device_run(True, 12, 2),
    "run-graph-tiles": lambda: device_run(True, 32, 1),
    "run-refined": lambda: device_run(True, 16, 4, BOX),
    "tasks-refined": task_run,
    "remesh": remesh,
    "mesh-solve-uniform": lambda: mesh_solve((), "mixed"),
    "mesh-solve-refined": lambda: mesh_solve(BOX, "fp64"),
    "array-solve-mixed": lambda: array_solve("mixed"),
    "array-solve-fp64": lambda: array_solve("fp64"),
    "served": served,
}


@pytest.mark.parametrize("name", list(CASES))
def test_errors_of_others_stay_theirs(name):
    print(f"case error state {name}", flush=True)
    hip = runtime()
    assert hip.hipGetLastError() == 0
    keep, run, result = CASES[name]()
    assert hip.hipPeekAtLastError() == 0
    assert hip.hipSetDevice(99) == 101  # hipErrorInvalidDevice, refused by the host
    for _ in range(2):
        run()
    assert hip.hipGetLastError() == 101  # still there for the code that it belongs to
    assert np.isfinite(result()).all()
    del keep, run, result
    gc.collect()
    assert hip.hipPeekAtLastError() == 0
