"""The refined-mesh multigrid's stages that read neighbour blocks in place: every smoother with
odd and even stage counts (the iterate ends in either of a level's two arrays), two levels of
refinement, and graph replay against eager launches. The residual is recomputed with the oracle's
leaf operator, the solution compared with the oracle's."""
import numpy as np
import pytest

from parthenon_amd.gmg import MeshMGParams, MeshMGSolver
from test_gpu_mg_tree import centres, from_bricks, make_meshes, rms, to_bricks

pytestmark = pytest.mark.gpu

MESHES = {
    "2d": ((32, 32, 1), (8, 8, 1), [((-0.4, -0.3, -0.4, -0.3, 0.0, 1.0), 2)]),
    "3d": ((16, 16, 16), (8, 8, 8), [((-0.4, -0.3, -0.4, -0.3, -0.4, -0.3), 1)]),
}


@pytest.mark.parametrize("smoother,pre,post", [("jacobi", 1, 2), ("jacobi", 3, 3),
                                               ("jacobi", 2, 1), ("SRJ2", 2, 2), ("SRJ3", 2, 2)])
@pytest.mark.parametrize("case", ["2d", "3d"])
def test_stage_counts(case, smoother, pre, post):
    print(f"case in place {case} {smoother} {pre} {post}", flush=True)
    nx, block, boxes = MESHES[case]
    m, om = make_meshes(nx, block, (-0.5,) * 3, (0.5,) * 3, boxes=boxes)
    md = m.mesh_data("base")
    c = centres(m)
    nd = 3 if case == "3d" else 2
    b = np.exp(-np.sum((c[:, :nd] - 0.1) ** 2, axis=1) / 0.02)
    md.upload("rhs", to_bricks(m, b, name="rhs"))
    runs = []
    for graph in (True, False):
        md.upload("u", np.zeros(m.field_shape("u")))
        s = MeshMGSolver(m, "u", "rhs", MeshMGParams(
            max_iters=200, residual_tolerance=1e-9, precision="fp64", smoother=smoother,
            pre_sweeps=pre, post_sweeps=post))
        s.set_graph(graph)
        s.setup(md)
        it, res = s.solve(md)
        runs.append((it, res, from_bricks(m, md.download("u"))))
    (it, res, u), (it2, res2, u2) = runs
    assert it == it2 and res == res2 and np.array_equal(u, u2)
    assert res <= 1e-9
    # the same residual in another order of summation
    assert rms(b - om.poisson_apply(u)) <= 1.01e-9
    # ||u - x|| <= ||A^-1|| ||r||, and the smallest eigenvalue of -A is about nd pi^2
    xo, _, _ = om.poisson_solve(b, tol=1e-13)
    assert rms(u - xo) <= 2 * 1e-9 / (nd * np.pi ** 2) * 4
