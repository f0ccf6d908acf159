"""A level's stages in one pass each way (column_sweeps=True) against a launch per stage
(column_sweeps=False): the two evaluate every cell by the same operations in the same order, so
the solutions agree bit for bit. Sizes around the tiles of the passes (32 x 8 and 64 x 16 cells,
2 planes at least), remainders in each direction, levels that are and are not powers of two
(FP64 divides there), every split of the sweeps into passes, and a second inner cycle (the
passes that start from the level's x)."""
import numpy as np
import pytest

from parthenon_amd.gmg import MGParams, MGSolver

pytestmark = pytest.mark.gpu


def solve(n, precision, columns, **params):
    print(f"case gmg passes n={n} {precision} columns={columns} {params}", flush=True)
    s = MGSolver(n, precision, MGParams(column_sweeps=columns, max_iters=3, **params))
    s.set_rhs(np.random.default_rng(n).standard_normal((n, n, n)))
    s.solve()
    return s.solution()


@pytest.mark.parametrize("precision", ["mixed", "fp64"])
@pytest.mark.parametrize("n", [18, 20, 40, 56, 64, 72, 192, 208])
def test_pass_matches_stages(n, precision):
    if precision == "fp64" and n in (18, 72, 208):  # coarsest level of 9 or 13 cells: refused
        with pytest.raises(RuntimeError, match="coarsest level"):
            MGSolver(n, precision)
        return
    a = solve(n, precision, True, inner_cycles=2)
    assert np.isfinite(a).all() and np.any(a)
    assert np.array_equal(a, solve(n, precision, False, inner_cycles=2))


@pytest.mark.parametrize("precision", ["mixed", "fp64"])
@pytest.mark.parametrize("pre,post", [(0, 1), (1, 0), (1, 1), (3, 2), (4, 3), (5, 5)])
def test_sweep_counts(pre, post, precision):
    p = dict(inner_cycles=2, pre_sweeps=pre, post_sweeps=post)
    assert np.array_equal(solve(40, precision, True, **p), solve(40, precision, False, **p))
