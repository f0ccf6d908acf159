"""Kept solutions of the server: copied out by one thread or several (from 2^18 values a thread),
of sizes about that line, and of a request that is solved again."""
import numpy as np
import pytest

from parthenon_amd.gmg import MGParams, MGSolver, Server

pytestmark = pytest.mark.gpu


def test_kept_solutions_match_single_solves():
    sizes = [16, 64, 80, 128, 24]  # 4096, 2^18, just under two parts, 8 parts, 13824 values
    p = MGParams(residual_tolerance=1e-6)
    s = Server("mixed", p, keep_solutions=True)
    ids = [s.submit(n, 7 + q) for q, n in enumerate(sizes)]
    with pytest.raises(RuntimeError, match="no kept solution"):
        s.solution(ids[0])
    s.run(realtime=False)
    first = [s.solution(q) for q in ids]
    for q, n in enumerate(sizes):
        print(f"case served solution {n}", flush=True)
        a = MGSolver(n, "mixed", p)
        a.set_rhs_blobs(7 + q)
        a.solve()
        assert np.array_equal(first[q], a.solution())
    s.run(realtime=False)  # the requests once more, into the memory they have
    for q, u in zip(ids, first):
        assert np.isfinite(s.solution(q)).all() and s.solution(q).shape == u.shape


@pytest.mark.parametrize("precision", ["mixed", "fp64"])
def test_requests_solved_again(precision):
    # the limit on V-cycles holds for each run by itself: every run gives the same counts,
    # residuals and bits, though the counts of three runs together are past the limit
    print(f"case served again {precision}", flush=True)
    s = Server(precision, MGParams(residual_tolerance=1e-8, max_iters=30), keep_solutions=True)
    ids = [s.submit(n, 3 + q) for q, n in enumerate((16, 24, 32, 64))]
    runs = []
    for _ in range(3):
        s.run(realtime=False)
        runs.append([(s.result(q)["iters"], s.result(q)["rel_residual"], s.solution(q))
                     for q in ids])
    for run in runs:
        for (it, rel, u), (it0, rel0, u0) in zip(run, runs[0]):
            assert it == it0 and 10 < it < 30 and rel == rel0 < 1e-8
            assert np.array_equal(u, u0) and np.abs(u).max() > 0
