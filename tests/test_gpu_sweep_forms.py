"""The block sweep's own arithmetic against the oracle at the edges of its range, through the
C ABI: WENO5Z formed from differences beside jumps far larger and far smaller than the
tests of the trajectories use."""
import numpy as np
import pytest

from oracle_lib import OracleBurgers, OracleMesh, lib
from parthenon_amd.burgers import DeviceBurgersDriver, make_burgers_mesh

pytestmark = pytest.mark.gpu


def assert_close(got, exp, what, tol=1e-13):
    scale = np.max(np.abs(exp))
    err = np.max(np.abs(got - exp)) / (scale if scale > 0 else 1.0)
    assert err <= tol, f"{what}: relative error {err:.3e}"


@pytest.mark.parametrize("jump", [1e45, 1e-150], ids=["large", "tiny"])
@pytest.mark.parametrize("n", [16, 8])
def test_sweep_scalar_jump_matches_oracle(n, jump):
    # a passive scalar with a jump, flat on both sides; 1e-13 of the scalar's own maximum is
    # the bound of every sweep test (two cycles of a few ulp each)
    print(f"case sweep jump {jump} block {n}", flush=True)
    m = make_burgers_mesh((2 * n,) * 3, (n,) * 3, 4, 4)
    d = DeviceBurgersDriver(m, cfl=0.4, use_graph=False, sweep=True)
    ob = OracleBurgers(OracleMesh((2 * n,) * 3, (n,) * 3, 4), 4, 0.4, 0)
    lib().orc_burgers_pgen_sinusoid(ob.h, 6)
    U = ob.get(0).reshape(m.field_shape("U"))
    g = m.ng[0]
    for b in range(m.nblocks):
        info = m.block(b)
        x = info["xmin"][0] + (np.arange(n) + 0.5) * (info["xmax"][0] - info["xmin"][0]) / n
        U[b, 4, g:-g, g:-g, g:-g] = np.where(x > 0.0, jump, 0.0)[None, None, :]
    ob.set(0, U.ravel())
    lib().orc_burgers_initialize(ob.h)
    d.base.upload("U", U)
    d.initialize("none")
    d.cycles(2)
    ob.cycles(2)
    got = d.base.download("U")
    exp = ob.get(0).reshape(got.shape)
    assert np.isfinite(got).all()
    for c in range(got.shape[1]):
        assert_close(got[:, c], exp[:, c], f"component {c}")
