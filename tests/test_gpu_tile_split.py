"""The split stage in tile-sweep shapes: the tile form over a list of blocks, on refined meshes
whose lists both hold blocks, split and whole, eager and captured, against the oracle. Bound 1e-13
relative, as for every sweep test."""
import numpy as np
import pytest

from oracle_lib import OracleBurgers, OracleMesh, lib
from parthenon_amd.burgers import DeviceBurgersDriver, make_burgers_mesh

pytestmark = pytest.mark.gpu

# 5 x 2 x 2 periodic base blocks with one in the middle column refined: the blocks of the two
# columns away from it have neighbours of their own level only
BOX = [((-0.05, 0.05, -0.4, -0.1, -0.4, -0.1), 1)]
CASES = {  # block, scalars, recon
    "32x16x16-V6": ((32, 16, 16), 3, 0),
    "32x16x16-V9-linear": ((32, 16, 16), 6, 1),
    "16-V8": ((16, 16, 16), 5, 0),
    "16-V12": ((16, 16, 16), 9, 0),
}


@pytest.mark.parametrize("name", list(CASES))
def test_tile_sweep_over_block_lists(name):
    print(f"case tile split {name}", flush=True)
    block, ns, recon = CASES[name]
    nx = (5 * block[0], 2 * block[1], 2 * block[2])
    ob = OracleBurgers(OracleMesh(nx, block, 4, boxes=BOX), ns, 0.4, recon)
    lib().orc_burgers_pgen_sinusoid(ob.h, 9)
    lib().orc_burgers_initialize(ob.h)
    drivers = []
    for split in (True, False):
        for use_graph in (False, True):
            m = make_burgers_mesh(nx, block, 4, ns, refine_boxes=BOX)
            level = [m.block(b)["level"] for b in range(m.nblocks)]
            inner = [b for b in range(m.nblocks)
                     if all(q["level"] == level[b] for q in m.neighbors(b))]
            assert 0 < len(inner) < m.nblocks
            d = DeviceBurgersDriver(m, cfl=0.4, recon=recon, use_graph=use_graph, sweep=True,
                                    split=split)
            d.initialize("sinusoid", seed=9)
            assert d.form() == "sweep"
            drivers.append(d)
    for _ in range(2):
        ob.cycles(2)
        exp, der = ob.get(0), ob.get(2)
        scale = np.max(np.abs(exp))
        for d in drivers:
            d.cycles(2)
            err = np.max(np.abs(d.base.download("U").ravel() - exp)) / scale
            assert err <= 1e-13, f"U: {err:.3e}"
            err = np.max(np.abs(d.base.download("derived").ravel() - der)) / np.max(np.abs(der))
            assert err <= 1e-13, f"derived: {err:.3e}"
            assert abs(d.clock()[0] - ob.dt) <= 1e-13 * ob.dt
