"""The tile sweep (x and y block sizes in multiples of 16, any component count that the sweep
takes) against the oracle: several tiles a block, non-cubic blocks, the smallest z size, every
LDS layout (a y difference tile beside the two staged planes up to 11 components, none at 12 and
13), same-level copies to other blocks and to the block itself, corrected fluxes
on refined meshes and physical faces. Bound 1e-13 relative, as for every sweep test."""
import numpy as np
import pytest

from oracle_lib import OracleBurgers, OracleMesh, lib
from parthenon_amd.burgers import DeviceBurgersDriver, make_burgers_mesh

pytestmark = pytest.mark.gpu

BOX = [((-0.1, 0.1, -0.4, -0.1, -0.4, -0.1), 1)]
OUT = ("outflow", "outflow", "reflect", "outflow", "periodic", "periodic")
# mesh, block, scalars, recon, refined boxes, face conditions
CASES = {
    "z8-V4": ((64, 32, 16), (32, 16, 8), 1, 0, (), None),
    "one-block-V11": ((32, 32, 32), (32, 32, 32), 8, 0, (), None),
    "V8": ((32, 32, 32), (16, 16, 16), 5, 0, (), None),
    "V10-linear": ((48, 32, 24), (48, 16, 12), 7, 1, (), None),
    "V12": ((32, 16, 40), (16, 16, 20), 9, 0, (), None),
    "V13": ((32, 32, 24), (16, 32, 12), 10, 0, (), None),
    "refined-V7": ((96, 32, 32), (32, 16, 16), 4, 0, BOX, None),
    "refined-V13": ((96, 32, 32), (32, 16, 16), 10, 0, BOX, None),
    "faces-V5": ((64, 64, 32), (32, 32, 16), 2, 0, (), OUT),
}


@pytest.mark.parametrize("name", list(CASES))
def test_tile_sweep_matches_oracle(name):
    print(f"case tile sweep {name}", flush=True)
    nx, block, ns, recon, boxes, bcs = CASES[name]
    periodic = (1, 1, 1) if bcs is None else (0, 0, 1)
    om = OracleMesh(nx, block, 4, periodic=periodic, boxes=boxes,
                    **({} if bcs is None else dict(bcs=bcs)))
    ob = OracleBurgers(om, ns, 0.4, recon)
    lib().orc_burgers_pgen_sinusoid(ob.h, 9)
    lib().orc_burgers_initialize(ob.h)
    drivers = []
    for use_graph in (False, True):
        m = make_burgers_mesh(nx, block, 4, ns, refine_boxes=boxes, bcs=bcs)
        d = DeviceBurgersDriver(m, cfl=0.4, recon=recon, use_graph=use_graph, sweep=True)
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


def test_bit_exact_choice_excludes_the_tile_sweep():
    # set_bit_exact keeps the flux form, whose bits are the oracle's, on blocks that the sweep
    # serves too
    print("case bit exact 32^3 blocks", flush=True)
    nx, block = (64, 32, 32), (32, 32, 32)
    ob = OracleBurgers(OracleMesh(nx, block, 4), 2, 0.4, 0)
    lib().orc_burgers_pgen_sinusoid(ob.h, 3)
    lib().orc_burgers_initialize(ob.h)
    d = DeviceBurgersDriver(make_burgers_mesh(nx, block, 4, 2), cfl=0.4, bit_exact=True)
    d.initialize("sinusoid", seed=3)
    assert d.form() == "serial"
    d.cycles(2)
    ob.cycles(2)
    assert np.array_equal(d.base.download("U").ravel(), ob.get(0))


@pytest.mark.parametrize("nx,block,ns,recon,form", [
    ((16, 16, 8), (16, 16, 8), 1, 0, "serial"), ((16, 32, 16), (16, 32, 16), 1, 0, "sweep"),
    ((32, 32, 24), (16, 16, 24), 3, 0, "serial"), ((32, 32, 25), (16, 16, 25), 3, 0, "sweep"),
    ((16, 16, 8), (16, 16, 8), 10, 1, "sweep")])
def test_few_planes_take_the_flux_form(nx, block, ns, recon, form):
    # below 100 planes of 16 x 16 cells (32 with up to 5 components), WENO5
    print(f"case few planes {nx} {block}", flush=True)
    ob = OracleBurgers(OracleMesh(nx, block, 4), ns, 0.4, recon)
    lib().orc_burgers_pgen_sinusoid(ob.h, 6)
    lib().orc_burgers_initialize(ob.h)
    d = DeviceBurgersDriver(make_burgers_mesh(nx, block, 4, ns), cfl=0.4, recon=recon)
    d.initialize("sinusoid", seed=6)
    assert d.form() == form
    d.cycles(4)
    ob.cycles(4)
    exp = ob.get(0)
    assert np.max(np.abs(d.base.download("U").ravel() - exp)) <= 1e-13 * np.max(np.abs(exp))
    assert abs(d.clock()[0] - ob.dt) <= 1e-13 * ob.dt
