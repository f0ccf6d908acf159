"""bit_exact without stored fluxes: on block shapes that the sweeps serve, a U declared without
WithFluxes still takes the form whose bits are the oracle's, eager and captured."""
import numpy as np
import pytest

import parthenon_amd as pa
from oracle_lib import OracleBurgers, OracleMesh, lib
from parthenon_amd.burgers import DeviceBurgersDriver

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("use_graph", [False, True])
@pytest.mark.parametrize("block,scalars,recon", [(32, 2, 0), (16, 4, 0), (16, 6, 1), (8, 1, 0),
                                                 (12, 2, 0)])
def test_bit_exact_without_fluxes(block, scalars, recon, use_graph):
    print(f"case bit exact {block} {scalars} {recon} {use_graph}", flush=True)
    nx = (2 * block, block, block)
    ob = OracleBurgers(OracleMesh(nx, (block,) * 3, 4), scalars, 0.4, recon)
    lib().orc_burgers_pgen_sinusoid(ob.h, 3)
    lib().orc_burgers_initialize(ob.h)
    m = pa.Mesh(nx, (block,) * 3, 4)
    m.add_field("U", 3 + scalars, pa.Metadata.FillGhost | pa.Metadata.Independent)
    m.add_field("derived", 1, pa.Metadata.OneCopy)
    m.finalize()
    d = DeviceBurgersDriver(m, cfl=0.4, recon=recon, use_graph=use_graph, bit_exact=True)
    d.initialize("sinusoid", seed=3)
    assert d.form() == "serial"
    d.cycles(2)
    ob.cycles(2)
    assert np.array_equal(d.base.download("U").ravel(), ob.get(0))
    assert d.clock()[0] == ob.dt
