"""CalculateFluxes and the driver's flux form on block shapes other than the cubic 8 / 16 ones,
against the oracle: the flux kernel's row pieces (63 new cells a wavefront) and column segments
(at most 9 faces) end at every kind of remainder."""
import numpy as np
import pytest

import parthenon_amd as pa
from oracle_lib import OracleBurgers, OracleMesh, lib
from parthenon_amd.burgers import DeviceBurgersDriver, make_burgers_mesh

pytestmark = pytest.mark.gpu

# mesh, block, scalars, recon; blocks of one segment (8), of segments 9 + 8 (16), of unequal
# ones (10, 12, 20, 32), a mesh of one block and more components than any fixed unroll
SHAPES = [
    ((24, 20, 16), (12, 10, 8), 4, 0),
    ((40, 16, 24), (20, 16, 12), 1, 0),
    ((32, 32, 32), (32, 32, 32), 8, 0),
    ((16, 16, 16), (16, 16, 16), 4, 0),
    ((20, 12, 16), (10, 12, 8), 15, 1),
]


@pytest.mark.parametrize("nx,block,ns,recon", SHAPES)
def test_fluxes_match_oracle_bit_for_bit(nx, block, ns, recon):
    print(f"case fluxes {nx} {block} scalars {ns} recon {recon}", flush=True)
    m = make_burgers_mesh(nx, block, 4, ns)
    ob = OracleBurgers(OracleMesh(nx, block, 4), ns, 0.4, recon)
    lib().orc_burgers_pgen_sinusoid(ob.h, 5)
    lib().orc_burgers_initialize(ob.h)
    md = m.mesh_data("base")
    md.upload("U", ob.get(0).reshape(m.field_shape("U")))
    pa.burgers_package.CalculateFluxes(md, recon)
    lib().orc_burgers_fluxes(ob.h)
    F = md.download("U", which=2)
    n, g = m.n, m.ng
    for d in range(3):
        exp = ob.get(4 + d).reshape(F[d].shape)
        sl = tuple(slice(g[2 - a], g[2 - a] + n[2 - a] + (1 if 2 - a == d else 0))
                   for a in range(3))
        assert np.array_equal(F[d][(slice(None), slice(None)) + sl],
                              exp[(slice(None), slice(None)) + sl]), f"x{d + 1} faces"


@pytest.mark.parametrize("nx,block,boxes", [
    ((24, 20, 24), (12, 10, 8), ()),
    ((48, 48, 48), (12, 12, 12), [((-0.1, 0.1, -0.1, 0.1, -0.1, 0.1), 1)]),
], ids=["uniform", "refined"])
def test_driver_other_blocks_matches_oracle(nx, block, boxes):
    print(f"case driver {nx} {block}", flush=True)
    m = make_burgers_mesh(nx, block, 4, 2, refine_boxes=boxes)
    d = DeviceBurgersDriver(m, cfl=0.4, use_graph=True)
    d.initialize("sinusoid", seed=4)
    ob = OracleBurgers(OracleMesh(nx, block, 4, boxes=boxes), 2, 0.4, 0)
    lib().orc_burgers_pgen_sinusoid(ob.h, 4)
    lib().orc_burgers_initialize(ob.h)
    for _ in range(2):
        d.cycles(2)
        ob.cycles(2)
        assert np.array_equal(d.base.download("U").ravel(), ob.get(0))
    assert d.clock()[0] == ob.dt


# the flux kernel's splits: small blocks that share workgroups (the last unit not full), components
# in groups, 2-D and 1-D; and meshes that it takes by column segments: 2304 blocks of one segment of
# 9 faces in units of several blocks, large blocks whose last segments are short, in stripes, 2-D
SPLITS = [
    ((88, 8, 8), (8, 8, 8), 6, 0),
    ((40, 40, 40), (10, 10, 10), 1, 1),
    ((72, 40, 1), (8, 8, 1), 5, 0),
    ((96, 1, 1), (8, 1, 1), 2, 0),
    ((128, 96, 96), (8, 8, 8), 1, 0),
    ((192, 100, 76), (96, 100, 76), 1, 1),
    ((1024, 1024, 1), (128, 128, 1), 1, 0),
]


@pytest.mark.parametrize("nx,block,ns,recon", SPLITS)
def test_flux_splits_match_oracle_bit_for_bit(nx, block, ns, recon):
    print(f"case flux split {nx} {block} scalars {ns} recon {recon}", flush=True)
    test_fluxes_match_oracle_bit_for_bit(nx, block, ns, recon)
