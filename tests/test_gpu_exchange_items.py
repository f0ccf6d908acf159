"""Boundary copies of one wavefront per item: region sizes around the wavefront's 64 elements and
the item's 1024, counts of items that do not fill the last workgroup, the smallest mesh. The
ghosts are the wrapped interior, bit for bit, in each form of the exchange."""
import numpy as np
import pytest

import parthenon_amd as pa
from meshcheck import global_index_field, interior_mask

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form", ["tasks", "fused"])
@pytest.mark.parametrize("nx,block,g,ncomp", [
    ((4, 4, 4), (4, 4, 4), 2, 1),        # one block: 8, 16 and 32 elements a region
    ((8, 8, 8), (4, 4, 8), 4, 1),        # 64, 64 and 128
    ((10, 6, 10), (5, 6, 5), 3, 1),      # 27 .. 90
    ((16, 16, 32), (16, 16, 16), 4, 1),  # faces of 1024
    ((12, 20, 20), (12, 10, 20), 3, 5),  # 135 .. 3000: several items a region
    ((34, 34, 17), (17, 17, 17), 4, 1),  # faces of 1156: an item of 132 after the first
])
def test_ghosts_are_the_wrapped_interior(nx, block, g, ncomp, form):
    print(f"case items nx={nx} block={block} g={g} ncomp={ncomp} {form}", flush=True)
    m = pa.Mesh(nx, block, g)
    m.add_field("q", ncomp, pa.Metadata.FillGhost | pa.Metadata.Independent)
    m.finalize()
    md = m.mesh_data("base")
    exp = global_index_field(m, ncomp, nx)
    md.upload("q", np.where(interior_mask(m)[None, None], exp, np.nan))
    (pa.exchange_fused if form == "fused" else pa.exchange)(md)
    assert np.array_equal(md.download("q"), exp)
