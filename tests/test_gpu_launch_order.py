"""The work-group order changes no result bit: XCD slabs, the hardware's order and XCD chunks,
on lattices whose block count is below one group of chunks, a whole number of groups, and
groups with a remainder (64 blocks a group)."""
import numpy as np
import pytest

import lbffs_amd as lb
from lbffs_amd import cases

pytestmark = pytest.mark.gpu

NO_XCD, XCD_CHUNK = 2, 64


@pytest.mark.parametrize("q", [19, 27])
@pytest.mark.parametrize("dims", [(40, 24, 12), (64, 32, 16), (70, 37, 15)])
def test_orders_agree(dims, q):
    nx, ny, nz = dims
    c = cases.cylinder_channel(nx=nx, ny=ny, nz=nz, D=ny // 4, cx=nx // 3, cy=ny // 2, spz_cells=4, q=q, ibb=True)
    ref = None
    for block in (64, 256):
        for tune in (0, NO_XCD, XCD_CHUNK):
            with lb.Lattice(nx, ny, nz, q=q, storage=lb.STORE_F16DEV, sgs=c.sgs, collision=c.coll, omega0=c.omega0) as lat:
                c.upload_to(lat)
                lat.set_launch(block, tune)
                lat.step(6, **c.params)
                f = lat.download("f")
            ref = f if ref is None else ref
            assert np.array_equal(f, ref), (block, tune)
