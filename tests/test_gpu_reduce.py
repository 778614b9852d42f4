"""The FP64 sums of lbffs_reduce against exact sums of the downloaded fields, on lattices
that leave the reduction's rows partly empty, that fill them once, and that fill them many times."""
import math

import numpy as np
import pytest

import lbffs_amd as lb
from lbffs_amd import cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(12, 8, 2), (37, 23, 11), (128, 128, 16), (129, 131, 17)])
@pytest.mark.parametrize("q", [19, 27])
def test_reduce_sums(dims, q):
    nx, ny, nz = dims
    c = cases.cylinder_channel(nx=nx, ny=ny, nz=nz, D=max(4, ny // 4), cx=nx // 3, cy=ny // 2, spz_cells=2, q=q)
    with lb.Lattice(nx, ny, nz, q=q, sgs=c.sgs, collision=c.coll, omega0=c.omega0) as lat:
        c.upload_to(lat)
        lat.step(3, **c.params)
        got = lat.reduce()
        assert np.array_equal(got, lat.reduce())
        fluid = c.arrays["solid"] == 0
        sums = [lat.download(k).astype(np.float64)[fluid] for k in ("Fwx", "Fwy", "Fwz", "GxIBM", "GyIBM", "GzIBM")]
        f = lat.download("f").astype(np.float64).reshape(q, -1)[:, fluid]
    n = int(fluid.sum())
    eps = np.finfo(np.float64).eps
    # an FP64 sum of n terms in any order is off by at most (n - 1) eps sum|x|; each cell's own
    # sum of q populations (total 1) and its difference from 1 add (q + 1) eps
    for k, x in enumerate(sums):
        assert abs(got[k] - math.fsum(x)) <= n * eps * np.abs(x).sum(), k
    excess = np.array([math.fsum(col) - 1.0 for col in f.T])
    assert abs(got[6] - math.fsum(excess)) <= n * eps * np.abs(excess).sum() + n * (q + 1) * 2 * eps
    assert got[7] == n
