"""The markers' spread against the sum of marker forcing times trilinear weight in FP64: a wave's
markers all in one cell (every corner shared), no two corners shared (the fullest table of a
work-group), and in between; FP32 and FP64.  Tolerance: each cell's sum of m terms rounds at most m
times, each term's weight and product 8 times more."""
import numpy as np
import pytest

import lbffs_amd as lb
from lbffs_amd import cases

pytestmark = pytest.mark.gpu


def markers(kind):
    rng = np.random.default_rng(7)
    if kind == "one cell":
        return np.array([20.0, 9.0, 11.0]) + rng.uniform(0.1, 0.9, (300, 3))
    grid = np.stack(np.meshgrid(np.arange(2, 38, 2), np.arange(2, 22, 2), np.arange(2, 18, 2), indexing="ij"), -1)
    if kind == "all apart":
        return grid.reshape(-1, 3) + rng.uniform(0.1, 0.9, (grid.size // 3, 3))
    return rng.uniform([1, 1, 1], [38, 22, 18], size=(1000, 3))


@pytest.mark.parametrize("storage", [lb.STORE_F32, lb.STORE_F64])
@pytest.mark.parametrize("kind", ["one cell", "all apart", "scattered"])
def test_spread(kind, storage):
    c = cases.periodic_box(40, 24, 20, ini=(0.05, 0.02, 0.01))
    with lb.Lattice(c.nx, c.ny, c.nz, storage=storage, sgs=c.sgs, omega0=c.omega0) as lat:
        real = lat.real
        xyz = markers(kind).astype(real)
        c.upload_to(lat)
        lat.ibm_set_markers(xyz)
        lat.ibm_set_motion(trans=(1e-3, 0, 0), center=(20, 12, 0), axis=(0, 0, 1), omega=1e-3)
        lat.step(1, **c.params)
        g = lat.ibm_download(lb.IBM_FORCING).reshape(3, -1).astype(np.float64)
        got = [lat.download(k).astype(np.float64) for k in ("GxIBM", "GyIBM", "GzIBM")]
    x = xyz.astype(np.float64)
    lo = np.floor(x).astype(int)
    assert np.abs(g).max() > 0
    for a in range(3):
        want, size, terms = (np.zeros(c.nx * c.ny * c.nz) for _ in range(3))
        for b in range(8):
            at = lo + [b & 1, (b >> 1) & 1, b >> 2]
            t = g[a] * np.prod(1 - np.abs(at - x), axis=1)
            ic = at[:, 0] + c.nx * (at[:, 1] + c.ny * at[:, 2])
            np.add.at(want, ic, t)
            np.add.at(size, ic, np.abs(t))
            np.add.at(terms, ic, 1)
        assert np.all(np.abs(got[a] - want) <= (terms + 8) * np.finfo(real).eps * size)
