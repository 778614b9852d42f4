"""Batches whose lattices together fit the Infinity Cache (80 MB to 256 MB a step, 16-bit values
224 MB) store their populations to stay there: bit for bit what the same batch gives with the stores
streamed past it (LBFFS_TUNE_NT_STORE on every lattice), below, inside and above that range."""
import numpy as np
import pytest

import lbffs_amd as lb
from lbffs_amd import cases

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("q,storage,edges", [(19, lb.STORE_F16DEV, (80, 70, 41)), (19, lb.STORE_F16DEV, (110, 90, 53)),
                                             (19, lb.STORE_F32, (20, 33)), (19, lb.STORE_F32, (90, 64, 31)),
                                             (19, lb.STORE_F32, (100, 90, 31)), (19, lb.STORE_F64, (64, 33, 40)),
                                             (27, lb.STORE_BF16DEV, (90, 40, 37)), (27, lb.STORE_F32, (75, 33))])
def test_kept_and_streamed(q, storage, edges):
    cs = [cases.cavity(e, q=q) if i % 2 else cases.periodic_box(e, e, e, sgs=lb.SGS_WALE, q=q, ini=(0.05, 0.02, 0.01))
          for i, e in enumerate(edges)]
    rng = np.random.default_rng(2)
    for c in cs:
        c.arrays["f"] = c.arrays["f"] * (1 + 0.01 * rng.standard_normal(c.arrays["f"].size).astype(np.float32))
    out = []
    for tune in (0, 1):
        batch = lb.Batch([(c.nx, c.ny, c.nz, c.omega0) for c in cs], q=q, storage=storage)
        for c, lat in zip(cs, batch.lattice):
            c.upload_to(lat)
            lat.set_launch(256, tune)
        batch.step(5, [c.params for c in cs])
        out.append([np.concatenate([lat.download(k) for k in ("f", "rho", "u", "v", "w")]) for lat in batch.lattice])
        del batch
    for a, b in zip(*out):
        assert np.isfinite(a).all()
        assert np.array_equal(a, b)
