"""New populations stored to stay in the Infinity Cache (steps of 80 MB to 256 MB) against the same
steps with the stores streamed past it (LBFFS_TUNE_NT_STORE): the two must agree bit for bit, over
cavity walls, rows that are no multiple of a wave, and both rounding modes of the 16-bit forms."""
import numpy as np
import pytest

import lbffs_amd as lb
from lbffs_amd import cases

pytestmark = pytest.mark.gpu

NT_STORE, SPLIT, FACE_FIRST = 1, 8, 32

# cells whose step takes just over 80 MB and just under 256 MB
CASES = [(19, lb.STORE_F32, (76, 76, 76)), (19, lb.STORE_F32, (128, 112, 100)), (19, lb.STORE_F64, (64, 64, 64)),
         (19, lb.STORE_F16DEV, (96, 97, 90)), (19, lb.STORE_BF16DEV, (129, 130, 131)), (27, lb.STORE_F32, (70, 70, 70)),
         (27, lb.STORE_F64, (65, 66, 67)), (27, lb.STORE_BF16DEV, (110, 120, 130))]


@pytest.mark.parametrize("q,storage,dims", CASES)
def test_kept_and_streamed(q, storage, dims):
    c = cases.cavity(dims[0], nz=dims[2], q=q) if dims[0] == dims[1] else cases.periodic_box(*dims, sgs=lb.SGS_WALE, q=q, ini=(0.05, 0.02, 0.01))
    rng = np.random.default_rng(1)
    c.arrays["f"] = (c.arrays["f"] * (1 + 0.01 * rng.standard_normal(c.arrays["f"].size).astype(np.float32)))
    ref = None
    for tune in (NT_STORE, 0, SPLIT, FACE_FIRST):
        with lb.Lattice(c.nx, c.ny, c.nz, q=q, storage=storage, sgs=c.sgs, omega0=c.omega0) as lat:
            c.upload_to(lat)
            lat.set_launch(128, tune)
            lat.step(5, **c.params)
            got = np.concatenate([lat.download(k) for k in ("f", "rho", "u", "v", "w")])
        assert np.isfinite(got).all()
        ref = got if ref is None else ref
        assert np.array_equal(got, ref), tune
