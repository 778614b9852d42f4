"""D3Q27 waves that mix x-face and interior cells: the kernel that runs them beside their
neighbours against the one where every wave takes its own path (LBFFS_TUNE_NO_PURE), bit for
bit, for the face codes that take either route; rows of whole waves, of a wave and a rest, and
several to a wave; the two cells whose diagonal pull leaves the lattice."""
import numpy as np
import pytest

import lbffs_amd as lb
from lbffs_amd import cases

pytestmark = pytest.mark.gpu

NO_PURE, SPLIT, FACE_FIRST = 16, 8, 32

X_FACES = [("FixedVelocity", "Outlet"), ("BounceBack", "BounceBack"), ("Cyclic", "Cyclic"),
           ("FixedVelocity", "FixedDensity"), ("Symmetry", "Symmetry"), ("Outlet", "FixedVelocity")]


@pytest.mark.parametrize("storage", [lb.STORE_F32, lb.STORE_F64, lb.STORE_BF16DEV])
@pytest.mark.parametrize("faces", X_FACES)
@pytest.mark.parametrize("dims", [(64, 12, 8), (70, 9, 7), (20, 11, 9), (2, 40, 6)])
def test_x_face_waves(dims, faces, storage):
    nx, ny, nz = dims
    codes = {f: ("Cyclic", "Cyclic", "Cyclic") for f in cases.FACES}
    codes["nxMin"], codes["nxMax"] = ((f, "Cyclic", "Cyclic") for f in faces)
    codes["nyMin"] = codes["nyMax"] = ("Cyclic", "BounceBack", "Cyclic")
    vels = {"nxMin": (0.5, 0.1, 0.05), "nxMax": (-0.4, 0.1, 0.0)}
    c = cases.make_case("x", nx, ny, nz, 1.0, 1.0, 0.05, 2e-3, codes, vels, ini=(0.3, 0.1, 0.0), q=27, spzWidth=0.2)
    rng = np.random.default_rng(3)
    c.arrays["f"] = (c.arrays["f"] * (1 + 0.01 * rng.standard_normal(c.arrays["f"].size))).astype(np.float32)
    ref = None
    for tune in (NO_PURE, 0, SPLIT, FACE_FIRST):
        with lb.Lattice(nx, ny, nz, q=27, storage=storage, sgs=c.sgs, collision=c.coll, omega0=c.omega0) as lat:
            c.upload_to(lat)
            lat.set_launch(128, tune)
            lat.step(5, **c.params)
            got = np.concatenate([lat.download(k) for k in ("f", "rho", "u", "v", "w")])
        assert np.isfinite(got).all()
        ref = got if ref is None else ref
        assert np.array_equal(got, ref), tune
