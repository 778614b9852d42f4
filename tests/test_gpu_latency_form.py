"""D3Q19's form for small lattices (flags, face velocities and WALE's neighbours loaded ahead) against
the form that runs the faces in work-groups of their own, bit for bit: every face code, 2-D and
one-cell-wide lattices, a wave and a rest, solid cells, and the largest lattice of each storage form
beside the next one, which takes the other form."""
import numpy as np
import pytest

import lbffs_amd as lb
from lbffs_amd import cases

pytestmark = pytest.mark.gpu

NO_PURE, SPLIT, FACE_FIRST = 16, 8, 32
DIMS = [(32, 32, 32), (64, 12, 8), (70, 9, 7), (20, 11, 1), (2, 40, 6), (3, 5, 4), (17, 3, 33)]
FACES = [("FixedVelocity", "Outlet"), ("BounceBack", "BounceBack"), ("Cyclic", "Cyclic"), ("FixedVelocity", "FixedDensity"),
         ("Symmetry", "Symmetry"), ("WallFunction", "WallFunction")]


def run(c, storage, sgs, tune, steps=5):
    with lb.Lattice(c.nx, c.ny, c.nz, storage=storage, sgs=sgs, omega0=c.omega0) as lat:
        c.upload_to(lat)
        lat.set_launch(128, tune)
        lat.step(steps, **c.params)
        return np.concatenate([lat.download(k) for k in ("f", "rho", "u", "v", "w", "tauSGS", "Fwx")])


def check(c, storage, sgs):
    rng = np.random.default_rng(5)
    c.arrays["f"] = (c.arrays["f"] * (1 + 0.01 * rng.standard_normal(c.arrays["f"].size))).astype(np.float32)
    ref = run(c, storage, sgs, SPLIT)
    assert np.isfinite(ref).all()
    for tune in (0, NO_PURE, FACE_FIRST):
        assert np.array_equal(run(c, storage, sgs, tune), ref), tune


@pytest.mark.parametrize("storage", [lb.STORE_F32, lb.STORE_F64, lb.STORE_F16DEV])
@pytest.mark.parametrize("sgs", [lb.SGS_WALE, lb.SGS_SMAGORINSKY])
@pytest.mark.parametrize("faces", FACES)
@pytest.mark.parametrize("dims", DIMS)
def test_small_lattices(dims, faces, sgs, storage):
    nx, ny, nz = dims
    codes = {f: ("Cyclic", "Cyclic", "Cyclic") for f in cases.FACES}
    if faces[0] == "WallFunction":  # wall faces of the y axis
        codes["nyMin"], codes["nyMax"] = (("Cyclic", f, "Cyclic") for f in faces)
    else:
        codes["nxMin"], codes["nxMax"] = ((f, "Cyclic", "Cyclic") for f in faces)
        codes["nyMin"] = codes["nyMax"] = ("Cyclic", "BounceBack", "Cyclic")
    vels = {"nxMin": (0.5, 0.1, 0.05), "nxMax": (-0.4, 0.1, 0.0)}
    c = cases.make_case("x", nx, ny, nz, 1.0, 1.0, 0.05, 2e-3, codes, vels, ini=(0.3, 0.1, 0.0), q=19, spzWidth=0.2)
    check(c, storage, sgs)


@pytest.mark.parametrize("storage,dims", [(lb.STORE_F64, (64, 32, 32)), (lb.STORE_F64, (65, 32, 32)),
                                          (lb.STORE_F32, (64, 64, 48)), (lb.STORE_F32, (64, 64, 49)),
                                          (lb.STORE_BF16DEV, (64, 64, 64)), (lb.STORE_BF16DEV, (64, 64, 65))])
def test_its_last_lattice(storage, dims):
    check(cases.periodic_box(*dims, sgs=lb.SGS_WALE, ini=(0.05, 0.02, 0.01)), storage, lb.SGS_WALE)


@pytest.mark.parametrize("storage", [lb.STORE_F32, lb.STORE_F64])
def test_solid_cells(storage):
    c = cases.cavity(24)
    solid = np.zeros((24, 24, 24), np.uint8)
    solid[8:12, 9:15, 7:13] = 1
    c.arrays["solid"] = solid.reshape(-1)
    c.arrays["neiSolid"] = cases.neisolid(19, 24, 24, 24, c.arrays["solid"])
    check(c, storage, lb.SGS_WALE)
