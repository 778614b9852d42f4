"""Uploads and downloads through the pinned ring (2 MiB chunks, eight of them): fields below
the ring's smallest copy, of whole and broken chunks, and longer than the ring; two threads at
once, one of which finds the ring taken; populations in every storage form."""
import threading

import numpy as np
import pytest

import lbffs_amd as lb
from lbffs_amd import cases

pytestmark = pytest.mark.gpu


def _round_trip(lat, name, rng):
    a = rng.standard_normal(lat.N).astype(lat.real)
    lat.upload(name, a)
    assert np.array_equal(lat.download(name), a)


# FP32 fields of 4 MiB - 128 B, 4 MiB, 4 MiB + 64 B, 7 chunks and a rest, 17 chunks and a rest
@pytest.mark.parametrize("dims", [(32, 32767, 1), (1024, 1024, 1), (16, 65537, 1), (1000, 997, 4), (1013, 1009, 9)])
def test_field_round_trip(dims):
    nx, ny, nz = dims
    rng = np.random.default_rng(nx)
    with lb.Lattice(nx, ny, nz) as lat:
        for name in ("u0", "sdf"):
            _round_trip(lat, name, rng)


@pytest.mark.parametrize("storage", [lb.STORE_F32, lb.STORE_F16DEV, lb.STORE_F64])
def test_populations_round_trip(storage):
    c = cases.channel(nx=130, ny=60, nz=33, tau=0.7)
    f = c.arrays["f"] * (1 + 0.01 * np.random.default_rng(1).standard_normal(c.arrays["f"].size))
    with lb.Lattice(c.nx, c.ny, c.nz, storage=storage, omega0=c.omega0) as lat:
        lat.upload("f", f)
        back = lat.download("f")
        lat.upload("f", back)
        assert np.array_equal(lat.download("f"), back)
        exact = f.astype(lat.real)
        if storage == lb.STORE_F16DEV:
            # half precision of the deviation from the weight, itself below 0.04 of it
            assert np.abs(back - exact).max() <= 2.0 ** -11 * 0.1
        else:
            assert np.array_equal(back, exact)


def test_two_threads():
    errors = []

    def work(seed):
        try:
            rng = np.random.default_rng(seed)
            with lb.Lattice(1024, 700, 8) as lat:
                for _ in range(6):
                    _round_trip(lat, "u0", rng)
        except BaseException as e:  # reported by the main thread
            errors.append(e)

    threads = [threading.Thread(target=work, args=(s,)) for s in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
