"""The packed copies of large lattices: allocated once for a handle's slots, not again for
every larger active set (a free waits for all work on the device, other handles' too)."""
import ctypes

import numpy as np
import pytest

import casmcode_monte_amd as M

pytestmark = pytest.mark.gpu


def _free_bytes():
    hip = ctypes.CDLL("libamdhip64.so")
    a, b = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip.hipMemGetInfo(ctypes.byref(a), ctypes.byref(b)) == 0
    return a.value


@pytest.mark.parametrize("shape,lattice", [((4096, 4096), M.LATTICE_SQUARE),
                                           ((256, 256, 256), M.LATTICE_SC)])
def test_larger_active_sets_allocate_nothing(shape, lattice):
    chains = 8
    print("packed memory", shape, flush=True)
    with M.Run([dict(shape=shape, temperature=2000.0, seed=i) for i in range(chains)],
               mode=M.MODE_CHECKERBOARD, lattice=lattice, J1=0.1, J2=-0.02) as r:
        r.reserve_samples(64)
        r.set_active([1] + [0] * (chains - 1))
        r.run(2)
        left = _free_bytes()
        for k in range(2, chains + 1):
            r.set_active([1] * k + [0] * (chains - k))
            r.run(2)
        # seven more packed copies are 14 to 29 MB
        assert left - _free_bytes() < 6 << 20
        rec = r.samples(chains - 1)
    with M.Run([dict(shape=shape, temperature=2000.0, seed=chains - 1)],
               mode=M.MODE_CHECKERBOARD, lattice=lattice, J1=0.1, J2=-0.02) as a:
        a.run(2)
        assert np.array_equal(a.samples(0), rec)
