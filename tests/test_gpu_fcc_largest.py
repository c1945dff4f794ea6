"""The largest FCC lattice whose lines the class-line kernel keeps in LDS, beside what the
kernel has static there (the handle refuses a kernel for which the two do not fit), against
the kernel on HBM."""
import numpy as np
import pytest

import casmcode_monte_amd as M
from casmcode_monte_amd import fcc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(32, 56, 64), (5, 56, 64), (3, 28, 127)])
def test_largest(shape):
    runs = []
    for options in (0, M.OPT_FORCE_STREAMING):
        print("fcc largest", shape, options, flush=True)
        with M.Run([dict(shape=shape, temperature=900.0, exchange_potential=0.1, seed=3)],
                   mode=M.MODE_CHECKERBOARD, lattice=M.LATTICE_FCC, eci=fcc.DEFAULT_ECI,
                   options=options) as r:
            r.set_occupation(0, np.random.default_rng(2).integers(0, 2, 4 * int(np.prod(shape)))
                             .astype(np.int8))
            r.run(2)
            runs.append((r.samples(0), r.get_occupation(0), r.counters(0)))
    (sa, oa, ca), (sb, ob, cb) = runs
    assert np.array_equal(sa, sb) and np.array_equal(oa, ob) and ca == cb
