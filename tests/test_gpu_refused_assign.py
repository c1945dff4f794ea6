"""A refused assignment leaves the handle as it was: its chains go on as if nothing had
been asked."""
import numpy as np
import pytest

import casmcode_monte_amd as M
import oracle as O

pytestmark = pytest.mark.gpu


def test_canonical_long_thin_shape():
    """As many sites as the slot holds in one line: its fold scratch does not fit LDS."""
    rows, cols, T = 193, 193, 2500.0
    occ = -np.ones(rows * cols, np.int8)
    occ[np.random.default_rng(5).permutation(rows * cols)[:9000]] = 1
    print("canonical refused", flush=True)
    with M.Run([dict(shape=(rows, cols), temperature=T, seed=31),
                dict(shape=(rows, cols), temperature=T, seed=32)], mode=M.MODE_CANONICAL,
               J1=0.1, sample_period=1) as r:
        for c in range(2):
            r.set_occupation(c, occ)
        r.run(1)
        with pytest.raises(RuntimeError, match="LDS"):
            r.assign(1, dict(shape=(1, rows * cols), temperature=T, seed=33))
        r.run(1)
        for c in range(2):
            o = O.canonical_run(rows, cols, 0.1, T, 2, occ, O.mt64_state(31 + c, 0))
            assert np.array_equal(r.get_occupation(c), o["occ"])
            assert np.array_equal(r.rng_dump(c), o["engine"])
            assert np.array_equal(r.samples(c)["S1"], o["S"])
