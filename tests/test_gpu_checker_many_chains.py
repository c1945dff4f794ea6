"""More chains on the bit-packed path than a grid's second dimension takes."""
import numpy as np
import pytest

import casmcode_monte_amd as M

pytestmark = pytest.mark.gpu


def test_seventy_thousand_chains():
    n = 70000
    chains = [dict(shape=(32, 2), temperature=1000.0 + i % 977, seed=i) for i in range(n)]
    look = [0, 1, 65534, 65535, 65536, n - 1]
    got = []
    for bands in (-1, 0):
        print("many chains", bands, flush=True)
        with M.Run(chains, mode=M.MODE_CHECKERBOARD, J1=0.1, options=M.OPT_FORCE_STREAMING) as r:
            r.set_schedule(band_lines=bands)
            for c in look:
                r.set_occupation(c, np.where(np.random.default_rng(c).random(64) < 0.5, 1, -1))
            r.run(1)
            r.run(2)
            got.append([(r.samples(c), r.get_occupation(c), r.counters(c)) for c in look])
    for (sa, oa, ca), (sb, ob, cb) in zip(*got):
        assert np.array_equal(sa, sb) and np.array_equal(oa, ob) and ca == cb
