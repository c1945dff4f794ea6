"""EXACT launches of a few attempts: chains on either side of the length from which a large
lattice takes the block walk, chains of both walks in one launch, a handle whose chains all
live in HBM.  Bit-exact against the scalar walk (OPT_EXACT_SCALAR_WALK)."""
import numpy as np
import pytest

import casmcode_monte_amd as cm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shapes", [[(1, 1)], [(400, 400)], [(512, 512), (64, 64)],
                                    [(600, 600), (390, 380), (30, 20)], [(600, 600), (513, 512)]])
@pytest.mark.parametrize("use_nlist", [True, False])
def test_short_launches(shapes, use_nlist):
    runs = []
    for options in (0, cm.OPT_EXACT_SCALAR_WALK):
        print("case:", shapes, use_nlist, options, flush=True)
        r = cm.Run([dict(shape=s, temperature=2400.0, exchange_potential=0.02, seed=70 + i)
                    for i, s in enumerate(shapes)], mode=cm.MODE_EXACT, J1=0.1,
                   use_nlist=use_nlist, options=options)
        for c, s in enumerate(shapes):
            n = s[0] * s[1]
            r.set_occupation(c, np.where(np.random.default_rng(n).random(n) < 0.5, 1, -1))
        for steps in (1, 493, 494, 532, 533, 873, 874, 2000, 7):
            r.run_steps(steps)
        runs.append(r)
    a, b = runs
    for c in range(len(shapes)):
        np.testing.assert_array_equal(a.get_occupation(c), b.get_occupation(c))
        np.testing.assert_array_equal(a.rng_dump(c), b.rng_dump(c))
        np.testing.assert_array_equal(a.samples(c), b.samples(c))
        assert a.counters(c) == b.counters(c) and a.position(c) == b.position(c)
    for r in runs:
        r.close()
