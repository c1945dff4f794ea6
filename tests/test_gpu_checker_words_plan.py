"""2D chains that fit a workgroup: the words kernel's plan follows the chains that run, when
others take part and when slots get other shapes.  Equal to the byte kernels
(OPT_CHECKER_QUAD_PATH) in every value."""
import numpy as np
import pytest

import casmcode_monte_amd as M

pytestmark = pytest.mark.gpu

SHAPES = [(128, 128), (30, 34), (31, 45), (8, 200), (250, 252), (101, 64)]


@pytest.mark.parametrize("J2", [0.0, -0.02])
def test_plan_follows_the_chains(J2):
    runs = []
    for options in (0, M.OPT_CHECKER_QUAD_PATH):
        print("words plan", J2, options, flush=True)
        r = M.Run([dict(shape=s, temperature=900.0 + 300.0 * i, exchange_potential=0.02,
                        seed=60 + i) for i, s in enumerate(SHAPES)], mode=M.MODE_CHECKERBOARD,
                  J1=0.1, J2=J2, options=options)
        out = []

        def run(passes):
            r.run(passes)
            out.extend((r.samples(c), r.get_occupation(c), r.counters(c))
                       for c in range(len(SHAPES)))

        r.set_active([0, 1, 0, 1, 0, 0])
        run(1)
        r.set_active([1, 1, 1, 0, 0, 0])  # larger, and one with an odd edge
        run(3)
        r.set_active([0, 0, 0, 0, 1, 1])
        run(2)
        r.assign(4, dict(shape=(251, 250), temperature=1500.0, exchange_potential=0.0, seed=70))
        r.assign(2, dict(shape=(44, 30), temperature=1500.0, exchange_potential=0.0, seed=71))
        run(2)
        r.set_active([1, 1, 1, 1, 1, 1])
        run(5)
        runs.append(out)
        r.close()
    for (sa, oa, ca), (sb, ob, cb) in zip(*runs):
        assert np.array_equal(sa, sb) and np.array_equal(oa, ob) and ca == cb
