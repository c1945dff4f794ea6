"""2D parity chains in LDS at lines that end anywhere in an octet of sites or a word: the
lattice's way into words and back, one pass a run.  One chain and many (other word sizes);
equal to the byte kernels (OPT_CHECKER_QUAD_PATH) in every value."""
import numpy as np
import pytest

import casmcode_monte_amd as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("J2", [0.0, -0.02])
@pytest.mark.parametrize("lines", [2, 6])
@pytest.mark.parametrize("chains", [1, 700])
def test_line_ends(chains, lines, J2):
    for L0 in (2, 4, 6, 14, 16, 18, 30, 32, 34, 46, 48, 50, 62, 64, 66, 80, 112, 126, 128, 130,
               1008, 4096):
        got = []
        for options in (0, M.OPT_CHECKER_QUAD_PATH):
            print("line ends", chains, lines, J2, L0, options, flush=True)
            with M.Run([dict(shape=(L0, lines), temperature=1700.0, exchange_potential=0.03,
                             seed=20 + i) for i in range(chains)], mode=M.MODE_CHECKERBOARD,
                       J1=0.1, J2=J2, options=options) as r:
                rng = np.random.default_rng(L0)
                for c in (0, chains - 1):
                    r.set_occupation(c, np.where(rng.random(L0 * lines) < 0.5, 1, -1))
                for passes in (1, 1, 2):
                    r.run(passes)
                got.append([(r.samples(c), r.get_occupation(c), r.counters(c))
                            for c in sorted({0, chains // 2, chains - 1})])
        for (sa, oa, ca), (sb, ob, cb) in zip(*got):
            assert np.array_equal(sa, sb) and np.array_equal(oa, ob) and ca == cb, L0
