"""3D J1+J2 lattices of few large planes, on either side of the size from which a plane a
workgroup is worth it, alone and beside small ones: equal to the kernels on bytes
(band_lines=0) in every value."""
import numpy as np
import pytest

import casmcode_monte_amd as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shapes", [[(512, 512, 2)], [(512, 512, 18)], [(192, 900, 4)],
                                    [(512, 640, 2), (64, 8, 6)], [(128, 1536, 4)],
                                    [(512, 512, 8), (512, 512, 10)]])
def test_large_planes(shapes):
    got = []
    for schedule in (dict(band_lines=0, graph_passes=1), dict(graph_passes=1),
                     dict(graph_passes=8)):
        print("large planes", shapes, schedule, flush=True)
        with M.Run([dict(shape=s, temperature=1500.0 + 500.0 * i, exchange_potential=0.02,
                         seed=80 + i) for i, s in enumerate(shapes)], mode=M.MODE_CHECKERBOARD,
                   lattice=M.LATTICE_SC, J1=0.1, J2=-0.02) as r:
            r.set_schedule(**schedule)
            for c, s in enumerate(shapes):
                r.set_occupation(c, np.where(np.random.default_rng(c).random(int(np.prod(s))) < 0.5,
                                             1, -1))
            for passes in (1, 9):
                r.run(passes)
            got.append([(r.samples(c), r.get_occupation(c), r.counters(c))
                        for c in range(len(shapes))])
    for other in got[1:]:
        for (sa, oa, ca), (sb, ob, cb) in zip(got[0], other):
            assert np.array_equal(sa, sb) and np.array_equal(oa, ob) and ca == cb
