"""Records of the paths on bytes, several passes a launch: the kernels per colour and per
line class (with and without LDS tiles) and the bands of lines, among them those above the
4096 sites that the bit-packed path takes; batches and graphs of every length around eight
passes, sample periods that fall inside them, chains put out of the run, an odd-edged chain
beside.  Equal to runs of one pass each, and to the per-colour kernels, in every value."""
import numpy as np
import pytest

import casmcode_monte_amd as M

pytestmark = pytest.mark.gpu


def _run(shapes, J2, passes, period, active, one_by_one=False, **schedule):
    chains = [dict(shape=s, temperature=1500.0 + 700.0 * i, exchange_potential=0.03, seed=40 + i)
              for i, s in enumerate(shapes)]
    lattice = M.LATTICE_SC if len(shapes[0]) == 3 else M.LATTICE_SQUARE
    with M.Run(chains, mode=M.MODE_CHECKERBOARD, lattice=lattice, J1=0.1, J2=J2,
               options=M.OPT_FORCE_STREAMING, sample_period=period) as r:
        r.set_schedule(**schedule)
        rng = np.random.default_rng(7)
        for c, s in enumerate(shapes):
            r.set_occupation(c, np.where(rng.random(int(np.prod(s))) < 0.5, 1, -1).astype(np.int8))
        if active is not None:
            r.set_active(active)
        for p in passes:
            for k in ([1] * p if one_by_one else [p]):
                r.run(k)
        return [(r.samples(c), r.get_occupation(c), r.counters(c)) for c in range(len(chains))]


def _same(a, b, tag):
    for (sa, oa, ca), (sb, ob, cb) in zip(a, b):
        assert np.array_equal(sa, sb) and np.array_equal(oa, ob) and ca == cb, tag


@pytest.mark.parametrize("J2", [0.0, -0.02])
@pytest.mark.parametrize("shapes,period,active", [
    ([(50, 8), (30, 6)], 1, None), ([(48, 8), (80, 6)], 3, None), ([(50, 8)], 7, None),
    ([(50, 8), (96, 6), (34, 4)], 2, [1, 0, 1]), ([(50, 8), (7, 9)], 3, None),
    ([(4128, 6), (8192, 4)], 2, None), ([(20, 6, 4), (16, 4, 6)], 3, None)])
def test_records(shapes, period, active, J2):
    passes = [1, 7, 8, 9, 25, 2]
    print("records of the byte paths", shapes, period, J2, flush=True)
    want = _run(shapes, J2, passes, period, active, one_by_one=True, band_lines=0,
                graph_passes=1)
    for schedule in (dict(band_lines=0, units_per_thread=1), dict(band_lines=0, line_tiles=1),
                     dict(band_lines=-1), dict(band_lines=2)):
        for graph in (1, 3, 8, 20):
            got = _run(shapes, J2, passes, period, active, graph_passes=graph, **schedule)
            _same(want, got, (schedule, graph))


@pytest.mark.parametrize("J2", [0.0, -0.02])
@pytest.mark.parametrize("shapes", [[(4128, 6)], [(8192, 4), (4112, 10)], [(6400, 64)],
                                    [(8192, 2)]])
def test_bands_of_long_lines(shapes, J2):
    """Lines of more than 4096 sites: the bands on bytes are the path that takes them."""
    print("bands of long lines", shapes, J2, flush=True)
    want = _run(shapes, J2, [3, 9], 1, None, band_lines=0, graph_passes=1)
    for band in (-1, 2, 4, 64):
        for graph in (1, 8):
            got = _run(shapes, J2, [3, 9], 1, None, band_lines=band, graph_passes=graph)
            _same(want, got, (band, graph))
