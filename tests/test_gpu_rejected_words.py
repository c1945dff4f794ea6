"""Engine words that a Lemire draw rejects, in the walks that take them on a path of
their own (KMC, OCCUPANT pairs and its general kernel, CANONICAL, N-fold): engines loaded
with zero words at the start of a window, inside it, in runs, and across the ends of
generations.  A zero word is below every rejection threshold as a draw (redrawn unless the
count is a power of two) and accepts as an acceptance word.  Bit-exact against the oracle,
by the walks and step by step (OPT_EXACT_SCALAR_WALK)."""
import numpy as np
import pytest

import casmcode_monte_amd as M
import oracle as O

pytestmark = pytest.mark.gpu

OPTIONS = (0, M.OPT_EXACT_SCALAR_WALK)


def _engine(seed, plant):
    """The seed's state at output 5 of a generation, zero at some words."""
    w = O.mt64_state(seed, 0).copy()
    w[312] = 5
    for at in plant:
        w[at] = 0
    assert np.count_nonzero(w[:312]) > 150
    return w


PLANTS = {
    "first": [[5], [6], [7], [8]],
    "inside": [[5 + 29, 5 + 30], [5 + 47], [5 + 62], [5 + 63, 5 + 64]],
    "run": [list(range(100, 140)) + list(range(0, 312, 7))],
    "ends": [list(range(303, 312)), [309], [310], [311], [311, 0, 1, 156, 157]],
}


@pytest.mark.parametrize("where", PLANTS)
@pytest.mark.parametrize("rows,cols,atoms,T,period", [
    (12, 13, 20, 900.0, 0.0), (5, 7, 16, 600.0, 0.0), (41, 53, 1000, 400.0, 0.01),
    (3, 3, 3, 2000.0, 0.2)])
def test_kmc(rows, cols, atoms, T, period, where):
    n = rows * cols
    occ = np.zeros(n, np.int8)
    occ[np.random.default_rng(n + atoms).permutation(n)[:atoms]] = 1
    for i, plant in enumerate(PLANTS[where]):
        eng = _engine(71 + i, plant)
        for options in OPTIONS:
            print("kmc", rows, cols, atoms, where, i, options, flush=True)
            with M.Run([dict(shape=(rows, cols), temperature=T, seed=1)], mode=M.MODE_KMC, J1=0.05,
                       sample_time_period=period, options=options) as r:
                r.set_occupation(0, occ)
                r.rng_load(0, eng)
                r.reserve_samples(1 << 14)
                total = 0
                for steps in (1, 30, 400):
                    r.run_steps(steps)
                    total += steps
                    o = O.kmc_run(rows, cols, 0.05, T, total, occ, eng, time_period=period)
                    s = r.samples(0)
                    assert len(s) == o["n_records"]
                    for f, k in (("time", "time"), ("S1", "S"), ("S2", "sum_sq"), ("S3", "sum_dx"),
                                 ("T3", "sum_dy")):
                        assert np.array_equal(np.asarray(s[f]).view(np.uint64),
                                              np.asarray(o[k]).view(np.uint64)), (f, steps)
                    assert np.array_equal(r.get_occupation(0), o["occ"])
                    assert np.array_equal(r.occ_location(0), o["loc"])
                    assert np.array_equal(r.atoms(0, atoms), o["atoms"])
                    assert np.array_equal(r.rng_dump(0), o["engine"])
                    assert sum(r.counters(0)[1:]) == o["attempts"]


SPECS = {1: [[0, 1]], 2: [[0, 1], [1], [1, 0]], 3: [[0, 1], [1, 0], [0], [0, 1]]}


@pytest.mark.parametrize("where", PLANTS)
@pytest.mark.parametrize("canonical", [False, True])
@pytest.mark.parametrize("units,rows,cols,T", [(1, 12, 11, 2000.0), (2, 17, 29, 900.0),
                                               (3, 24, 20, 3000.0), (1, 3, 3, 1e5)])
def test_occupant(units, rows, cols, T, canonical, where):
    spec = SPECS[units]
    n = rows * cols
    rng = np.random.default_rng(rows * cols)
    asym = rng.integers(0, len(spec), n).astype(np.int8)
    asym[:6] = [0, 0, len(spec) - 1, len(spec) - 1, 0, 0]
    occ = np.array([rng.integers(0, len(spec[b])) for b in asym], np.int8)
    occ[:6] = [0, 1, 0, 1, 0, 1]
    # semi-grand: unit by unit (the pair kernel) and, with two units or more, interleaved
    # (the general kernel); canonical: all swaps (the general kernel)
    cands = O.occ_candidates(spec)
    pairs = []
    for b in range(len(spec)):
        if len(spec[b]) > 1:
            z, one = cands.index((b, spec[b][0])), cands.index((b, spec[b][1]))
            pairs.append([(z, one), (one, z)])
    if canonical:
        forms = [O.occ_canonical_swaps(spec)]
    else:
        forms = [[s for p in pairs for s in p]]
        if len(pairs) > 1:
            forms.append([p[0] for p in pairs] + [p[1] for p in pairs])
    mu = [0.0, 0.0] if canonical else [0.0, 0.03]
    for swaps in forms:
        for i, plant in enumerate(PLANTS[where]):
            eng = _engine(81 + i, plant)
            for options in OPTIONS:
                print("occupant", units, rows, cols, canonical, where, i, options, flush=True)
                with M.Run([dict(shape=(rows, cols), temperature=T, seed=1)],
                           mode=M.MODE_OCCUPANT, J1=0.1, sample_period=1, options=options,
                           occupant=dict(asym_species=spec, n_species=2, canonical=canonical,
                                         swaps=swaps,
                                         **({} if canonical else
                                            dict(exchange_potential=[mu])))) as r:
                    r.set_site_asym(0, asym)
                    r.set_occupation(0, occ)
                    r.rng_load(0, eng)
                    total = 0
                    for steps in (1, 29, 500):
                        r.run_steps(steps)
                        total += steps
                        o = O.occ_run(rows, cols, asym, spec, mu, swaps, canonical, 0.1, T, total,
                                      occ, eng)
                        s = r.samples(0)
                        assert np.array_equal(np.array(s["e_run"]).view(np.uint64),
                                              np.asarray(o["e_run"]).view(np.uint64))
                        assert np.array_equal(s["S1"], o["S"]) and np.array_equal(s["M"], o["M"])
                        assert np.array_equal(r.get_occupation(0), o["occ"])
                        assert np.array_equal(r.occ_location(0), o["loc_sites"])
                        assert np.array_equal(r.rng_dump(0), o["engine"])
                        assert tuple(r.counters(0)[1:]) == (o["n_accept"], o["n_reject"])


@pytest.mark.parametrize("where", PLANTS)
@pytest.mark.parametrize("rows,cols,up,T", [(12, 10, 37, 2000.0), (16, 16, 128, 1500.0),
                                            (1, 40, 7, 2500.0), (31, 67, 1000, 1e5)])
def test_canonical(rows, cols, up, T, where):
    n = rows * cols
    occ = -np.ones(n, np.int8)
    occ[np.random.default_rng(n + up).permutation(n)[:up]] = 1
    for i, plant in enumerate(PLANTS[where]):
        eng = _engine(91 + i, plant)
        for options in OPTIONS:
            print("canonical", rows, cols, up, where, i, options, flush=True)
            with M.Run([dict(shape=(rows, cols), temperature=T, seed=1)], mode=M.MODE_CANONICAL,
                       J1=0.1, sample_period=1, options=options) as r:
                r.set_occupation(0, occ)
                r.rng_load(0, eng)
                for passes in (1, 4):
                    r.run(passes if passes == 1 else passes - 1)
                    o = O.canonical_run(rows, cols, 0.1, T, passes, occ, eng, use_nlist=True)
                    s = r.samples(0)
                    assert np.array_equal(s["e_run"].view(np.uint64),
                                          np.asarray(o["e_run"]).view(np.uint64))
                    assert np.array_equal(s["S1"], o["S"])
                    assert np.array_equal(r.get_occupation(0), o["occ"])
                    assert np.array_equal(r.occ_location(0), o["loc"])
                    assert np.array_equal(r.rng_dump(0), o["engine"])
                    assert r.counters(0)[1:] == (o["n_accept"], o["n_reject"])


@pytest.mark.parametrize("where", PLANTS)
@pytest.mark.parametrize("rows,cols,T", [(7, 9, 1500.0), (16, 16, 900.0), (2, 9, 2500.0),
                                         (33, 31, 2000.0)])
def test_nfold(rows, cols, T, where):
    n = rows * cols
    occ = np.where(np.random.default_rng(n).random(n) < 0.5, 1, -1).astype(np.int8)
    for i, plant in enumerate(PLANTS[where]):
        eng = _engine(61 + i, plant)
        print("nfold", rows, cols, where, i, flush=True)
        with M.Run([dict(shape=(rows, cols), temperature=T, exchange_potential=0.02, seed=1)],
                   mode=M.MODE_NFOLD, J1=0.1, sample_period=1) as r:
            r.set_occupation(0, occ)
            r.rng_load(0, eng)
            for passes in (1, 5):
                r.run(passes if passes == 1 else passes - 1)
                o = O.nfold_run(rows, cols, 0.1, T, 0.02, passes, occ, eng, sample_period=1)
                s = r.samples(0)
                np.testing.assert_array_equal(s["S1"], o["S"])
                np.testing.assert_array_equal(s["M"], o["M"])
                np.testing.assert_allclose(s["time"], o["time"], rtol=1e-12)
                np.testing.assert_allclose(s["weight"], o["weight"], rtol=1e-12)
                np.testing.assert_array_equal(r.get_occupation(0), o["occ"])
                np.testing.assert_array_equal(r.occ_location(0), o["arr"])
                np.testing.assert_array_equal(r.rng_dump(0), o["engine"])
