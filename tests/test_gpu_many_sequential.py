"""Handles of one to so many sequential chains that the read-back of their states goes through
the staging memory in parts: positions, records and counters of every chain follow runs that
differ from chain to chain."""
import numpy as np
import pytest

import casmcode_monte_amd as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("chains", [1, 24, 25, 390, 400, 2600, 5200])
@pytest.mark.parametrize("mode", ["kmc", "occupant", "nfold"])
def test_states_of_every_chain(mode, chains):
    print("many sequential", mode, chains, flush=True)
    ch = [dict(shape=(6, 5), temperature=1500.0, exchange_potential=0.02, seed=5 + c % 7)
          for c in range(chains)]
    extra = dict(mode=M.MODE_KMC, J1=0.05, sample_time_period=0.05)
    if mode == "occupant":
        extra = dict(mode=M.MODE_OCCUPANT, J1=0.1,
                     occupant=dict(asym_species=[[0, 1]], n_species=2, canonical=False,
                                   swaps=[(0, 1), (1, 0)],
                                   exchange_potential=[[0.0, 0.02]] * chains))
    elif mode == "nfold":
        extra = dict(mode=M.MODE_NFOLD, J1=0.1, sample_time_period=0.05)
    with M.Run(ch, **extra) as r:
        r.reserve_samples(2000)
        for c in range(chains):
            v = (np.random.default_rng(c % 7).random(30) < 0.4).astype(np.int8)
            v[c % 7] = 1 - v[(c + 1) % 7]
            v[:2] = [0, 1]
            r.set_occupation(c, 2 * v - 1 if mode == "nfold" else v)
        r.run(2)
        if mode == "nfold":
            r.kmc_advance(7)
        else:
            r.run_steps(7)
        out = []
        for c in range(chains):
            rec = r.samples(c)
            out.append((rec.tobytes(), r.counters(c), r.position(c), r.get_occupation(c).tobytes()))
            assert r.position(c)[1] == 7 and r.counters(c)[0] == 2
        for c in range(7, chains):  # seven different chains, over and over
            assert out[c] == out[c % 7], c
