"""GPU: a population whose abandoned units are more than its list holds is
walked a second time as a whole: the sets' results are those of single runs,
and the next run, which fits, starts from clean counters."""
import numpy as np
import pytest

from gsmfretda_amd import pda, synth

pytestmark = pytest.mark.gpu


def test_list_overflow(gpu_mc):
    m = gpu_mc
    rng = np.random.default_rng(3)
    n, R, nsets = 3, 40, 40
    sets = [synth.make_args(np.sort(rng.uniform(0.1, 0.9, n)),
                            synth.loguniform_rates(rng, 6, 1e2, 2e3)) for _ in range(nsets)]
    d = synth.generate(2000, sets[0], n, seed=9, bg_dd=1.5e5, bg_ad=7e4)
    m.load(d, SgDivSr=rng.uniform(0, 1, 2000).astype(np.float32), nbins=50, left_pad=2)
    m.set_photophysics(0, *synth.PHOTOPHYSICS)
    m.set_burst_range(0, -1, 0)
    for graph in (True, False):
        m.set_population([n] * nsets, sets)
        m.run_population(R=R, seed=8, set_base=1, graph=graph)
        hist, c64, _, _ = m.get_population_result()
        for i in (0, 17, nsets - 1):
            h, c, _, _ = pda.evaluate(m, n, sets[i], R, 8, set_id=1 + i)
            # three quarters of the units are abandoned: of all sets above 2^20
            assert m.run_stats(0)[1] * nsets > (1 << 20)
            assert np.array_equal(hist[i], h) and c64[i] == c
        m.set_population([n] * 3, sets[:3])
        m.run_population(R=R, seed=8, set_base=1, graph=graph)
        few = m.get_population_result()[0]
        assert m.population_stats()[1] > 0  # replayed, not repeated
        assert np.array_equal(few, hist[:3])
