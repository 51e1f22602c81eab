"""GPU: models with distance broadening over bursts whose windows need draws
beyond the fast form's -- counts of 128 and more, by inversion and by
rejection, and background means above 64 -- for single sets and populations:
the oracle's histograms, and next to no unit walked a second time."""
import numpy as np
import pytest

from gsmfretda_amd import pda, synth
from tests.test_noalloc_graph import Graph
from tests.test_zz_no_alloc import HDR, DeviceBuffer

pytestmark = pytest.mark.gpu

BRIGHT = dict(base_photons=50, mean_geom=300.0)
# (data, efficiencies of the truth, of the sets, background, photophysics)
CASES = [
    (BRIGHT, [0.985, 0.99], (0.98, 1.0), 0.0, synth.PHOTOPHYSICS),
    (BRIGHT, [0.01, 0.015], (0.0, 0.03), 1e3, synth.PHOTOPHYSICS),
    (BRIGHT, [0.985, 0.99], (0.2, 0.8), 1e3, (1.0, 0.0, 0.0, 52.0)),
    (dict(mean_geom=60.0), [0.3, 0.7], (0.1, 0.9), 1.2e5, synth.PHOTOPHYSICS),
    (dict(mean_geom=60.0, p_neither=0.1), [0.3, 0.7], (0.1, 0.9), 4e5, (4.0, 0.0, 0.0, 52.0)),
]


@pytest.mark.parametrize("data,truth,between,bg,ph", CASES)
def test_draws_beyond_the_fast_form(gpu_mc, oracle, data, truth, between, bg, ph):
    m = gpu_mc
    rng = np.random.default_rng(5)
    R, B, seed = 6, 50, 17
    d = synth.generate(500, synth.make_args(truth, [120.0, 250.0]), 2, seed=4, bg_dd=bg,
                       bg_ad=bg / 2, **data)
    m.load(d, SgDivSr=rng.uniform(0, 1, d.nbursts).astype(np.float32), nbins=B, left_pad=2)
    m.set_photophysics(0, *ph)
    sets = [(n, synth.make_args(np.sort(rng.uniform(*between, n)),
                                synth.loguniform_rates(rng, n * (n - 1), 1e2, 3e3),
                                np.full(n, 3.0))) for n in (2, 3, 2, 4)]
    od = oracle.Data.from_bursts(d)
    try:
        for b0, b1 in ((0, -1), (7, 300)):
            m.set_burst_range(b0, b1, 0)
            end = d.nbursts if b1 < 0 else b1
            units = (end - b0) * R
            want = [oracle.run(od, oracle.make_params(n, a, *ph), R=R, seed=seed, set_id=3 + i,
                               b0=b0, b1=end, B=B) for i, (n, a) in enumerate(sets)]
            for i, (n, a) in enumerate(sets):
                h = pda.evaluate(m, n, a, R, seed, set_id=3 + i, begin=b0, end=b1, samples=True)[0]
                assert np.array_equal(h.astype(np.int64), want[i]["hist"]), i
                assert np.array_equal(m.get_samples(0, units)[1], want[i]["acc"])
                assert m.run_stats(0)[1] <= units // 100
            m.set_population([n for n, _ in sets], [a for _, a in sets])
            m.run_population(R=R, seed=seed, set_base=3, set_stride=1)
            hist = m.get_population_result()[0]
            for i, w in enumerate(want):
                assert np.array_equal(hist[i].astype(np.int64), w["hist"]), i
            assert m.population_stats()[1] <= 4 * units // 100
    finally:
        m.set_photophysics(0, *synth.PHOTOPHYSICS)
        m.set_burst_range(0, -1, 0)


def test_recorded_without_allocation(gpu_mc):
    """The same draws in a run recorded into a graph, replayed."""
    m = gpu_mc
    rng = np.random.default_rng(8)
    d = synth.generate(700, synth.make_args([0.985, 0.99], [120.0, 250.0]), 2, seed=6, **BRIGHT)
    m.load(d, SgDivSr=rng.uniform(0, 1, d.nbursts).astype(np.float32), nbins=50, left_pad=2)
    m.set_photophysics(0, *synth.PHOTOPHYSICS)
    m.set_burst_range(0, -1, 0)
    sets = [synth.make_args(np.sort(rng.uniform(lo, hi, 3)),
                            synth.loguniform_rates(rng, 6, 1e2, 3e3), np.full(3, 3.0))
            for lo, hi in ((0.97, 1.0), (0.3, 0.7))]
    assert m.set_params(3, 0, sets[0])
    buf = DeviceBuffer(HDR.itemsize + 4 * 50)
    graph = Graph(m, buf.hip, lambda: m.run_noalloc(buf.ptr.value, buf.nbytes, R=20, seed=5,
                                                    set_id=2, sid=0))
    try:
        for i in (0, 1, 0):
            assert m.set_params(3, 0, sets[i])
            graph.launch()
            got = buf.read()[HDR.itemsize:].view(np.int32)
            assert np.array_equal(got, pda.evaluate(m, 3, sets[i], 20, 5, set_id=2)[0])
            assert m.run_stats(0)[1] <= 140
    finally:
        graph.free()
        buf.free()
