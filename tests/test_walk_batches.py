"""GPU: the walk kernels start units 64 at a time and bin ended ones 64 at a
time; runs of less than that, of that and a unit more, units that end where
they start, and populations whose batches hold a few units each, so that a
wave goes through many sets."""
import numpy as np
import pytest

from gsmfretda_amd import pda, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bursts,R,B,nsets,v", [
    (1, 1, 50, 3, 0.0),
    (63, 1, 7, 5, 0.0),
    (13, 5, 200, 300, 0.0),
    (64, 2, 1, 9, 4.0),
    (129, 7, 50, 40, 0.0),
    (43, 3, 1024, 70, 4.0),
])
def test_walk_batches(gpu_mc, oracle, bursts, R, B, nsets, v):
    rng = np.random.default_rng(bursts + nsets)
    # some rates so slow that most units end in their first window
    sets = []
    for i in range(nsets):
        n = int(rng.integers(2, 5))
        a = synth.make_args(np.sort(rng.uniform(0.1, 0.9, n)),
                            synth.loguniform_rates(rng, n * (n - 1), *((1.0, 9.0), (3e2, 8e3))[i % 2]))
        a = np.array(a, np.float32)
        a[n * n:] = v * (i % 3 == 0)
        sets.append((n, a))
    d = synth.generate(bursts, sets[1][1], sets[1][0], seed=bursts)
    m = gpu_mc
    m.load(d, SgDivSr=rng.uniform(0, 1, bursts).astype(np.float32), nbins=B, left_pad=0)
    m.set_photophysics(0, *synth.PHOTOPHYSICS)
    m.set_burst_range(0, -1, 0)
    m.set_population([n for n, _ in sets], [a for _, a in sets])
    m.run_population(R=R, seed=31, set_base=2, set_stride=5)
    hist, _, _, _ = m.get_population_result()
    od = oracle.Data.from_bursts(d)
    for i, (n, a) in enumerate(sets):
        p = oracle.make_params(n, a, *synth.PHOTOPHYSICS)
        want = oracle.run(od, p, R=R, seed=31, set_id=2 + 5 * i, B=B, want_units=False)["hist"]
        assert np.array_equal(hist[i].astype(np.int64), want), f"set {i}"
        if i < 4:
            h1, _, _, _ = pda.evaluate(m, n, a, R, 31, set_id=2 + 5 * i)
            assert np.array_equal(h1.astype(np.int64), want), f"set {i} alone"


@pytest.mark.parametrize("B,left_pad", [(1, 0), (63, 2), (64, 64), (65, 0), (129, 63), (1024, 5)])
@pytest.mark.parametrize("bg", [0.0, 6e4])
def test_run_end(gpu_mc, oracle, B, left_pad, bg):
    """The end of a run by one wave, 64 bins at a time, with units replayed
    (a background whose mean leaves the fast form) and without, twice: the
    last workgroup leaves the rows and the counters zero."""
    n, R, seed = 3, 6, 77
    rng = np.random.default_rng(B)
    args = synth.make_args([0.2, 0.5, 0.8], synth.loguniform_rates(rng, 6, 3e2, 8e3))
    d = synth.generate(300, args, n, seed=B + 1)
    if bg:
        d.bg_dd, d.bg_ad = bg, bg
    obs = rng.uniform(0, 1, 300).astype(np.float32)
    m = gpu_mc
    m.load(d, SgDivSr=obs, nbins=B, left_pad=left_pad)
    m.set_photophysics(0, *synth.PHOTOPHYSICS)
    m.set_burst_range(0, -1, 0)
    od = oracle.Data.from_bursts(d)
    p = oracle.make_params(n, args, *synth.PHOTOPHYSICS)
    want = oracle.run(od, p, R=R, seed=seed, set_id=3, B=B, want_units=False)["hist"]
    c32, c64, eff = oracle.chi2(oracle.hist(obs, B).astype(np.float32), want, R, n,
                                left_pad=left_pad)
    m.set_population([n, n], [args, args])
    for _ in range(2):
        h, g64, g32, geff = pda.evaluate(m, n, args, R, seed, set_id=3)
        assert np.array_equal(h.astype(np.int64), want)
        # the oracle's sums, operation for operation
        assert geff == eff and np.array_equal([g32, g64], [c32, c64], equal_nan=True)
        assert (m.run_stats(0)[1] > 0) == (bg > 0)
        m.run_population(R=R, seed=seed, set_base=3, set_stride=0)
        h, g64, g32, geff = m.get_population_result()
        for i in range(2):
            assert np.array_equal(h[i].astype(np.int64), want)
            assert geff[i] == eff
            assert np.array_equal([g32[i], g64[i]], [c32, c64], equal_nan=True)


@pytest.mark.parametrize("bursts,R", [(1, 3), (31, 70), (33, 2), (1000, 5)])
@pytest.mark.parametrize("spread", ["usual", "equal", "zeros", "one long"])
def test_bursts_started_by_duration(gpu_mc, oracle, bursts, R, spread):
    """A run over all bursts starts them by duration, one over a part of them
    as they come: the same units, at the same places, whatever the durations
    (all the same, none for some, one far longer than the rest)."""
    n, seed = 3, 5
    rng = np.random.default_rng(bursts)
    args = synth.make_args([0.2, 0.5, 0.8], synth.loguniform_rates(rng, 6, 3e2, 8e3))
    d = synth.generate(bursts, args, n, seed=bursts + 7)
    d.T = np.array(d.T, np.float32)
    if spread == "equal":
        d.T[:] = d.T[0]
    elif spread == "zeros":
        d.T[::3] = 0.0
        d.T[1::7] = -1.0
    elif spread == "one long":
        d.T[bursts // 2] = 1.0
    m = gpu_mc
    m.load(d, SgDivSr=rng.uniform(0, 1, bursts).astype(np.float32), nbins=50, left_pad=0)
    m.set_photophysics(0, *synth.PHOTOPHYSICS)
    assert m.set_params(n, 0, args)
    m.reSampleTimes = R

    def units(b0, b1):
        k = m.set_burst_range(b0, b1, 0)
        m.run_kernel(sid=0, seed=seed, set_id=4, samples=True)
        m.synchronize(0)
        h = m.get_hist_chi2(0)[0]
        return (h, *m.get_samples(0, k * R))
    whole = units(0, -1)
    o = oracle.run(oracle.Data.from_bursts(d), oracle.make_params(n, args, *synth.PHOTOPHYSICS),
                   R=R, seed=seed, set_id=4, B=50)
    assert np.array_equal(whole[0].astype(np.int64), o["hist"])
    assert np.array_equal(whole[2], o["acc"])
    if bursts > 1:
        k = bursts // 2
        a, b = units(0, k), units(k, bursts)
        assert np.array_equal(whole[0], a[0] + b[0])
        for x, y, z in zip(whole[1:], a[1:], b[1:]):
            assert np.array_equal(np.asarray(x).view(np.uint32),
                                  np.concatenate([y, z]).view(np.uint32))
    m.set_burst_range(0, -1, 0)


def test_run_times(gpu_mc):
    """The runs' times from the kernels' clock readings: parts of the time the
    calls took, that of another run for another run."""
    import time
    n = 3
    rng = np.random.default_rng(3)
    args = synth.make_args([0.2, 0.5, 0.8], synth.loguniform_rates(rng, 6, 3e2, 8e3))
    d = synth.generate(2000, args, n, seed=8)
    m = gpu_mc
    m.load(d, SgDivSr=rng.uniform(0, 1, 2000).astype(np.float32), nbins=50, left_pad=2)
    m.set_photophysics(0, *synth.PHOTOPHYSICS)
    m.set_burst_range(0, -1, 0)
    ms = {}
    for R in (2, 2000):
        t0 = time.perf_counter()
        pda.evaluate(m, n, args, R, 9)
        wall = (time.perf_counter() - t0) * 1e3
        w, f = m.last_pass_ms(0)
        assert 0 < w < wall and 0 < f < wall
        assert abs(m.last_run_ms(0) - (w + f)) <= 1e-5 * wall
        ms[R] = w
    assert ms[2000] > ms[2]
    t0 = time.perf_counter()
    m.rb_forward(R=20, seed=1, set_id=0)
    m.rb_result()
    wall = (time.perf_counter() - t0) * 1e3
    w, f, a = m.rb_stats()
    assert 0 < w < f < wall and a == 0
    m.rb_adjoint(np.ones(50), n)
    assert m.rb_stats()[2] > 0
