"""GPU: the RB per-unit passes at the edges of their tiles -- runs of one unit,
of a tile and a unit, of no units for most workgroups -- with one bin and with
1,024, and with photophysics whose corrected counts are zero or tiny (the
passes' quick quotient does not take those)."""
import numpy as np
import pytest

from gsmfretda_amd import synth

pytestmark = pytest.mark.gpu

DEFAULT = synth.PHOTOPHYSICS


@pytest.mark.parametrize("n,bursts,R,B,ph", [
    (2, 1, 2, 7, DEFAULT),
    (3, 67, 3, 1024, DEFAULT),
    (4, 130, 5, 50, DEFAULT),
    (3, 2051, 2, 1, DEFAULT),
    (2, 700, 100, 300, DEFAULT),
    (3, 300, 4, 50, (0.05, 0.0, 0.05, 52.0)),
    (3, 300, 4, 50, (1e-13, 0.0, 0.0, 52.0)),
])
def test_rb_tiles(gpu_mc, oracle, n, bursts, R, B, ph):
    rng = np.random.default_rng(n * bursts)
    args = synth.make_args(np.sort(rng.uniform(0.1, 0.9, n)),
                           synth.loguniform_rates(rng, n * (n - 1), 3e2, 8e3))
    d = synth.generate(bursts, args, n, seed=bursts)
    gpu_mc.load(d, SgDivSr=rng.uniform(0, 1, bursts).astype(np.float32), nbins=B, left_pad=0)
    gpu_mc.set_photophysics(0, *ph)
    gpu_mc.set_burst_range(0, -1, 0)
    assert gpu_mc.set_params(n, 0, args)
    gpu_mc.rb_forward(R=R, seed=9, set_id=1)
    _, fixed, _, _ = gpu_mc.rb_result()
    od = oracle.Data.from_bursts(d)
    p = oracle.make_params(n, args, *ph)
    assert np.array_equal(fixed, oracle.rb_run(od, p, R, 9, 1, B=B))
    J = gpu_mc.rb_jacobian(n, B)
    g = rng.integers(-4, 5, size=B).astype(np.float64)  # differences exact in float
    adj = gpu_mc.rb_adjoint(g, n)
    # both are sums of the same terms in double, in other orders: each within
    # their count (below 2^21 here) times 2^-53 of the terms' magnitudes, which
    # the rows' sums of magnitudes bound up to the cancellation inside a row
    scale = np.abs(g) @ np.abs(J) + np.abs(J).max() * R
    assert np.all(np.abs(g @ J - adj) <= 1e-9 * scale), (g @ J, adj)
    gpu_mc.set_photophysics(0, *DEFAULT)


@pytest.mark.parametrize("nsets,bursts,R", [(1, 40, 5), (2, 7, 700), (3, 300, 3), (8, 33, 7)])
def test_rb_sets_beside_each_other(gpu_mc, nsets, bursts, R):
    """Sets of an RB population, on as many streams as there are sets or
    fewer, forward and Jacobian twice: each equal to its run alone (with an
    odd number of resamples, and with one whose scores of a burst exceed the
    mean kernel's stage)."""
    rng = np.random.default_rng(nsets)
    sets = [(n, synth.make_args(np.sort(rng.uniform(0.1, 0.9, n)),
                                synth.loguniform_rates(rng, n * (n - 1), 3e2, 8e3)))
            for n in rng.integers(2, 5, 1).repeat(nsets)]
    n = sets[0][0]
    d = synth.generate(bursts, sets[0][1], n, seed=bursts)
    m = gpu_mc
    m.load(d, SgDivSr=rng.uniform(0, 1, bursts).astype(np.float32), nbins=20, left_pad=1)
    m.set_photophysics(0, *DEFAULT)
    m.set_burst_range(0, -1, 0)
    m.set_population([k for k, _ in sets], [a for _, a in sets])
    for seed in (5, 6):
        m.rb_forward_population(R=R, seed=seed, set_base=1, set_stride=2)
        _, fixed, chi2, eff = m.rb_population_result()
        J = m.rb_jacobian_population(n, 20)
        for k, (_, a) in enumerate(sets):
            assert m.set_params(n, 0, a)
            m.rb_forward(R=R, seed=seed, set_id=1 + 2 * k)
            _, f1, c1, e1 = m.rb_result()
            assert np.array_equal(fixed[k], f1) and eff[k] == e1
            assert np.array_equal([chi2[k]], [c1], equal_nan=True)
            # the same terms in double, fewer than 2^20, in another order
            J1 = m.rb_jacobian(n, 20)
            assert np.all(np.abs(J[k] - J1) <= 1e-9 * (np.abs(J1).max() + R))
