"""GPU: the RB Jacobian with so many bins that few copies of its rows fit a
workgroup (its lanes' outcomes are then taken in different orders), over few
bursts of many resamples, whose units fall into the same bins."""
import numpy as np
import pytest

from gsmfretda_amd import synth

pytestmark = pytest.mark.gpu


def _setup(m, n, bursts, B, seed):
    rng = np.random.default_rng(seed)
    args = synth.make_args(np.sort(rng.uniform(0.1, 0.9, n)),
                           synth.loguniform_rates(rng, n * (n - 1), 3e2, 8e3))
    d = synth.generate(bursts, args, n, seed=seed)
    m.load(d, SgDivSr=rng.uniform(0, 1, bursts).astype(np.float32), nbins=B, left_pad=0)
    m.set_photophysics(0, *synth.PHOTOPHYSICS)
    m.set_burst_range(0, -1, 0)
    assert m.set_params(n, 0, args)
    return d, args, rng


@pytest.mark.parametrize("n,bursts,R,B", [(2, 3, 700, 1024), (2, 40, 9, 900), (3, 2, 1500, 700),
                                          (3, 70, 31, 1024), (4, 2, 1000, 200), (4, 65, 20, 1021),
                                          (4, 300, 3, 400)])
def test_jacobian(gpu_mc, n, bursts, R, B):
    m = gpu_mc
    _, _, rng = _setup(m, n, bursts, B, n * bursts)
    m.rb_forward(R=R, seed=9, set_id=1)
    M = m.rb_result()[0]
    J = m.rb_jacobian(n, B)
    # sums of the same terms in double, in other orders: within their count
    # (below 2^21) times 2^-53 of the terms' magnitudes, which the rows' sums
    # of magnitudes bound up to the cancellation inside a row
    for g in (rng.integers(-4, 5, size=B).astype(np.float64), np.eye(B)[0], np.eye(B)[B // 3]):
        adj = m.rb_adjoint(g, n)
        scale = np.abs(g) @ np.abs(J) + np.abs(J).max() * R
        assert np.all(np.abs(g @ J - adj) <= 1e-9 * scale), (g @ J, adj)
    assert M.sum() > 0
