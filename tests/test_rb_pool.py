"""GPU: the RB adjoint just below and at the number of units from which it keeps
the memo's first pmfs in LDS, against the Jacobian."""
import numpy as np
import pytest

from gsmfretda_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 3, 4])
@pytest.mark.parametrize("bursts,R", [(1023, 1024), (1024, 1024)])
def test_adjoint(gpu_mc, n, bursts, R):
    m, B = gpu_mc, 50
    rng = np.random.default_rng(n)
    args = synth.make_args(np.sort(rng.uniform(0.1, 0.9, n)),
                           synth.loguniform_rates(rng, n * (n - 1), 3e2, 8e3))
    d = synth.generate(bursts, args, n, seed=n)
    m.load(d, SgDivSr=rng.uniform(0, 1, bursts).astype(np.float32), nbins=B, left_pad=0)
    m.set_photophysics(0, *synth.PHOTOPHYSICS)
    m.set_burst_range(0, -1, 0)
    assert m.set_params(n, 0, args)
    m.rb_forward(R=R, seed=9, set_id=1)
    m.rb_result()
    J = m.rb_jacobian(n, B)
    g = rng.integers(-4, 5, size=B).astype(np.float64)  # differences exact in float
    adj = m.rb_adjoint(g, n)
    # the same terms in double in other orders, below 2^26 of them: their
    # number times 2^-53 of the magnitudes, which the rows' sums of magnitudes
    # bound up to the cancellation inside a row
    scale = np.abs(g) @ np.abs(J) + np.abs(J).max() * R
    assert np.all(np.abs(g @ J - adj) <= 1e-8 * scale), (g @ J, adj)
