"""GPU: the mean scores of bursts whose scores are up to, just above and far above
what is staged at a time, by the rate gradients they enter."""
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


@pytest.mark.parametrize("n,R", [(3, 682), (3, 683), (3, 1365), (3, 4000), (4, 342), (4, 1000),
                                 (2, 2048), (2, 5000)])
def test_score_means(gpu_mc, oracle, n, R):
    """Against the oracle's FP64 gradient, with the tolerance of the other
    gradient tests: 1e-3 of a component, or of a hundredth of the largest
    rate's."""
    m = gpu_mc
    d, args, rng = _setup(m, n, 5, 50, n + R)
    m.rb_forward(R=R, seed=4, set_id=2)
    m.rb_result()
    g = rng.integers(-4, 5, size=50).astype(np.float64)
    got = m.rb_adjoint(g, n)[n:n * n]
    od = oracle.Data.from_bursts(d)
    p = oracle.make_params(n, np.asarray(args, np.float32), *synth.PHOTOPHYSICS)
    want = oracle.rb_grad(od, p, R, 4, g, set_id=2)[1][n:]
    scale = np.abs(want).max()
    assert scale > 0
    assert np.all(np.abs(got - want) <= 1e-3 * np.maximum(np.abs(want), 1e-2 * scale))
