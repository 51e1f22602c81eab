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
