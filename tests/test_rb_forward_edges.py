"""GPU: the RB adjoint where no unit has an acceptor outcome past 0, with a
cotangent beyond float's range, and the RB forward on a stream that is being
recorded."""
import ctypes

import numpy as np
import pytest

from gsmfretda_amd import pda, synth

pytestmark = pytest.mark.gpu


def _load(m, ph, seed, **kw):
    rng = np.random.default_rng(seed)
    args = synth.make_args([0.3, 0.7], synth.loguniform_rates(rng, 2, 3e2, 8e3))
    d = synth.generate(300, args, 2, seed=seed, **kw)
    m.load(d, SgDivSr=rng.uniform(0, 1, d.nbursts).astype(np.float32), nbins=50, left_pad=0)
    m.set_photophysics(0, *ph)
    m.set_burst_range(0, -1, 0)
    assert m.set_params(2, 0, args)


def test_adjoint_of_a_cotangent_beyond_float(gpu_mc):
    """Corrected counts too small for a binomial trial: every unit has the
    outcome 0 alone, so no difference of two bins' cotangents is taken and the
    efficiencies have the gradient 0, however large the cotangent (the rates'
    terms are h (S - Sbar) in double)."""
    m = gpu_mc
    _load(m, (0.01, 0.99, 0.0, 52.0), 3, base_photons=8, mean_geom=4.0)
    m.rb_forward(R=5, seed=2, set_id=1)
    M = m.rb_result()[0]
    assert M[0] == 300 * 5 and not M[1:].any()
    one = m.rb_adjoint(np.ones(50), 2)
    grad = m.rb_adjoint(np.full(50, 1e39), 2)
    m.set_photophysics(0, *synth.PHOTOPHYSICS)
    assert np.array_equal(one[:2], [0.0, 0.0]) and np.array_equal(grad[:2], [0.0, 0.0])
    assert np.isfinite(grad).all()


def test_forward_on_a_recording_stream(gpu_mc):
    """Refused, as the other RB calls are: a replay would pair the recorded
    set's tables with whatever model the slot holds by then."""
    m = gpu_mc
    _load(m, synth.PHOTOPHYSICS, 5)
    m.rb_forward(R=6, seed=2, set_id=1)
    want = m.rb_result()
    hip = ctypes.CDLL("libamdhip64.so.7")
    stream, graph = ctypes.c_void_p(m.getStreams()[0]), ctypes.c_void_p()
    assert hip.hipStreamBeginCapture(stream, 1) == 0
    try:
        with pytest.raises(pda.PdaError):
            m.rb_forward(R=6, seed=2, set_id=1)
    finally:
        hip.hipStreamEndCapture(stream, ctypes.byref(graph))
        if graph:
            hip.hipGraphDestroy(graph)
    m.rb_forward(R=6, seed=2, set_id=1)
    got = m.rb_result()
    assert np.array_equal(got[1], want[1]) and got[2] == want[2]
