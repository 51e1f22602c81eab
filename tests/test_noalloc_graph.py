"""GPU: pda_run_noalloc recorded into a graph and replayed after the slot's
parameters and photophysics changed: a replay walks the model that the device
then holds, as a run made after the change does -- another Foerster radius
(the reciprocal of the old one does not go with it), more states than the
recorded set had, rates outside the quick quotient's range."""
import ctypes

import numpy as np
import pytest

from gsmfretda_amd import synth
from tests.test_zz_no_alloc import HDR, DeviceBuffer

pytestmark = pytest.mark.gpu

B, R, SEED, SET = 50, 30, 71, 4


class Graph:
    """What `record` enqueues on a slot's stream, to be launched again."""

    def __init__(self, m, hip, record):
        self.m, self.hip = m, hip
        self.stream = ctypes.c_void_p(m.getStreams()[0])
        graph, self.exec = ctypes.c_void_p(), ctypes.c_void_p()
        assert hip.hipStreamBeginCapture(self.stream, 1) == 0  # thread-local
        try:
            record()
        finally:
            rc = hip.hipStreamEndCapture(self.stream, ctypes.byref(graph))
        assert rc == 0
        assert hip.hipGraphInstantiate(ctypes.byref(self.exec), graph, None, None, 0) == 0
        assert hip.hipGraphDestroy(graph) == 0

    def launch(self):
        assert self.hip.hipGraphLaunch(self.exec, self.stream) == 0
        self.m.synchronize(0)

    def free(self):
        assert self.hip.hipGraphExecDestroy(self.exec) == 0


def _args(rng, n, v, rates=(3e2, 8e3)):
    return synth.make_args(np.sort(rng.uniform(0.1, 0.9, n)),
                           synth.loguniform_rates(rng, n * (n - 1), *rates), np.full(n, v))


def _slow(args, n):
    """The same with the rates out of the last state zero and one tiny."""
    a = np.array(args, np.float32)
    k = a[n:n * n].reshape(n, n - 1)  # row j: rates into j
    k[:-1, -1] = 0.0
    k[-1, 0] = 1e-14
    return a


@pytest.mark.parametrize("v", [0.0, 4.0])
def test_replay_follows_the_model(gpu_mc, v):
    m = gpu_mc
    rng = np.random.default_rng(int(v) + 1)
    first = _args(rng, 2, v)
    d = synth.generate(1500, first, 2, seed=3)
    m.load(d, SgDivSr=rng.uniform(0, 1, d.nbursts).astype(np.float32), nbins=B, left_pad=2)
    ph = synth.PHOTOPHYSICS
    m.set_photophysics(0, *ph)
    assert m.set_params(2, 0, first)
    m.set_burst_range(0, -1, 0)
    buf = DeviceBuffer(HDR.itemsize + 4 * B)
    m.run_noalloc(buf.ptr.value, buf.nbytes, R=R, seed=SEED, set_id=SET, sid=0)
    m.synchronize(0)
    graph = Graph(m, buf.hip, lambda: m.run_noalloc(buf.ptr.value, buf.nbytes, R=R, seed=SEED,
                                                    set_id=SET, sid=0))
    five = _args(rng, 5, v)
    changes = [(2, first, ph[3]), (2, first, 70.0), (5, five, 70.0), (5, five, 1e-15),
               (3, _slow(_args(rng, 3, v), 3), 52.0), (2, first, ph[3])]
    try:
        for n, args, r0 in changes:
            m.set_photophysics(0, *ph[:3], r0)
            assert m.set_params(n, 0, args)
            buf.write(np.full(buf.nbytes, 0xAB, np.uint8))
            graph.launch()
            got = buf.read()[HDR.itemsize:].view(np.int32)
            m.reSampleTimes = R
            m.run_kernel(sid=0, seed=SEED, set_id=SET)
            m.synchronize(0)
            assert np.array_equal(got, m.get_hist_chi2(0)[0]), (n, r0)
    finally:
        graph.free()
        buf.free()
        m.set_photophysics(0, *ph)
