"""CPU: the rule by which models with distance broadening make the draws beyond
the fast form's in place, and those draws, compiled for the host."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from gsmfretda_amd import synth

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("host") / "liblongruns.so")
    csrc = os.path.join(ROOT, "gsmfretda_amd", "csrc")
    subprocess.run(["hipcc", "-x", "hip", "--offload-host-only", "-O2", "-fPIC", "-std=c++17",
                    "-ffp-contract=off", "-fno-fast-math", "-shared", "-I", csrc, "-I",
                    os.path.join(ROOT, "include"),
                    os.path.join(ROOT, "tests", "host", "host_long_runs.cpp"),
                    os.path.join(csrc, "pda_layout.cpp"), "-o", so], check=True,
                   capture_output=True)
    return ctypes.CDLL(so)


def _run(host, d, k=128, range_=None, ph=(1.0, 0.0, 0.0), n=2, args=None, R=0):
    out = (ctypes.c_int64 * 9)()
    keep = [np.ascontiguousarray(x, t) for x, t in (
        (d.start, np.int64), (d.stop, np.int64), (d.istart, np.int64), (d.phcount, np.int32),
        (d.times, np.int64), (d.mask_ad, np.uint8), (d.mask_dd, np.uint8), (d.T, np.float32),
        (synth.make_args([0.3, 0.7], [300.0, 500.0], [3.0, 3.0]) if args is None else args,
         np.float32))]
    p = [x.ctypes.data_as(ctypes.c_void_p) for x in keep]
    f = ctypes.c_float
    rc = host.hl_run(p[0], p[1], p[2], p[3], ctypes.c_int64(d.nbursts), p[4], p[5], p[6],
                     ctypes.c_int64(d.nphotons), p[7], f(d.clk_p), f(d.bg_ad), f(d.bg_dd),
                     f(ph[0]), f(ph[1]), f(ph[2]), ctypes.c_uint32(k),
                     ctypes.c_int64(d.nbursts if range_ is None else range_), n, p[8], R,
                     ctypes.c_uint32(9), out)
    assert rc == 0
    return list(out)


def _bursts(E, n_bursts=200, seed=1, **kw):
    return synth.generate(n_bursts, synth.make_args([E, E], [120.0, 250.0]), 2, seed=seed, **kw)


@pytest.mark.parametrize("neither", [0.0, 0.2])
def test_runs_counted(host, neither):
    """Every 16th photon with k of its run to come, against a scan; a photon in
    both channels ends the run before it."""
    d = _bursts(0.9, mean_geom=200.0, p_neither=neither, bg_dd=3e4, bg_ad=1e4)
    rng = np.random.default_rng(2)
    both = rng.random(d.nphotons) < 0.01
    d.mask_ad, d.mask_dd = d.mask_ad | both, d.mask_dd | both
    for k in (1, 2, 7, 40):
        want = [0, 0]
        for i0, P in zip(d.istart, d.phcount):
            colour = d.mask_dd[i0:i0 + P] + 2 * d.mask_ad[i0:i0 + P].astype(int)
            for i in range(0, P, 16):  # from the first channel photon at or after i
                f = next((j for j in range(i, P) if colour[j]), P)
                if f < P and colour[f] < 3:
                    end = next((j for j in range(f, P) if colour[j] & (3 - colour[f])), P)
                    want[colour[f] - 1] += end - f >= k
        assert _run(host, d, k)[:2] == want
    dur = np.maximum(d.T, np.float32(d.clk_p) * (d.stop - d.start).astype(np.float32))
    assert _run(host, d)[2] == int((dur * np.float32(3e4) > 64).sum())


@pytest.mark.parametrize("E,geom,ph,bg,single,pop", [
    (0.5, 40.0, (1.0, 0.0, 0.0), 1e3, 0, 0),
    (0.95, 40.0, (1.0, 0.0, 0.0), 1e3, 0, 0),       # a run of 128 in 0.1 % of the places
    (0.99, 300.0, (1.0, 0.0, 0.0), 1e3, 1, 1),
    (0.99, 300.0, (1.0, 0.0, 1.0), 1e3, 0, 0),      # acceptors count nothing
    (0.99, 300.0, (1.0, 0.0, 0.9), 1e3, 0, 0),      # 1,275 acceptors to a count of 128
    (0.01, 300.0, (1.0, 1.0, 0.0), 1e3, 0, 0),
    (0.01, 300.0, (6.0, 0.0, 0.0), 1e3, 1, 1),
    (0.8, 300.0, (1.0, 0.0, -9.0), 1e3, 1, 1),      # ten to an acceptor: runs of 13
    (0.5, 40.0, (1.0, 0.0, 0.0), 6e4, 1, 1),
    (0.5, 40.0, (1.0, 0.0, 0.0), 0.0, 0, 0),
])
def test_rule(host, E, geom, ph, bg, single, pop):
    d = _bursts(E, n_bursts=2000, mean_geom=geom, bg_dd=bg, bg_ad=bg / 2)
    assert _run(host, d, ph=ph)[3:5] == [single, pop]


def test_rule_of_a_part(host):
    """A part of the bursts may hold all of the long runs."""
    d = _bursts(0.5, n_bursts=2000)
    assert _run(host, d)[3:5] == [0, 0]
    few = _bursts(0.99, n_bursts=2000, mean_geom=300.0)
    dim = _bursts(0.5, n_bursts=2000, mean_geom=300.0)
    bright = np.repeat(np.arange(2000) < 20, few.phcount)
    few.mask_ad = np.where(bright, few.mask_ad, dim.mask_ad[np.arange(few.nphotons) % dim.nphotons])
    few.mask_dd = 1 - few.mask_ad
    assert _run(host, few)[3:5] == [0, 0]
    assert _run(host, few, range_=20)[3:5] == [1, 1]


@pytest.mark.parametrize("E,Em,bg,ph", [(0.99, (0.97, 1.0), 0.0, (1.0, 0.05, 0.0)),
                                        (0.01, (0.0, 0.03), 1e3, (1.0, 0.05, 0.0)),
                                        (0.99, (0.2, 0.8), 1e3, (1.0, 0.05, 0.0)),
                                        (0.5, (0.1, 0.9), 2e5, (1.0, 0.05, 0.0)),
                                        (0.5, (0.1, 0.9), 5e5, (4.0, 0.0, 0.1))])
@pytest.mark.parametrize("n", [2, 5])
def test_draws_in_place(host, E, Em, bg, ph, n):
    rng = np.random.default_rng(n)
    args = synth.make_args(np.sort(rng.uniform(*Em, n)),
                           synth.loguniform_rates(rng, n * (n - 1), 1e2, 3e3), np.full(n, 3.0))
    d = _bursts(E, n_bursts=150, mean_geom=300.0, bg_dd=bg, bg_ad=bg / 2)
    units, left, different, acceptors = _run(host, d, ph=ph, n=n, args=args, R=10)[5:]
    assert units == 1500 and different == 0 and acceptors > 0
    # uniforms within 2^-38 of one of at most 128 thresholds
    assert left <= 2
