"""The walk's fast form against the general form, piece by piece, on the CPU
(the same header compiled for the host)."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from gsmfretda_amd import synth

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def host(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("host") / "libfastform.so")
    csrc = os.path.join(ROOT, "gsmfretda_amd", "csrc")
    subprocess.run(["hipcc", "-x", "hip", "--offload-host-only", "-O2", "-fPIC", "-std=c++17",
                    "-ffp-contract=off", "-fno-fast-math", "-shared", "-I", csrc, "-I",
                    os.path.join(ROOT, "include"),
                    os.path.join(ROOT, "tests", "host", "host_fast_form.cpp"),
                    os.path.join(csrc, "pda_layout.cpp"), "-o", so], check=True,
                   capture_output=True)
    return ctypes.CDLL(so)


def _out(n):
    return (ctypes.c_int64 * n)()


def test_log_of_every_uniform(host):
    out = _out(2)
    host.hf_log(out)
    assert list(out) == [1 << 24, 0]


def test_quotient_exp_normal_and_efficiency(host):
    """Equal bit for bit: correctly rounded quotients over the divisors'
    range, exp over [0, 64], normals, efficiencies at every distance (zero,
    tiny, infinite and NaN ones too)."""
    out = _out(8)
    host.hf_math(ctypes.c_int64(3_000_000), ctypes.c_uint64(11), out)
    assert list(out)[0::2] == [3_000_000] * 4
    assert list(out)[1::2] == [0, 0, 0, 0]


def test_broad_binomial(host):
    """Every count it gives equals the inversion's; uniforms within its band
    of a threshold are left to the general form, others practically never."""
    out = _out(5)
    host.hf_binomial(60, 200, ctypes.c_uint64(3), out)
    compared, different, left, at, decided = list(out)
    assert compared == 60 * 127 * 200 and different == 0
    # 2^-38 on each side of at most 128 thresholds (and of 1, where they crowd)
    assert left <= 2 + compared * 128 * 2.0 ** -37
    assert at > 100_000
    assert decided == 0


@pytest.mark.parametrize("n,v,bg,r0", [(2, 4.0, (1000.0, 500.0), 52.0), (3, 6.0, (0.0, 0.0), 52.0),
                                       (5, 2.5, (8000.0, 9000.0), 30.5),
                                       (8, 5.0, (1000.0, 500.0), 1e-15)])
def test_broadened_units(host, n, v, bg, r0):
    rng = np.random.default_rng(n)
    args = synth.make_args(np.sort(rng.uniform(0.0, 1.0, n)),
                           synth.loguniform_rates(rng, n * (n - 1), 1e2, 1e4),
                           v * rng.integers(0, 2, n) if n > 2 else [v, v])
    d = synth.generate(300, args, n, base_photons=20, mean_geom=60.0, seed=n)
    out = _out(4)
    keep = [np.ascontiguousarray(x, t) for x, t in (
        (d.start, np.int64), (d.stop, np.int64), (d.istart, np.int64), (d.phcount, np.int32),
        (d.times, np.int64), (d.mask_ad, np.uint8), (d.mask_dd, np.uint8), (d.T, np.float32),
        (args, np.float32))]
    k = [x.ctypes.data_as(ctypes.c_void_p) for x in keep]
    f = ctypes.c_float
    rc = host.hf_walk(k[0], k[1], k[2], k[3], ctypes.c_int64(d.nbursts), k[4], k[5], k[6],
                      ctypes.c_int64(d.nphotons), k[7], f(d.clk_p), f(bg[1]), f(bg[0]), n, k[8],
                      f(r0), 12, ctypes.c_uint32(9), out)
    assert rc == 0
    units, abandoned, different, acceptors = list(out)
    assert units == 300 * 12 and different == 0 and acceptors > 0
    assert abandoned < units // 20
