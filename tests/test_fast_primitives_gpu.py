"""GPU: the fast form's elementary functions as the GPU computes them (hardware
reciprocals and fused steps where the host divides), against the general
form's: equal bit for bit, every 24-bit uniform for the logarithm."""
import numpy as np
import pytest

from tests.conftest import bits
from tests.test_gpu_parity import BINOM_DT

pytestmark = pytest.mark.gpu


def _same(got, want):
    both_nan = np.isnan(got) & np.isnan(want)
    bad = (bits(got) != bits(want)) & ~both_nan
    assert not bad.any(), (int(bad.sum()), got[bad][:4], want[bad][:4])


def test_log_of_every_uniform(gpu_mc):
    rng = np.random.default_rng(1)
    k = np.arange(1 << 24, dtype=np.uint32)
    x = (k << 8) | rng.integers(0, 256, 1 << 24, dtype=np.uint32)
    u = (k + 1).astype(np.float32) * np.float32(2.0 ** -24)
    _same(gpu_mc.debug_primitive(10, x, np.float32, len(x)),
          gpu_mc.debug_primitive(1, u, np.float32, len(u)))


def test_exp(gpu_mc):
    rng = np.random.default_rng(2)
    lam = np.concatenate([rng.uniform(0, 64, 1 << 20), 2.0 ** rng.uniform(-140, 6, 1 << 18),
                          [0.0, 64.0, 1e-45]]).astype(np.float32)
    _same(gpu_mc.debug_primitive(11, lam, np.float32, len(lam)),
          gpu_mc.debug_primitive(2, -lam, np.float32, len(lam)))


def test_quotient(gpu_mc):
    rng = np.random.default_rng(3)
    k = 1 << 21
    mant = rng.integers(0, 1 << 23, k, dtype=np.uint32)
    edge = rng.random(k) < 0.1  # next to a power of two, or next below one
    mant[edge] = (rng.integers(-3, 4, edge.sum()) % (1 << 23)).astype(np.uint32)
    b = np.ldexp((mant | 0x3F800000).view(np.float32), rng.integers(-40, 40, k)).astype(np.float32)
    # logs of uniforms, times, and dividends of any size
    a = np.where(rng.random(k) < 0.3, np.log(rng.uniform(2.0 ** -24, 1, k)),
                 np.ldexp(rng.uniform(0.5, 1, k), rng.integers(-24, 24, k))).astype(np.float32)
    b *= rng.choice(np.array([-1, 1], np.float32), k)
    got = gpu_mc.debug_primitive(12, np.stack([a, b], 1), np.float32, k)
    _same(got, a / b)


def test_normal(gpu_mc):
    rng = np.random.default_rng(4)
    w = rng.integers(0, 1 << 32, (1 << 21, 2), dtype=np.uint64).astype(np.uint32)
    w[:9, 1] = np.arange(9, dtype=np.uint32) * 0x1FFFFFFF
    w[9:18, 0] = [0, 255, 256, 0xFFFFFFFF, 0xFFFFFF00, 0xFFFFFE00, 1 << 31, 0xB504F300, 0xB504F400]
    _same(gpu_mc.debug_primitive(13, w, np.float32, len(w)),
          gpu_mc.debug_primitive(6, w, np.float32, len(w)))


def test_efficiency(gpu_mc):
    rng = np.random.default_rng(5)
    k = 1 << 21
    r0 = np.where(rng.random(k) < 0.5, 52.0, rng.uniform(1, 200, k)).astype(np.float32)
    r0[::17] = 2.0 ** rng.uniform(-39, 39, len(r0[::17]))
    rd = (r0 * rng.uniform(-0.3, 3, k)).astype(np.float32)
    rd[::5] = np.ldexp(rng.uniform(0.5, 1, len(rd[::5])), rng.integers(-126, 126, len(rd[::5])))
    rd[:6] = [0.0, -0.0, np.inf, -np.inf, np.nan, 1e-45]
    with np.errstate(all="ignore"):
        q = rd / r0
        q2 = q * q
        want = np.float32(1) / (np.float32(1) + (q2 * q2) * q2)
    _same(gpu_mc.debug_primitive(14, np.stack([rd, r0], 1), np.float32, k), want)


def test_reciprocal(gpu_mc):
    """Within the 2^-50 that binomial_broad's band counts with."""
    rng = np.random.default_rng(6)
    x = np.concatenate([rng.uniform(0.5, 1, 1 << 21), np.arange(1.0, 128.0),
                        1.0 - 2.0 ** -np.arange(1.0, 53.0)])
    got = gpu_mc.debug_primitive(16, x, np.float64, len(x))
    # 1 / x of numpy is within half an ulp (2^-53 relative)
    assert np.all(np.abs(got * x - 1.0) <= 2.0 ** -50)
    assert np.all(np.abs(got / (1.0 / x) - 1.0) <= 2.0 ** -50)


def test_broad_binomial(gpu_mc):
    """Random uniforms, and uniforms around the cumulative sums: every count it
    gives is the general draw's; within the band it gives none, and of the
    others next to none is left."""
    rng = np.random.default_rng(7)
    ps = np.concatenate([[0.0, 1.0, 0.5, 2.0 ** -140, 1 - 2.0 ** -24, np.nan, 0.50000006],
                         rng.uniform(0, 1, 53)]).astype(np.float32)
    n = np.arange(1, 128)
    items = []
    for p in ps:
        u = rng.integers(0, 1 << 53, (127, 200)).astype(np.int64)
        items.append((np.repeat(n, 200), np.full(127 * 200, p), u.ravel(),
                      np.full(127 * 200, 1 << 62)))
        pp = np.longdouble(p if p <= 0.5 else 1 - np.float64(p)) if p == p else None
        if pp is None:
            continue
        for m in range(1, 128, 3):
            k = np.arange(m + 1)
            ratio = np.concatenate([[1], (m - k[:-1]) * pp / ((k[:-1] + 1) * (1 - pp))])
            C = np.cumsum(np.cumprod(ratio.astype(np.longdouble)) * (1 - pp) ** m)
            t = np.minimum(C * np.longdouble(2) ** 53, np.longdouble(2) ** 53 - 1).astype(np.int64)
            for e in (-(1 << 20), -1025, -1, 0, 1, 1025, 1 << 20):
                u = t + e
                ok = (u >= 0) & (u < 1 << 53)
                items.append((np.full(ok.sum(), m), np.full(ok.sum(), p), u[ok],
                              np.full(ok.sum(), abs(e))))
    nn, pp, u, off = (np.concatenate([x[i] for x in items]) for i in range(4))
    it = np.zeros(len(u), BINOM_DT)
    it["n"], it["p"] = nn, pp
    it["hi"] = ((u >> 26) << 5).astype(np.uint32)
    it["lo"] = ((u & ((1 << 26) - 1)) << 6).astype(np.uint32)
    for f, v in (("seed", 1), ("set", 2), ("r", 3), ("b", 4), ("w", 7)):
        it[f] = v
    want = gpu_mc.debug_primitive(7, it, np.int64, len(it))
    got = gpu_mc.debug_primitive(15, it, np.int64, len(it))
    given = got >= 0
    assert np.array_equal(got[given], want[given])
    random = off == 1 << 62
    # 2^-38 on each side of at most 128 thresholds (and of 1, where they crowd)
    assert (~given & random).sum() <= 2 + random.sum() * 128 * 2.0 ** -37
    near = off < 1024
    # a threshold beyond the grid's last point was moved onto it
    assert near.sum() > 50_000 and not (given & near & (u < (1 << 53) - (1 << 21))).any()
