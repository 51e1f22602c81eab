"""The work a user of the library has it do, as measurable cases.

A case is one call pattern of the Python host interface (gsmfretda_amd.pda.MC)
on a data set that is already loaded, which is how a fit uses the library: the
bursts are loaded once, then parameter sets are evaluated one after another.
Every pass sets its parameters first, as every evaluation of a fit does.

kind:
  evaluate             one parameter set, blocking: set, walk, histogram, chi2
  samples              the same with the per-unit efficiencies read back
  streams              a round of parameter sets over three stream slots in
                       flight (one set per call, as the reference's worker)
  population           a generation of mixed-size parameter sets in one call
  rb_adjoint           Rao-Blackwellised forward and the chi2 gradient
  rb_jacobian          the same with the Jacobian of the expected histogram,
                       for `sets` parameter sets (1: the single-set calls)

Sizes: `bursts` x `resamples` units; a burst has base + Geometric(mean geom)
photons over a LogNormal(median dur_ms, dur_sigma) duration.  `states` is the
largest state count of the case's parameter sets; rates are log-uniform in
[rate_lo, rate_hi] per second; `broadening` is the largest distance width v in
Angstrom (0: none); bg_dd / bg_ad are the background rates in 1/s.
"""
import numpy as np
import torch

from gsmfretda_amd import pda, synth

SLOW = dict(base=50, geom=40.0, dur_ms=1.0, dur_sigma=0.5, rate_lo=1e2, rate_hi=1e4)
FAST = dict(base=30, geom=80.0, dur_ms=2.0, dur_sigma=0.6, rate_lo=1e3, rate_hi=1e5)
PLAIN = dict(sets=1, broadening=0.0, bg_dd=1000.0, bg_ad=500.0, bins=50)


def listed():
    return [
        # the smallest evaluation: a short two-state measurement, where the
        # launches and the host's part of the call count
        dict(PLAIN, **SLOW, name="evaluate_2state_small", kind="evaluate", states=2, bursts=5_000,
             resamples=20),
        # the reference's defaults: 4 resamples, 200 bins, a model with
        # distance broadening
        dict(PLAIN, **SLOW, name="evaluate_defaults", kind="evaluate", states=3, bursts=20_000,
             resamples=4) | dict(bins=200, broadening=4.0),
        # the repository's benchmark evaluation
        dict(PLAIN, **SLOW, name="evaluate_3state", kind="evaluate", states=3, bursts=100_000,
             resamples=100),
        # a large evaluation with distance broadening in the model
        dict(PLAIN, **SLOW, name="evaluate_broadened", kind="evaluate", states=3, bursts=50_000,
             resamples=50) | dict(broadening=5.0),
        # a measurement with a high background: part of the units needs the
        # draws beyond the common case
        dict(PLAIN, **SLOW, name="evaluate_background", kind="evaluate", states=3, bursts=50_000,
             resamples=50) | dict(bg_dd=30_000.0, bg_ad=15_000.0),
        # the simulated efficiencies themselves, read back per unit
        dict(PLAIN, **FAST, name="samples_5state", kind="samples", states=5, bursts=20_011,
             resamples=16),
        # a genetic algorithm's individuals one set per call, three in flight
        dict(PLAIN, **SLOW, name="streams_3state", kind="streams", states=3, bursts=50_000,
             resamples=32) | dict(sets=12),
        # a generation of a genetic algorithm in one call: the repository's
        # 256-set population
        dict(PLAIN, **SLOW, name="population_256", kind="population", states=4, bursts=50_000,
             resamples=32) | dict(sets=256),
        # a generation under fast dynamics: about ten windows per unit
        dict(PLAIN, **FAST, name="population_fast", kind="population", states=4, bursts=60_000,
             resamples=32) | dict(sets=64),
        # a generation of models with distance broadening
        dict(PLAIN, **SLOW, name="population_broadened", kind="population", states=4,
             bursts=20_000, resamples=16) | dict(sets=64, broadening=5.0),
        # a gradient step of a fit: forward and adjoint
        dict(PLAIN, **SLOW, name="rb_adjoint_3state", kind="rb_adjoint", states=3, bursts=100_000,
             resamples=64),
        # a step of a batched Levenberg-Marquardt fit under fast dynamics:
        # forward and Jacobian of four chains
        dict(PLAIN, **FAST, name="rb_jacobian_4state", kind="rb_jacobian", states=4, bursts=50_000,
             resamples=8) | dict(sets=4),
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(np.exp(rng.uniform(np.log(lo), np.log(hi)))))

    kind = rng.choice(["evaluate", "evaluate", "evaluate", "samples", "streams", "population",
                       "population", "rb_adjoint", "rb_jacobian"])
    rb = kind.startswith("rb_")
    c = dict(PLAIN, **rng.choice([SLOW, SLOW, FAST]), kind=kind)
    c["bins"] = rng.choice([50, 50, 100, 200])
    c["states"] = rng.randint(2, 4 if rb else 8 if kind == "samples" else 5)
    c["sets"] = {"streams": log_int(3, 12), "population": log_int(4, 256),
                 "rb_jacobian": rng.choice([1, 1, 4])}.get(kind, 1)
    c["bursts"] = log_int(2_000, 60_000 if kind == "rb_jacobian" else 100_000)
    c["resamples"] = log_int(4, 100)
    # no case above the listed ones: units of all sets, fewer under fast
    # dynamics (about six times the windows per unit)
    fast = c["rate_hi"] > 2e4
    most = {"evaluate": 10_000_000, "samples": 400_000, "streams": 12_000_000,
            "population": 100_000_000, "rb_adjoint": 6_000_000, "rb_jacobian": 6_000_000}[kind]
    if not rb and rng.random() < 0.35:
        c["broadening"] = round(rng.uniform(0.5, 6.0), 2)
        most //= 6
    if fast:
        most //= 4
    if rng.random() < 0.2:
        c["bg_dd"], c["bg_ad"] = rng.choice([(0.0, 0.0), (30_000.0, 15_000.0), (5_000.0, 8_000.0)])
    while c["bursts"] * c["resamples"] * c["sets"] > most:
        c["bursts"] = max(1_003, c["bursts"] * 2 // 3)
        c["resamples"] = max(4, c["resamples"] * 3 // 4)
        c["sets"] = max(1 if kind in ("evaluate", "samples", "rb_adjoint", "rb_jacobian") else 3,
                        c["sets"] * 3 // 4)
    return c


def _device():
    return torch.device("cuda", 0)


def _bursts(case, args, seed):
    """Bursts of the true kinetic model `args` (the distributions of
    gsmfretda_amd.synth.generate, drawn on the GPU)."""
    dev = _device()
    g = torch.Generator(device=dev).manual_seed(seed)

    def rand(n):
        return torch.rand(n, generator=g, device=dev, dtype=torch.float64)

    N, n = case["bursts"], case["states"]
    P = case["base"] + torch.floor(torch.log1p(-rand(N)) / np.log(1 - 1 / (case["geom"] + 1))).long()
    dur = 1e-3 * case["dur_ms"] * torch.exp(
        case["dur_sigma"] * torch.randn(N, generator=g, device=dev, dtype=torch.float64))
    dur = torch.clamp(torch.round(dur / synth.CLK_P).long(), 1, (1 << 31) - 2)
    istart = torch.cumsum(P, 0) - P
    owner = torch.repeat_interleave(torch.arange(N, device=dev), P)
    total = owner.numel()
    key = torch.sort((owner << 32) | (rand(total) * dur[owner]).long()).values
    start = 1_000_000 + torch.cumsum(dur + 200_000, 0) - (dur + 200_000)
    # the true trajectory: segments (burst, end tick, state)
    K = synth.rate_matrix(n, args)
    out_rate = torch.tensor(K.sum(axis=0), device=dev)
    jump = torch.tensor(np.cumsum(K / K.sum(axis=0), axis=0).T.copy(), device=dev)
    pi = torch.tensor(np.cumsum(synth.stationary(K)), device=dev)
    state = torch.clamp((rand(N)[:, None] > pi).sum(1), max=n - 1)
    t = torch.zeros(N, device=dev, dtype=torch.float64)
    act = torch.arange(N, device=dev)
    seg_key, seg_s = [], []
    while act.numel():
        s = state[act]
        end = t[act] - torch.log1p(-rand(act.numel())) / out_rate[s] / synth.CLK_P
        seg_key.append((act << 32) | torch.minimum(torch.ceil(end).long(), dur[act]))
        seg_s.append(s)
        t[act] = end
        state[act] = torch.clamp((rand(act.numel())[:, None] > jump[s]).sum(1), max=n - 1)
        act = act[end < dur[act]]
    seg_key, order = torch.sort(torch.cat(seg_key))
    seg = torch.searchsorted(seg_key, key, right=True)
    ph_state = torch.cat(seg_s)[order][torch.clamp(seg, max=seg_key.numel() - 1)]
    acc = rand(total) < torch.tensor(np.asarray(args[:n], np.float64), device=dev)[ph_state]
    host = lambda x, t: x.cpu().numpy().astype(t)  # noqa: E731
    return synth.BurstData(
        start=host(start, np.int64), stop=host(start + dur - 1, np.int64),
        istart=host(istart, np.int64), phcount=host(P, np.int32),
        times=host(start[owner] + (key & 0xFFFFFFFF), np.int64), mask_ad=host(acc, np.uint8),
        mask_dd=host(~acc, np.uint8), T=host(dur * synth.CLK_P, np.float32),
        bg_ad=case["bg_ad"], bg_dd=case["bg_dd"])


def _parameters(case, rng, n):
    E = np.sort(rng.uniform(0.05, 0.95, size=n))
    v = case["broadening"] * rng.uniform(0.2, 1.0, size=n)
    return synth.make_args(
        E, synth.loguniform_rates(rng, n * (n - 1), case["rate_lo"], case["rate_hi"]), v)


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    n = case["states"]
    truth = _parameters(case, rng, n)
    data = _bursts(case, truth, seed)
    # the sets a pass evaluates: a population mixes state counts, a round of
    # individuals and the chains of a fit share one
    sizes = [n] * case["sets"]
    if case["kind"] == "population" and n > 2:
        sizes = [int(x) for x in rng.integers(2, n + 1, size=case["sets"])]
    sets = [(k, _parameters(case, rng, k)) for k in sizes]
    slots = 3 if case["kind"] == "streams" else 1
    m = pda.MC(0, slots)
    m.load(data, SgDivSr=None)
    # observed efficiencies: one resample of the truth
    m.set_observed_hist(np.zeros(case["bins"], np.float32))
    for sid in range(slots):
        m.set_photophysics(sid, *synth.PHOTOPHYSICS)
        m.set_burst_range(0, -1, sid)
    m.set_params(n, 0, truth)
    m.reSampleTimes = 1
    m.run_kernel(sid=0, seed=seed & 0xFFFF, samples=True)
    m.synchronize(0)
    observed = m.get_samples(0, data.nbursts)[0]
    m.set_observed(observed, case["bins"], 2)
    m.reSampleTimes = case["resamples"]
    hist, _ = np.histogram(observed[(observed >= 0) & (observed < 1)], case["bins"], (0.0, 1.0))
    return dict(case=case, mc=m, sets=sets, seed=(seed * 7 + 3) & 0x7FFFFFFF,
                observed=hist.astype(np.float64))


def _read(m, sid):
    hist, c64, c32, eff = m.get_hist_chi2(sid)
    return dict(hist=hist, chi2=c64, chi2_ref=np.float32(c32), bins=eff)


def _run_evaluate(s):
    m, (n, args) = s["mc"], s["sets"][0]
    m.set_params(n, 0, args)
    m.run_kernel(sid=0, seed=s["seed"], set_id=0)
    m.synchronize(0)
    return _read(m, 0)


def _run_samples(s):
    m, (n, args) = s["mc"], s["sets"][0]
    m.set_params(n, 0, args)
    m.run_kernel(sid=0, seed=s["seed"], set_id=0, samples=True)
    m.synchronize(0)
    E, acc, F = m.get_samples(0, s["case"]["bursts"] * s["case"]["resamples"])
    return dict(_read(m, 0), E=E, acc=acc, F=F)


def _run_streams(s):
    m, sets = s["mc"], s["sets"]
    k = m.streamNum
    out = [None] * len(sets)
    for i, (n, args) in enumerate(sets):
        if i >= k:
            m.synchronize(i % k)
            out[i - k] = _read(m, i % k)
        m.set_params(n, i % k, args)
        m.run_kernel(sid=i % k, seed=s["seed"], set_id=i)
    for i in range(max(0, len(sets) - k), len(sets)):
        m.synchronize(i % k)
        out[i] = _read(m, i % k)
    return {key: np.stack([o[key] for o in out]) for key in out[0]}


def _run_population(s):
    m, sets = s["mc"], s["sets"]
    m.set_population([n for n, _ in sets], [a for _, a in sets])
    m.run_population(R=s["case"]["resamples"], seed=s["seed"])
    hist, c64, c32, eff = m.get_population_result()
    return dict(hist=hist, chi2=c64, chi2_ref=c32, bins=eff)


def _cotangent(s, M, n):
    """d chi2 / d M of the reduced chi2 on the expected counts."""
    R, B = s["case"]["resamples"], s["case"]["bins"]
    keep = (np.arange(B) >= 2) & (M > 0)
    g = np.zeros(M.shape)
    mm, O = M / R, np.broadcast_to(s["observed"], M.shape)
    dof = np.maximum(keep.sum(-1, keepdims=True) - n * (n + 1), 1)
    g[keep] = ((1.0 - (O / np.where(keep, mm, 1.0)) ** 2) / (R * dof))[keep]
    return g


def _run_rb_adjoint(s):
    m, (n, args) = s["mc"], s["sets"][0]
    m.set_params(n, 0, args)
    m.rb_forward(seed=s["seed"], set_id=0)
    M, fixed, c2, eff = m.rb_result()
    return dict(M=M, fixed=fixed.astype(np.int64), chi2=c2, bins=eff,
                grad=m.rb_adjoint(_cotangent(s, M, n), n))


def _run_rb_jacobian(s):
    m, sets, B = s["mc"], s["sets"], s["case"]["bins"]
    n = sets[0][0]
    if len(sets) == 1:
        m.set_params(n, 0, sets[0][1])
        m.rb_forward(seed=s["seed"], set_id=0)
        M, fixed, c2, eff = m.rb_result()
        J = m.rb_jacobian(n, B)
    else:
        m.set_population([k for k, _ in sets], [a for _, a in sets])
        m.rb_forward_population(seed=s["seed"], set_base=0, set_stride=0)
        M, fixed, c2, eff = m.rb_population_result()
        J = m.rb_jacobian_population(n, B)
    return dict(M=M, fixed=fixed.astype(np.int64), chi2=c2, bins=eff, jacobian=J)


def run(state):
    return {"evaluate": _run_evaluate, "samples": _run_samples, "streams": _run_streams,
            "population": _run_population, "rb_adjoint": _run_rb_adjoint,
            "rb_jacobian": _run_rb_jacobian}[state["case"]["kind"]](state)


def exact(case, seed):
    """No output has a value in 64 bits: the histograms, and the expected
    counts and derivatives conditional on the walks, are functions of which
    photons fall into which dwell window, and that is decided by the keyed
    random stream through the library's own 32-bit dwell times."""
    return None


def work(case):
    """What the path cannot do without.  Bytes: every photon's tick and
    channel (5 B) and every burst's descriptor (16 B) read once, the results
    written once (the derivative passes also hand over the per-unit counts,
    F and scores of the walk: written once, read once).  Operations: per
    dwell window two blocks of the random stream (about 100 integer
    operations each counting a 32 x 32 -> 64 bit product as one) and about
    100 for the dwell, the window's count and the draws; models with
    broadening one more block and a normal variate; per unit 40 for its bin;
    in the Rao-Blackwellised form per outcome and derivative a multiply-add."""
    units = case["bursts"] * case["resamples"] * case["sets"]
    photons = case["bursts"] * (case["base"] + case["geom"])
    n = case["states"]
    rate = 1e-3 * case["dur_ms"] * float(np.sqrt(case["rate_lo"] * case["rate_hi"])) * (n - 1)
    windows = 1.0 + min(0.45 * rate, 12.0)
    per_window = 300.0 if case["broadening"] == 0 else 450.0
    if case["bg_dd"] == 0:
        per_window -= 130.0
    bytes_ = 5.0 * photons + 16.0 * case["bursts"] + 4.0 * case["bins"] * case["sets"]
    flops = units * (windows * per_window + 40.0)
    if case["kind"] == "samples":
        bytes_ += 12.0 * units
    if case["kind"].startswith("rb_"):
        K = n * (n - 1)
        bytes_ += 2.0 * units * (12.0 + 4.0 * K)
        flops += units * 7.0 * (20.0 + 2.0 * (n + K))
    return {"bytes": bytes_, "flops": flops}
