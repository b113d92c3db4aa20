"""Workloads of the framework's public entry points, for timing.

Each case is one call that a user's program makes, with what that program has
in hand before it: a search plan with its spectrum set, a candidate list, the
series of a batch of DM trials.  listed() covers the range of sizes and options
that the configurations, tests and bench.py use; draw() gives others of the
same ranges.  prepare() makes the inputs on the GPU (or, for the candidate
stage, on the host, where its entry point takes them), run() makes one call and
returns everything it computed, exact() gives the same outputs in 64 bits where
plain numpy or torch can.
"""
import math

import numpy as np
import torch

from prestozl_amd import binding as B

# The lengths that realfft takes: n/2 a product of 2, 3, 5, 7 and 11.
_PRIMES = (2, 3, 5, 7, 11)

MAXCANDS = 8192  # candidates a search may return


def listed():
    return [
        # An acceleration search of a short pointing, as a survey runs by the
        # thousand: a few rsteps, so launches and host work are the cost.
        dict(name="accel_short", kind="search", N=1 << 17, dt=64e-6, zmax=20, wmax=0, jerk=False, numharm=4,
             sigma=3.0, batch=8, tuned=False),
        # bench.py's smallest shape: N = 2^20, zmax 20, -wmax 0, 4 harmonics.
        dict(name="accel_config1", kind="search", N=1 << 20, dt=64e-6, zmax=20, wmax=0, jerk=True, numharm=4,
             sigma=2.0, batch=8, tuned=False),
        # The acceleration search of the served stream: (50, 0, 8) at 2^21.
        dict(name="accel_served", kind="search", N=1 << 21, dt=1e-4, zmax=50, wmax=0, jerk=True, numharm=8,
             sigma=4.0, batch=8, tuned=False),
        # One DM trial of a dedispersion run: (200, 300, 8) at 2^18, read from
        # device memory.
        dict(name="jerk_dm_trial", kind="search", N=1 << 18, dt=6.4e-4, zmax=200, wmax=300, jerk=True, numharm=8,
             sigma=5.0, batch=8, tuned=False),
        # The served stream's and the headline's jerk search, (200, 300, 16),
        # tuned as bench.py tunes it, at a quarter of the headline's length.
        dict(name="jerk_long", kind="search", N=1 << 22, dt=1e-4, zmax=200, wmax=300, jerk=True, numharm=16,
             sigma=5.0, batch=8, tuned=True),
        # The widest kernels configured: wmax 500, a 4096-point fundamental.
        dict(name="jerk_wide", kind="search", N=1 << 20, dt=1e-4, zmax=200, wmax=500, jerk=True, numharm=16,
             sigma=5.0, batch=8, tuned=False),
        # The candidate stage after a jerk search: every candidate's harmonics
        # polished on the oversampled (r, z, w) volume.
        dict(name="polish_jerk", kind="polish", N=1 << 20, ncand=96, zmax=200, wmax=300, maxharm=16, fdot=False),
        # ... and after an acceleration search: the downhill simplex.
        dict(name="polish_accel", kind="polish", N=1 << 20, ncand=32, zmax=60, wmax=0, maxharm=8, fdot=True),
        # realfft of the headline's series.
        dict(name="realfft_long", kind="realfft", n=1 << 24, nseries=1, isign=-1),
        # realfft of every DM trial of a dedispersion run in one call.
        dict(name="realfft_trials", kind="realfft", n=1 << 18, nseries=564, isign=-1),
        # The inverse, at a length that is no power of two (choose_good_N's).
        dict(name="realfft_inverse", kind="realfft", n=2112000, nseries=3, isign=1),
        # Dedispersion of 64 subbands into the 564 trials.
        dict(name="dedisp_trials", kind="dedisp", nsamp=1 << 18, nsub=64, worklen=16384, numdms=564, maxoff=6000),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _smooth_even(rng, lo, hi):
    """An even length with n/2 = 2^a 3^b 5^c 7^d 11^e, near a log-uniform point."""
    target = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    m = 1
    for p in rng.choices(_PRIMES, k=rng.randint(0, 4)):
        if m * p * 2 <= target:
            m *= p
    while m * 4 <= target:
        m *= 2
    return 2 * m


def draw(rng):
    kind = rng.choice(["accel", "accel", "jerk", "jerk", "jerk", "polish", "realfft", "realfft", "dedisp"])
    if kind == "accel":
        return dict(kind="search", N=2 * _log_int(rng, 1 << 16, 1 << 20), dt=rng.choice([64e-6, 1e-4, 6.4e-4]),
                    zmax=2 * rng.randint(0, 60), wmax=0, jerk=rng.random() < 0.5, numharm=rng.choice([1, 2, 4, 8, 16]),
                    sigma=round(rng.uniform(2.5, 5.0), 2), batch=rng.choice([4, 8, 8, 16]), tuned=False)
    if kind == "jerk":
        return dict(kind="search", N=2 * _log_int(rng, 1 << 15, 1 << 19), dt=rng.choice([1e-4, 6.4e-4]),
                    zmax=2 * rng.randint(5, 100), wmax=20 * rng.randint(1, 25), jerk=True,
                    numharm=rng.choice([1, 2, 4, 8, 16]), sigma=round(rng.uniform(4.5, 6.0), 2),
                    batch=rng.choice([4, 8, 8, 16]), tuned=False)
    if kind == "polish":
        fdot = rng.random() < 0.4
        return dict(kind="polish", N=2 * _log_int(rng, 1 << 17, 1 << 19), ncand=_log_int(rng, 1, 32 if fdot else 96),
                    zmax=2 * rng.randint(5, 30 if fdot else 100), wmax=0 if fdot else 20 * rng.randint(1, 15),
                    maxharm=rng.choice([1, 2, 4, 8, 16]), fdot=fdot)
    if kind == "realfft":
        n = _smooth_even(rng, 1 << 10, 1 << 24)
        return dict(kind="realfft", n=n, nseries=_log_int(rng, 1, max(1, min(564, (1 << 26) // n))),
                    isign=rng.choice([-1, 1]))
    worklen = _log_int(rng, 1000, 16384)
    return dict(kind="dedisp", nsamp=worklen * rng.randint(1, 16), nsub=_log_int(rng, 8, 320), worklen=worklen,
                numdms=_log_int(rng, 4, 564), maxoff=rng.randint(0, worklen))


# ---- inputs ----------------------------------------------------------------

def _rng(seed):
    return np.random.Generator(np.random.PCG64(seed))


def _spectrum(N, rng, signals, normalise=True):
    """numbins complex64 in realfft's packing: noise of unit mean power plus
    signals (power over the noise, fraction of the band, z, w)."""
    t = np.arange(N, dtype=np.float64) / N
    x = rng.standard_normal(N)
    for power, f, z, w in signals:
        r = f * (N // 2)
        x += math.sqrt(4.0 * power / N) * np.cos(2.0 * np.pi * t * (r + t * (0.5 * z + t * w / 6.0)))
    X = np.fft.rfft(x)
    out = np.empty(N // 2, dtype=np.complex128)
    out[0] = complex(X[0].real, X[-1].real)
    out[1:] = X[1:N // 2]
    if normalise:
        out /= math.sqrt(N)
    return out.astype(np.complex64)


def _config(case):
    return B.make_config(N=case["N"], dt=case["dt"], numbins=case["N"] // 2, zmax=case["zmax"], wmax=case["wmax"],
                         wmaxP=case["jerk"], numharm=case["numharm"], sigma=case["sigma"], batchsize=case["batch"])


def _search_spectrum(case, seed):
    rng = _rng(seed)
    z, w = 0.8 * case["zmax"], 0.8 * case["wmax"]
    # two pulsars (with harmonics) and a tone, of the strengths searches find
    sig = []
    for k in range(2):
        f, zz, ww = rng.uniform(0.02, 0.1), rng.uniform(-z, z), rng.uniform(-w, w)
        for h in range(1, min(case["numharm"], 4) + 1):
            sig.append((rng.uniform(20.0, 60.0), f * h, zz * h / case["numharm"], ww * h / case["numharm"]))
    sig.append((rng.uniform(60.0, 200.0), rng.uniform(0.1, 0.45), rng.uniform(-z, z), rng.uniform(-w, w)))
    return _spectrum(case["N"], rng, sig)


def _polish_inputs(case, seed):
    rng = _rng(seed)
    N, zmax, wmax = case["N"], case["zmax"], case["wmax"]
    nbins = N // 2
    cands, sig = [], []
    for k in range(case["ncand"]):
        nh = 2 ** (k % (int(math.log2(case["maxharm"])) + 1))
        # a search's candidate: on the grid of its highest harmonic
        z = 2.0 * rng.integers(-zmax // 2, zmax // 2 + 1) / nh
        w = 20.0 * rng.integers(-wmax // 20, wmax // 20 + 1) / nh
        r = rng.integers(int(0.04 * nbins), int(1.9 * nbins * 0.45)) * 0.5 / nh + 2000.0 / nh
        cands.append((float(r), float(z), float(w), nh))
        if k % 8 == 0:  # signals for some of them; the others are noise peaks
            f0 = r - 0.5 * z + w / 12.0
            for h in range(1, nh + 1):
                sig.append((rng.uniform(20.0, 60.0), f0 * h / nbins, (z - 0.5 * w) * h, w * h))
    return _spectrum(N, rng, sig[:24]), cands


def _dedisp_inputs(case, seed):
    rng = _rng(seed)
    x = rng.standard_normal((case["nsamp"], case["nsub"]), dtype=np.float32) + np.float32(0.5)
    f = np.linspace(0.6, 1.0, case["nsub"])
    d = 1.0 / f ** 2 - 1.0 / f[-1] ** 2
    dm = np.linspace(rng.uniform(0.0, 0.2), 1.0, case["numdms"])
    offs = np.rint(dm[:, None] * (d / max(d.max(), 1e-30))[None, :] * case["maxoff"]).astype(np.int32)
    return x, np.minimum(offs, case["worklen"])


def _realfft_input(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.randn(case["nseries"], case["n"], generator=g, device="cuda", dtype=torch.float32)


def prepare(case, seed):
    if case["kind"] == "search":
        fft = torch.from_numpy(_search_spectrum(case, seed)).cuda()
        plan = B.Plan(_config(case))
        plan.set_spectrum_device(fft.data_ptr(), fft.numel())
        if case["tuned"]:
            plan.autotune(reps=2)
        return dict(kind="search", plan=plan, fft=fft)
    if case["kind"] == "polish":
        fft, cands = _polish_inputs(case, seed)
        return dict(kind="polish", fft=fft, cands=cands, fdot=case["fdot"])
    if case["kind"] == "realfft":
        x = _realfft_input(case, seed)
        return dict(kind="realfft", x=x, buf=torch.empty_like(x), n=case["n"], nseries=case["nseries"],
                    isign=case["isign"])
    x, offs = _dedisp_inputs(case, seed)
    return dict(kind="dedisp", x=torch.from_numpy(x).cuda(), offs=torch.from_numpy(offs).cuda(),
                out=torch.empty(case["numdms"], case["nsamp"], device="cuda", dtype=torch.float32), case=case)


# ---- one pass --------------------------------------------------------------

def run(state):
    kind = state["kind"]
    if kind == "search":
        # the candidate list, in a table of fixed length as the C call fills one
        cands, _ = state["plan"].search(maxcands=MAXCANDS, stats=False)
        a = np.zeros((MAXCANDS, 6))
        a[:len(cands)] = np.array(cands, dtype=np.float64).reshape(-1, 6)
        return dict(count=len(cands), power=a[:, 0].astype(np.float32), sigma=a[:, 1].astype(np.float32),
                    numharm=a[:, 2].astype(np.int32), r=a[:, 3], z=a[:, 4], w=a[:, 5])
    if kind == "polish":
        got = B.optimize_spectrum(state["fft"], state["cands"], fdot_only=state["fdot"])
        # the powers and derivatives come from single-precision amplitudes
        keys = ("pow", "phs", "dpow", "dphs", "d2pow", "d2phs", "locpow")
        der = [[d[k] for k in keys] for g in got for d in g["derivs"]]
        return dict(rzw=np.array([[g["r"], g["z"], g["w"]] for g in got]),
                    pows=np.array([p for g in got for p in g["pows"]], dtype=np.float32),
                    **{k: np.array([d[i] for d in der], dtype=np.float32) for i, k in enumerate(keys)})
    if kind == "realfft":
        # the transform is in place: the program's series go into its buffer first
        state["buf"].copy_(state["x"])
        B.realfft_device(state["buf"].data_ptr(), state["n"], state["isign"], nseries=state["nseries"])
        return state["buf"]
    c = state["case"]
    B.dedisperse(state["x"].data_ptr(), c["nsamp"], c["nsub"], c["worklen"], c["numdms"], state["offs"].data_ptr(),
                 state["out"].data_ptr())
    return state["out"]


# ---- what one pass cannot do without ---------------------------------------

def work(case):
    if case["kind"] == "search":
        g = B.geometry(_config(case))
        # the spectrum is read once; every power of every (z, w, r) plane is one
        # point of a correlation of fftlen points (5 log2 n) times its kernel (6)
        # and squared (3), and every fundamental cell sums its harmonics
        planes = g.plane_bytes_per_rstep / 4.0
        cells = float(g.corr_uselen) * g.numz * max(g.numw, 1)
        return dict(bytes=8.0 * (case["N"] // 2),
                    flops=g.nrsteps * (planes * (5.0 * math.log2(g.fftlen) + 9.0) + cells * (case["numharm"] - 1)))
    if case["kind"] == "polish":
        # per candidate harmonic (half of maxharm on average): the 17 x 17 grid
        # of responses of about 1024 chirp samples in 64 bits and 24 fine r
        # steps of 300 bins each; the simplex: about 100 points of 200 bins
        jobs = case["ncand"] * max(1.0, case["maxharm"] / 2.0)
        flops = jobs * 100 * 200 * 60.0 if case["fdot"] else jobs * 289 * (1024 * 60.0 + 24 * 300 * 8.0)
        return dict(bytes=8.0 * (case["N"] // 2), flops=flops)
    if case["kind"] == "realfft":
        total = float(case["n"]) * case["nseries"]
        return dict(bytes=8.0 * total, flops=2.5 * total * math.log2(case["n"]))
    return dict(bytes=4.0 * case["nsamp"] * (case["nsub"] + case["numdms"]) + 4.0 * case["numdms"] * case["nsub"],
                flops=float(case["nsamp"]) * case["nsub"] * case["numdms"])


# ---- the same in 64 bits ---------------------------------------------------

def exact(case, seed):
    if case["kind"] == "realfft":
        n, ns = case["n"], case["nseries"]
        x = _realfft_input(case, seed)
        out = torch.empty(ns, n, device="cuda", dtype=torch.float64)
        for s in range(ns):
            if case["isign"] == -1:
                X = torch.fft.rfft(x[s].double())
                out[s] = torch.view_as_real(X[:-1]).reshape(-1)
                out[s, 1] = X[-1].real
            else:
                v = torch.view_as_complex(x[s].double().reshape(-1, 2))
                X = torch.cat([v, v[:1].imag.to(v.dtype)])
                X[0] = v[0].real.to(v.dtype)
                out[s] = torch.fft.irfft(X, n=n)
        return out
    if case["kind"] == "dedisp":
        x, offs = _dedisp_inputs(case, seed)
        n = case["nsamp"]
        sub = torch.zeros(case["nsub"], n + case["worklen"], device="cuda", dtype=torch.float64)
        sub[:, :n] = torch.from_numpy(x).cuda().T
        out = torch.empty(case["numdms"], n, device="cuda", dtype=torch.float64)
        idx = torch.arange(n, device="cuda")
        for d in range(case["numdms"]):
            o = torch.from_numpy(offs[d].astype(np.int64)).cuda()
            out[d] = torch.gather(sub, 1, idx[None, :] + o[:, None]).sum(dim=0)
        return out
    # A search's candidate list and a polished candidate need every response,
    # correlation and maximum of the method in 64 bits: far over 20 seconds in
    # numpy at these sizes.
    return None
