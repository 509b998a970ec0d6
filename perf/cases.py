"""The workloads this library is timed on, through its public entry points.

Every case is one pass of one job: a network's records (or a station pair's rows)
in, its correlations out.  Device cases hold their records in HBM and keep a
DeviceRunner (job, workspace and output buffer), as a program does that correlates
a network day after day; the host cases hand numpy rows to the reference's own
entry points.  listed() names the cases, draw() takes one more from the ranges
they stand for, exact() computes a case in 64 bits with plain torch.
"""
import math

import torch

from fastpcc_amd import api

# What each listed case stands for, with the sizes of this repository's benchmark
# and tests or ragged neighbours of them:
_LISTED = [
    # a handful of stations, one hour: the smallest job, bound by launches and latency
    dict(name="hour_8st_pcc2", entry="device", kind="pcc2", stack="plain", S=8, W=1, N=3600, lag1=-500, lag2=500),
    # the benchmark's headline: a 256-station day in hourly windows, mean stack, split-FP16 Gram
    dict(name="day_256st_gram16", entry="device", kind="pcc2", stack="gram16", S=256, W=24, N=3600, lag1=-1000,
         lag2=1000),
    # the FP32 stack of an odd network: 97 stations, 17 windows of 2880 samples, one-sided lags
    dict(name="ragged_97st_gram", entry="device", kind="pcc2", stack="gram", S=97, W=17, N=2880, lag1=-250, lag2=750),
    # 64 stations, every hour's correlation on its own, then the mean (no spectral stack)
    dict(name="day_64st_pcc2", entry="device", kind="pcc2", stack="plain", S=64, W=24, N=3600, lag1=-1000, lag2=1000),
    # geometrically normalised correlation of the same network, FP64 as the reference
    dict(name="day_64st_gncc", entry="device", kind="gncc", stack="plain", S=64, W=24, N=3600, lag1=-1000, lag2=1000),
    # 1-bit correlation of an odd network in half-hour windows, every window kept
    dict(name="halfhour_45st_cc1b", entry="device", kind="cc1b", stack="none", S=45, W=30, N=1800, lag1=-600, lag2=600),
    # phase-weighted stack of a day
    dict(name="day_48st_pws", entry="device", kind="pcc2", stack="pws", S=48, W=24, N=3600, lag1=-1000, lag2=1000),
    # PCC of power 1: time-domain sums, no FFT form
    dict(name="day_16st_pcc1", entry="device", kind="pcc1", stack="plain", S=16, W=24, N=3600, lag1=-1000, lag2=1000),
    # the reference's published benchmark: one pair, 649 day-long windows at 4 s, every window kept
    dict(name="pair_649x21600_pcc2", entry="device", kind="pcc2", stack="none", S=2, W=649, N=21600, lag1=-3000,
         lag2=3000),
    # a network's whole days at 1 Hz as one window each
    dict(name="wholeday_32st_pcc2", entry="device", kind="pcc2", stack="plain", S=32, W=1, N=86400, lag1=-2000,
         lag2=2000),
    # wavelet PCC of whole days: 56 scales, periods 2 to 200 samples
    dict(name="wholeday_24st_wpcc", entry="device", kind="wpcc", stack="plain", S=24, W=1, N=86400, lag1=-2000,
         lag2=2000, pmin=2.0, pmax=200.0, V=8),
    # the drop-in call on host rows, one station pair over a day's hours
    dict(name="host_pair_24x3600_pcc2", entry="host", kind="pcc2", stack="none", S=2, W=24, N=3600, lag1=-1000,
         lag2=1000),
]


def listed():
    return [dict(c) for c in _LISTED]


def _logint(rng, a, b):
    return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))


_ROUND_N = (600, 900, 1200, 1500, 1800, 2000, 2400, 2880, 3000, 3200, 3600, 3750, 4000)


def _window(rng):
    """A window of the hourly kind: mostly round lengths, else any."""
    return rng.choice(_ROUND_N) if rng.random() < 0.7 else rng.randint(600, 4096)


def _lags(rng, N, most):
    m = min(most, N // 2)
    hi = _logint(rng, max(2, m // 8), m)
    r = rng.random()
    if r < 0.6:
        return -hi, hi
    if r < 0.8:
        return -rng.randint(0, hi), hi
    return rng.randint(-hi, hi - 1), hi


def _fits(c):
    top = [max(work(l)[k] for l in _LISTED) for k in ("bytes", "flops")]
    w = work(c)
    return w["bytes"] <= top[0] and w["flops"] <= top[1]


def draw(rng):
    """One more case of the listed ones' ranges: networks of 8 to 256 stations with a
    spectral stack; of 2 to 64 with every window transformed; time-domain sums of 2 to
    16; long windows of a pair or of up to 32 stations; wavelet PCC of 2 to 24; host
    pairs.  No larger than the largest listed case."""
    while True:
        what = rng.choice(("spectral", "windows", "windows", "time", "long", "long", "wpcc", "host"))
        c = dict(entry="device")
        if what == "spectral":
            c.update(kind=rng.choice(("pcc2", "pcc2", "cc1b")), stack=rng.choice(("gram16", "gram")),
                     S=_logint(rng, 8, 256), W=rng.randint(4, 32), N=_window(rng))
            lag = 1000
        elif what == "windows":
            c.update(kind=rng.choice(("pcc2", "gncc", "cc1b")), stack=rng.choice(("none", "plain", "pws")),
                     S=_logint(rng, 2, 64), W=rng.randint(1, 32), N=_window(rng))
            lag = 1000
            if c["stack"] == "pws" and c["kind"] == "pcc2":  # the analytic signal in one workgroup
                c["N"] = rng.choice(_ROUND_N)
        elif what == "time":
            c.update(kind=rng.choice(("pcc1", "pccv")), stack=rng.choice(("none", "plain")), S=_logint(rng, 2, 16),
                     W=rng.randint(1, 24), N=_window(rng))
            if c["kind"] == "pccv":
                c.update(v=rng.choice((0.5, 1.0, 1.5, 2.0)), S=_logint(rng, 2, 10))
            lag = 1000
        elif what == "long":
            c.update(kind=rng.choice(("pcc2", "pcc2", "gncc", "cc1b")), stack=rng.choice(("none", "plain")))
            if rng.random() < 0.5:
                c.update(S=2, W=_logint(rng, 8, 400), N=_logint(rng, 5000, 30000))
            else:
                c.update(S=_logint(rng, 3, 32), W=1, N=_logint(rng, 10000, 86400))
            lag = 3000
        elif what == "wpcc":
            c.update(kind="wpcc", stack="plain", S=_logint(rng, 2, 24), W=1, N=_logint(rng, 7200, 86400), pmin=2.0,
                     pmax=float(rng.choice((32, 100, 200))), V=rng.choice((4, 8)))
            lag = 2000
        else:
            c.update(entry="host", kind=rng.choice(("pcc2", "gncc", "cc1b", "pcc1")), stack="none", S=2,
                     W=rng.randint(1, 48), N=_logint(rng, 1800, 21600))
            lag = 1000
        c["lag1"], c["lag2"] = _lags(rng, c["N"], lag)
        if _fits(c):
            return c


# ---- inputs ----

def _device():
    return torch.device("cuda:0" if torch.cuda.is_available() else "cpu")


def _records(case, seed):
    """[S][W*N] float32 records: each station's own noise, a band-limited source all
    stations share at true delays, and now and then (one window in about 24) an event
    some 30 times the noise that decays over a few hundred samples."""
    dev = _device()
    S, n = case["S"], case["W"] * case["N"]
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    most = min(200, case["N"] // 8)
    m = n + 2 * most
    f = torch.fft.rfftfreq(m, device=dev)
    band = torch.exp(-((f - 0.11) / 0.05) ** 2)
    src = torch.fft.irfft(torch.fft.rfft(torch.randn(m, generator=g, device=dev)) * band, m)
    src = src / src.std()
    t = torch.arange(m, device=dev)
    for _ in range(max(1, case["W"] // 24)):
        t0 = int(torch.randint(0, m, (1,), generator=g, device=dev))
        age = (t - t0).float()
        src = src + torch.where(age >= 0, 30 * torch.exp(-age / 150) * torch.sin(age * 0.6), torch.zeros_like(age))
    shift = torch.randint(0, 2 * most + 1, (S,), generator=g, device=dev).tolist()
    x = torch.randn((S, n), generator=g, device=dev)
    for s in range(S):
        x[s] += 0.5 * src[shift[s]:shift[s] + n]
    return x


def prepare(case, seed):
    x = _records(case, seed)
    if case["entry"] == "host":
        rows = x.view(2, case["W"], case["N"]).cpu().numpy()
        return dict(case=case, x1=rows[0].copy(), x2=rows[1].copy())
    kw = {k: case[k] for k in ("v", "pmin", "pmax", "V") if k in case}
    job = api.make_job(case["kind"], case["S"], case["W"], case["N"], case["lag1"], case["lag2"], case["stack"], **kw)
    return dict(case=case, x=x, runner=api.DeviceRunner(job, str(x.device)))


_HOST = {"pcc2": api.pcc2_set, "gncc": api.ccgn_set, "cc1b": api.cc1b_set, "pcc1": api.pcc1_set}


def run(state):
    case = state["case"]
    if case["entry"] == "host":
        return _HOST[case["kind"]](state["x1"], state["x2"], case["lag1"], case["lag2"])
    return state["runner"].run(state["x"])


# ---- work and tolerance ----

def _sizes(case):
    S, W, N = case["S"], case["W"], case["N"]
    L = case["lag2"] - case["lag1"] + 1
    if case["kind"] == "wpcc":
        L = abs(case["lag2"] - case["lag1"]) + 1
    Nz = 1
    while Nz < N + max(abs(case["lag1"]), abs(case["lag2"])):
        Nz *= 2
    return S, W, N, L, Nz, S * (S - 1) // 2


def work(case):
    """Records read once, correlations written once; the transforms of every window
    once, a multiply-add per pair, window and kept bin, one inverse per output row
    (per window where each window is normalised or weighted by itself), or the
    time-domain sums.  A transform of n complex points counts 5 n log2 n."""
    S, W, N, L, Nz, P = _sizes(case)
    rows = P * W if case["stack"] == "none" else P
    nbytes = 4 * S * W * N + 4 * rows * L

    def fft(n):
        return 5 * n * math.log2(n)

    kind = case["kind"]
    if kind in ("pcc1", "pccv"):
        terms = sum(N - abs(l) for l in range(case["lag1"], case["lag2"] + 1))
        flops = S * W * 2 * fft(N) + 12 * P * W * terms
    elif kind == "wpcc":
        fam = _bank_sizes(case)
        flops = S * W * (1 + 2 * fam["S"]) * fft(fam["Nz"]) + P * W * fam["S"] * fam["Nz"] * 8 + rows * fft(fam["Nz"])
    else:
        each = case["stack"] in ("none", "pws") or kind == "gncc"
        station = 2 * fft(N) + fft(Nz) if kind == "pcc2" else fft(Nz) / 2
        inverse = fft(Nz) / 2 * (2 if case["stack"] == "pws" else 1)
        bins = (2 if kind == "pcc2" else 1) * (Nz // 2 + 1)
        flops = S * W * station + P * W * bins * 8 + (P * W if each else P) * inverse
    return dict(bytes=int(nbytes), flops=int(flops))


def tolerance(case):
    """About four times the largest differences seen between the present code and
    exact() over the listed and some twenty drawn cases: FP32 transforms and sums
    leave about 1e-7 in a correlation of full scale 1, which is up to 1e-6 of the
    0.005 to 0.05 these records correlate at (1e-5 at single lags, 2e-5 where a phase
    stack divides by |a|); wavelet PCC, whose phasors of every scale add up, 5e-6 and
    2.6e-5; GNCC up to 8192 points is FP64 rounded to float at the end."""
    if case["kind"] == "wpcc":
        return {"rel": 2e-5, "max": 1e-4}
    if case["kind"] == "gncc" and _sizes(case)[4] <= 8192 and case["stack"] != "pws":
        return {"rel": 4e-7, "max": 2e-6}
    return {"rel": 4e-6, "max": 8e-5 if case["stack"] == "pws" else 4e-5}


# ---- the same outputs in 64 bits ----

def _phasors(x):
    """[..., N] float64 records -> unit phasors of the analytic signal, regularised."""
    N = x.shape[-1]
    X = torch.fft.fft(x)
    mask = torch.zeros(N, dtype=torch.float64, device=x.device)
    mask[0] = 1
    mask[1:(N + 1) // 2] = 2
    if N % 2 == 0:
        mask[N // 2] = 1
    z = torch.fft.ifft(X * mask)
    a = z.abs()
    return z / (a + 1e-6 * a.amax(-1, keepdim=True))


def _pairs(S):
    return [(i, j) for i in range(S) for j in range(i + 1, S)]


def _stacked(case, c):
    return c if case["stack"] == "none" else c.mean(-2)


def _exact_spectral(case, x):
    S, W, N, L, Nz, P = _sizes(case)
    kind, stack, dev = case["kind"], case["stack"], x.device
    lags = torch.arange(case["lag1"], case["lag2"] + 1, device=dev)
    over = (N - lags.abs()).double()
    if kind == "pcc2":
        a = b = torch.fft.fft(_phasors(x), n=Nz)
    elif kind == "cc1b":
        one = torch.ones((), dtype=torch.float64, device=dev)
        a = torch.fft.fft(torch.where(x >= 0, one, -one), n=Nz)
        b = torch.fft.fft(torch.where(x > 0, one, -one), n=Nz)
    else:
        a = b = torch.fft.fft(x, n=Nz)
        E = torch.zeros((S, W, N + 1), dtype=torch.float64, device=dev)
        E[..., 1:] = torch.cumsum(x * x, -1)
        e1 = E[..., torch.clamp(N - lags, max=N)] - E[..., torch.clamp(-lags, min=0)]
        e2 = E[..., torch.clamp(N + lags, max=N)] - E[..., torch.clamp(lags, min=0)]
    out = []
    step = max(1, (1 << 27) // (W * Nz))
    half = torch.zeros(Nz, dtype=torch.float64, device=dev)
    half[0] = half[Nz // 2] = 1
    half[1:Nz // 2] = 2
    for i in range(S - 1):
        for j0 in range(i + 1, S, step):
            j = slice(j0, min(S, j0 + step))
            Y = a[i].conj() * b[j]  # [pairs][W][Nz]
            if stack not in ("none", "pws") and kind != "gncc":
                Y = Y.mean(1, keepdim=True)
            c = torch.fft.ifft(Y)
            r = c.real[..., lags % Nz]
            if kind == "pcc2":
                r = r / N
            elif kind == "cc1b":
                r = r / over
            else:
                r = r / (e1[i] * e2[j]).sqrt()
            if stack == "none":
                out.append(r)
                continue
            r = r.mean(1)
            if stack == "pws":
                z = torch.fft.ifft(torch.fft.fft(c.real) * half)[..., lags % Nz]
                r = r * (z / z.abs()).mean(1).abs() ** 2
            out.append(r)
    return torch.cat(out)


def _exact_time(case, x):
    S, W, N, L, Nz, P = _sizes(case)
    phi = _phasors(x)
    v = case.get("v", 1.0)
    out = torch.zeros((P, W, L), dtype=torch.float64, device=x.device)
    ij = torch.tensor(_pairs(S), device=x.device)
    for l in range(L):
        lag = case["lag1"] + l
        n0, n1 = max(0, -lag), min(N, N - lag)
        b = phi[:, :, n0:n1]
        a = phi[:, :, n0 + lag:n1 + lag]
        for p0 in range(0, P, 128):
            A, B = a[ij[p0:p0 + 128, 1]], b[ij[p0:p0 + 128, 0]]
            s, d = (A + B).abs(), (A - B).abs()
            if case["kind"] == "pcc1":
                out[p0:p0 + 128, :, l] = (s - d).sum(-1) / (2 * (n1 - n0))
            else:
                out[p0:p0 + 128, :, l] = (s ** v - d ** v).sum(-1) / (2 ** (v / 2) * (n1 - n0))
    return _stacked(case, out)


def _bank_sizes(case):
    """Scales of the Morlet bank: s0 2^(m/V), supports 2 ceil(5 s) + 1, the zero-pad length."""
    _, _, N, _, Nz, _ = _sizes(case)
    w0 = math.pi * math.sqrt(2 / math.log(2))
    s0 = case["pmin"] * w0 / (2 * math.pi)
    S = int(math.floor(1 / case["V"] + math.log2(case["pmax"] / case["pmin"]) + 0.5)) * case["V"]
    scale = [s0 * 2 ** (m / case["V"]) for m in range(S)]
    Ls = [min(2 * math.ceil(5 * s) + 1, Nz) for s in scale]
    if Nz - (N + max(abs(case["lag1"]), abs(case["lag2"]))) < Ls[-1]:
        Nz *= 2
    return dict(S=S, scale=scale, Ls=Ls, Nz=Nz, w0=w0)


def _exact_wpcc(case, x):
    S, _, N, L, _, P = _sizes(case)
    f = _bank_sizes(case)
    Nz, dev = f["Nz"], x.device
    W = torch.zeros((f["S"], Nz), dtype=torch.complex128, device=dev)
    for s, (sc, n) in enumerate(zip(f["scale"], f["Ls"])):
        u = torch.arange(n, device=dev) - n // 2
        t = u.double() / sc
        amp = torch.exp(-0.5 * t * t) / math.sqrt(math.sqrt(math.pi) * sc)
        W[s, u % Nz] = torch.polar(amp, f["w0"] * t)
    W = torch.fft.fft(W)
    pad = torch.zeros((S, Nz), dtype=torch.float64, device=dev)
    pad[:, f["Ls"][-1]:f["Ls"][-1] + N] = x[:, 0] / Nz
    X = torch.fft.fft(pad)
    F = torch.empty((S, f["S"], Nz), dtype=torch.complex128, device=dev)
    weight = torch.tensor([math.sqrt(1 / s) for s in f["scale"]], dtype=torch.float64, device=dev)[:, None]
    for s in range(S):
        z = torch.fft.ifft(X[s] * W) * Nz
        m = (z.real ** 2 + z.imag ** 2)
        F[s] = torch.fft.fft(z / torch.sqrt(m + 1e-6 * m.amax(-1, keepdim=True))) * weight
    idx = torch.arange(min(case["lag1"], case["lag2"]), min(case["lag1"], case["lag2"]) + L, device=dev) % Nz
    K0 = sum(1 / s for s in f["scale"])
    out = []
    for i in range(S - 1):
        Y = (F[i].conj() * F[i + 1:]).sum(1)
        out.append(torch.fft.ifft(Y).real[:, idx] / (K0 * N))
    return torch.cat(out)


def exact(case, seed):
    x = _records(case, seed).view(case["S"], case["W"], case["N"]).double()
    if case["kind"] in ("pcc1", "pccv"):
        y = _exact_time(case, x)
    elif case["kind"] == "wpcc":
        y = _exact_wpcc(case, x)
    else:
        y = _exact_spectral(case, x)
    return y[0].cpu().numpy() if case["entry"] == "host" else y
