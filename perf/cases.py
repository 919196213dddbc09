"""Performance cases of the GLS path: what a user's program runs, through the
public entry points, over the range of sizes it runs them at.

``listed()`` names twelve cases, ``draw(rng)`` gives further ones of the same
ranges; ``prepare``/``run`` make and run one, ``work`` counts what a pass cannot
do without and ``exact`` gives its results in 64 bits.

A case is one of these kinds:

``batch``      light curves resident on the device, periodograms left there
               (engine.LombBatch on the NFFT path)
``direct``     the same by direct sums (use_fft=False)
``custom``     the same at explicit, arbitrarily spaced frequencies
``run``        the drop-in class, host arrays in and out:
               LombScargleAsyncProcess().run(...) and finish()
``best``       batched_run_const_nfreq(only_return_best_freqs=True)
``harmonics``  LombScargleAsyncProcess(nharmonics=H).run(...)
``nfft``       adjoint NFFTs with memory allocated once
               (NFFTAsyncProcess.allocate, run(memory=...), finish)
``serve``      a burst of requests through GLSServer, zero-copy results

Its sizes: ``curves`` light curves of ``n_lo`` .. ``n_hi`` points (log-uniform),
on baselines of ``t_lo`` .. ``t_hi`` days (uniform), with ``nf`` frequencies up to
``fmax`` per day each, or, where ``nf`` is 0, 5 frequencies per 1/baseline up to
``fmax``.  ``window`` "es" is the tuned configuration of the batched engine,
"gaussian" the drop-in classes' default (sigma = 4, m = 8); ``mode`` is the
periodogram (floating mean, standard or spectral window).  ``use_double`` has no
case: it widens the same single-precision pipeline's results.
"""
import math

import numpy as np
import torch

from cuvarbase_amd import _lib, tuning
from cuvarbase_amd._device import Stream
from cuvarbase_amd.cunfft import NFFTAsyncProcess
from cuvarbase_amd.engine import LombBatch
from cuvarbase_amd.lombscargle import LombScargleAsyncProcess
from cuvarbase_amd.serve import GLSServer

MODES = {"floating": _lib.MODE_FLOATING_MEAN, "standard": _lib.MODE_STANDARD,
         "window": _lib.MODE_WINDOW}


def _case(name, kind, curves, n_lo, n_hi, t_lo, t_hi, nf, fmax, window="es", mode="floating",
          harmonics=1):
    c = dict(kind=kind, curves=curves, n_lo=n_lo, n_hi=n_hi, t_lo=t_lo, t_hi=t_hi, nf=nf,
             fmax=fmax, window=window, mode=mode, harmonics=harmonics)
    return c if name is None else dict(c, name=name)


def listed():
    return [
        # one light curve from a program that keeps its plan: latency
        _case("one_curve", "batch", 1, 1000, 1000, 10.0, 10.0, 10_000, 50.0),
        # a survey's batch: 50-5,000 points over 30 days to 10 years to 24 /d
        _case("survey", "batch", 1000, 50, 5000, 30.0, 3650.0, 0, 24.0),
        # many sparse curves of one season on one grid
        _case("short_curves", "batch", 2000, 20, 300, 85.0, 90.0, 20_000, 40.0),
        # one very long, finely sampled curve
        _case("long_curve", "batch", 1, 200_000, 200_000, 3650.0, 3650.0, 0, 100.0),
        # the reference's window and oversampling, a ragged handful of curves
        _case("gaussian", "batch", 37, 400, 3000, 200.0, 1500.0, 50_021, 20.0,
              window="gaussian"),
        # exact sums for a few curves, as a check of the fast path or for short grids
        _case("direct", "direct", 10, 300, 2000, 100.0, 1000.0, 10_007, 20.0),
        # refining candidate periods of a few curves on lists of frequencies
        _case("custom", "custom", 4, 500, 3000, 100.0, 2000.0, 4_001, 30.0),
        # the smallest use: one curve through the drop-in class at its defaults
        _case("run_one", "run", 1, 300, 300, 60.0, 60.0, 3_750, 12.5, window="gaussian"),
        # best periods of a field of well-measured variables on one grid
        _case("best_periods", "best", 200, 60, 400, 85.0, 90.0, 20_000, 40.0),
        # two-harmonic model for eclipsing or pulsating shapes
        _case("harmonics", "harmonics", 8, 200, 2000, 100.0, 1000.0, 20_000, 10.0,
              window="gaussian", harmonics=2),
        # plain transforms on memory allocated once
        _case("nfft", "nfft", 6, 1000, 4000, 50.0, 500.0, 30_000, 0.0, window="gaussian"),
        # requests of survey curves arriving together at the server
        _case("served", "serve", 32, 100, 50_000, 30.0, 3650.0, 0, 24.0),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["batch", "batch", "batch", "batch", "direct", "custom", "run", "best",
                       "harmonics", "nfft", "serve"])
    t_lo = rng.uniform(10.0, 1000.0)
    t_hi = t_lo * rng.uniform(1.0, 4.0)
    window, mode, harmonics = rng.choice(["es", "gaussian"]), "floating", 1
    if kind == "batch":
        nf = _log(rng, 500, 1_000_000)
        curves = _log(rng, 1, max(1, min(1000, 50_000_000 // nf)))
        n_lo = _log(rng, 20, max(20, min(50_000, 1_000_000 // curves)))
        mode = rng.choice(["floating", "floating", "standard", "window"])
    elif kind in ("direct", "custom"):
        nf = _log(rng, 500, 100_000 if kind == "direct" else 20_000)
        curves = _log(rng, 1, 40)
        n_lo = _log(rng, 20, max(20, min(5000, 1_000_000_000 // (nf * curves))))
        mode, window = rng.choice(["floating", "standard", "window"]), "es"
    elif kind == "run":
        nf, curves, n_lo = _log(rng, 500, 60_000), _log(rng, 1, 20), _log(rng, 20, 5000)
    elif kind == "best":
        nf, curves, n_lo = _log(rng, 2000, 50_000), _log(rng, 1, 300), _log(rng, 60, 2000)
    elif kind == "harmonics":
        nf, curves, n_lo = _log(rng, 500, 40_000), _log(rng, 1, 20), _log(rng, 50, 4000)
        window, harmonics = "gaussian", rng.choice([2, 2, 3])
    elif kind == "nfft":
        nf, curves, n_lo = _log(rng, 500, 100_000), _log(rng, 1, 12), _log(rng, 50, 20_000)
        window = "gaussian"
    else:
        nf, curves, n_lo = _log(rng, 2000, 200_000), _log(rng, 1, 64), _log(rng, 50, 10_000)
        window = "es"
    n_hi = int(n_lo * rng.uniform(1.0, 3.0))
    # up to a few frequencies per 1/baseline, as an oversampled grid has
    fmax = nf / (t_hi * rng.uniform(3.0, 8.0))
    return _case(None, kind, curves, n_lo, n_hi, t_lo, t_hi, nf, fmax, window, mode, harmonics)


# ---- inputs ---------------------------------------------------------------------
def _sizes(case):
    """Points and baseline of every curve: the case's own, whatever the seed."""
    rng = np.random.default_rng([case["curves"], case["n_lo"], case["n_hi"], case["nf"]])
    n = np.exp(rng.uniform(np.log(case["n_lo"]), np.log(case["n_hi"] + 1), case["curves"]))
    n = np.clip(n.astype(np.int64), case["n_lo"], case["n_hi"])
    return n, rng.uniform(case["t_lo"], case["t_hi"], case["curves"])


def _grid(case, T):
    if not case["nf"]:
        return np.arange(1, int(5.0 * T * case["fmax"])) / (5.0 * T)
    df, first = case["fmax"] / case["nf"], 1
    if case["harmonics"] > 1:
        # several harmonics are searched from 3 cycles over the shortest baseline on
        first = 1 + int(3.0 / (df * case["t_lo"]))
    return df * np.arange(first, first + case["nf"])


def _inputs(case, seed):
    """Light curves [(t, y, dy)] in days and magnitudes and a grid for each:
    nightly observations in seasons of 0.6 of a year (dense curves anywhere in
    time), a sinusoid of random period, heteroscedastic noise."""
    rng = np.random.default_rng([int(seed), case["curves"], case["n_lo"], case["nf"]])
    n, base = _sizes(case)
    data, freqs, shared = [], [], None
    for i in range(case["curves"]):
        T = float(base[i])
        if n[i] < 10 * T:
            nights = rng.integers(0, max(1, int(T)), n[i])
            nights = np.where(nights % 365 < 219, nights, nights - 146)
            t = np.sort(nights + rng.uniform(-0.15, 0.15, n[i]))
        else:
            t = np.sort(rng.uniform(0.0, T, n[i]))
        amp, s = rng.uniform(0.05, 1.0), rng.uniform(0.01, 0.5)
        if case["kind"] == "best":     # well-measured variables
            amp, s = rng.uniform(0.5, 1.0), rng.uniform(0.01, 0.1)
        if shared is None or not case["nf"]:
            shared = _grid(case, T) if case["kind"] != "nfft" else None
        f_true = np.exp(rng.uniform(np.log(0.02), np.log(0.9))) * \
            (shared[-1] if shared is not None else 10.0)
        dy = s * rng.uniform(0.7, 1.4, n[i])
        y = 15.0 + amp * np.sin(2 * np.pi * (f_true * t + rng.uniform())) + \
            dy * rng.standard_normal(n[i])
        data.append((t, y, dy))
        freqs.append(shared)
    if case["kind"] == "custom":
        # trial frequencies anywhere up to fmax, in no order
        freqs = [rng.uniform(0.01, 1.0, case["nf"]) * case["fmax"] for _ in data]
    return data, freqs


def _config(case):
    if case["window"] == "es":
        c = tuning.choose_nfft_config(1e-4)
        return dict(sigma=c["sigma"], m=c["m"], window=c["window"], window_beta=c["window_beta"])
    return dict(sigma=4.0, m=8)


class _DeviceView:
    """The engine's device array as a tensor sees it."""

    def __init__(self, arr, count):
        self.owner = arr
        self.__cuda_array_interface__ = dict(shape=(int(count),), typestr=arr.dtype.str,
                                             data=(arr.ptr, False), version=2)


def prepare(case, seed):
    kind = case["kind"]
    data, freqs = _inputs(case, seed)
    st = {"kind": kind, "data": data, "freqs": freqs}
    if kind in ("batch", "direct", "custom"):
        cfg = _config(case) if kind == "batch" else {}
        b = LombBatch(data, freqs, mode=MODES[case["mode"]], use_fft=kind == "batch",
                      custom_freqs=kind == "custom", **cfg)
        st["stream"] = Stream()
        b.upload(stream=st["stream"])
        st["stream"].synchronize()
        st["batch"] = b
        st["power"] = torch.as_tensor(_DeviceView(b.d_power, b.total_out), device="cuda")
    elif kind == "serve":
        st["server"] = GLSServer(hbm_budget=4e9, zero_copy=True, result_buffer_bytes=256 << 20)
        st["held"] = []
    elif kind == "nfft":
        proc = NFFTAsyncProcess()
        items = [(t, y - np.mean(y), case["nf"]) for t, y, _ in data]
        st.update(proc=proc, items=items, memory=proc.allocate(items))
    else:
        cfg = dict(nharmonics=case["harmonics"])
        if case["window"] == "es":
            c = _config(case)
            cfg.update(sigma=c["sigma"], m=c["m"], nfft_window="es",
                       window_beta=c["window_beta"])
        st["proc"] = LombScargleAsyncProcess(**cfg)
    return st


def run(st):
    kind, data, freqs = st["kind"], st["data"], st["freqs"]
    if kind in ("batch", "direct", "custom"):
        st["batch"].execute(stream=st["stream"])
        return st["power"]
    if kind == "serve":
        srv = st["server"]
        for r in st["held"]:
            r.release()
        srv.completed.clear()
        st["held"] = [srv.submit(t, y, dy, f) for (t, y, dy), f in zip(data, freqs)]
        srv.drain()
        return [r.power for r in st["held"]]
    proc = st["proc"]
    if kind == "best":
        best, significance = proc.batched_run_const_nfreq(
            data, batch_size=100, freqs=freqs[0], only_return_best_freqs=True)
        return {"freq": np.array(best), "significance": np.array(significance)}
    if kind == "nfft":
        out = proc.run(st["items"], memory=st["memory"])
        proc.finish()
        return out
    out = proc.run(data, freqs=freqs)
    proc.finish()
    return [p for _, p in out]


# ---- what a pass cannot do without -------------------------------------------------
def work(case):
    """Bytes: the inputs (and explicit frequencies) once, the results once.
    Operations: by direct sums, 24 per point and frequency (three complex sums
    by rotation) or 40 where each phase is evaluated by itself; by the NFFT,
    2m + 1 taps of 4 per point and transform, 5 n log2 n per transform of
    n = sigma nf cells and 40 per power."""
    kind, C = case["kind"], case["curves"]
    n, base = _sizes(case)
    nf = np.full(C, case["nf"]) if case["nf"] else (5.0 * base * case["fmax"]).astype(np.int64) - 1
    pts, out = float(n.sum()), float(nf.sum())
    if kind in ("direct", "custom"):
        per = 24.0 if kind == "direct" else 40.0
        return {"bytes": 24.0 * pts + (4.0 if kind == "direct" else 12.0) * out,
                "flops": per * float((n * nf).sum())}
    sigma, m = (1.35, 5) if case["window"] == "es" else (4.0, 8)
    transforms = {"nfft": 1, "harmonics": 3 * case["harmonics"]}.get(kind, 3)
    cells = sigma * nf
    flops = transforms * (4.0 * (2 * m + 1) * pts + float((5.0 * cells * np.log2(cells)).sum()))
    res = {"nfft": 8.0 * out, "best": 16.0 * C}.get(kind, 4.0 * out)
    return {"bytes": (16.0 if kind == "nfft" else 24.0) * pts + res,
            "flops": flops + (0.0 if kind == "nfft" else 40.0 * out)}


# ---- the same results in 64 bits ----------------------------------------------------
def _turns(x):
    x = 2 * math.pi * (x - torch.round(x))
    return torch.complex(torch.cos(x), torch.sin(x))


def _linear_sums(t, vals, f0, df, nf, mult):
    """sum_j v_j exp(2 pi i mult (f0 + k df) t_j), k < nf, for each v: the phase
    split as k = a B + b, a matrix product over the points."""
    B = max(1, int(math.sqrt(nf)))
    A = -(-nf // B)
    out = [torch.zeros(A, B, dtype=torch.complex128, device=t.device) for _ in vals]
    ka = torch.arange(A, dtype=torch.float64, device=t.device) * B
    kb = torch.arange(B, dtype=torch.float64, device=t.device)
    for lo in range(0, len(t), 8192):
        tt = mult * t[lo:lo + 8192]
        e1 = _turns((f0 + ka[:, None] * df) * tt[None, :])
        e2 = _turns((kb[None, :] * df) * tt[:, None])
        for o, v in zip(out, vals):
            o += torch.matmul(e1 * v[None, lo:lo + 8192], e2)
    return [o.reshape(-1)[:nf] for o in out]


def _listed_sums(t, vals, f, mult):
    out = [torch.zeros(len(f), dtype=torch.complex128, device=t.device) for _ in vals]
    for lo in range(0, len(t), 512):
        e = _turns((mult * f[:, None]) * t[None, lo:lo + 512])
        for o, v in zip(out, vals):
            o += torch.matmul(e, v[lo:lo + 512].to(torch.complex128))
    return out


def _gls(yw_f, w_f, w_2f, yy, ybar, mode):
    C, S, C2, S2 = w_f.real, w_f.imag, w_2f.real, w_2f.imag
    cc, ss, cs = 0.5 * (1 + C2), 0.5 * (1 - C2), 0.5 * S2
    bc, bs, den = yw_f.real, yw_f.imag, yy
    if mode == "floating":
        cc, ss, cs = cc - C * C, ss - S * S, cs - C * S
    elif mode == "standard":
        bc, bs, den = bc + ybar * C, bs + ybar * S, yy + ybar * ybar
    else:
        bc, bs, den = 2 * C, 2 * S, 1.0
    return (ss * bc * bc + cc * bs * bs - 2 * cs * bc * bs) / (den * (cc * ss - cs * cs))


def _harmonic_gls(sums, w, H, yy):
    """Floating-mean model of H harmonics, the normal equations per frequency."""
    wz = {0: torch.full_like(w[1].real, sums["sum_w"])}
    c = {h: w[h].real for h in w} | wz
    s = {h: w[h].imag for h in w} | {0: torch.zeros_like(w[1].real)}
    K = len(c[0])
    M = torch.zeros(K, 2 * H, 2 * H, dtype=torch.float64)
    b = torch.zeros(K, 2 * H, dtype=torch.float64)
    for i in range(1, H + 1):
        b[:, i - 1] = (sums["yw"][i].real - sums["ybar"] * c[i]).cpu()
        b[:, H + i - 1] = (sums["yw"][i].imag - sums["ybar"] * s[i]).cpu()
        for j in range(1, H + 1):
            d, sg = abs(i - j), 1.0 if i >= j else -1.0
            M[:, i - 1, j - 1] = (0.5 * (c[i + j] + c[d]) - c[i] * c[j]).cpu()
            M[:, H + i - 1, H + j - 1] = (0.5 * (c[d] - c[i + j]) - s[i] * s[j]).cpu()
            x = (0.5 * (s[i + j] - sg * s[d]) - c[i] * s[j]).cpu()
            M[:, i - 1, H + j - 1] = x
            M[:, H + j - 1, i - 1] = x
    theta = torch.from_numpy(np.linalg.solve(M.numpy(), b.numpy()[..., None])[..., 0])
    return (theta * b).sum(1) / yy


def _significance(t, dy, z, fmax):
    """1 - false-alarm probability of a peak (Baluev 2008, as the reference writes it)."""
    N = len(t)
    w = dy ** -2.0
    tbar = np.dot(w, t) / w.sum()
    teff = math.sqrt(4 * math.pi * np.dot(w, (t - tbar) ** 2) / w.sum())
    g = math.exp(math.lgamma(0.5 * (N - 1)) - math.lgamma(0.5 * (N - 2)))
    tau = g * math.sqrt(math.pi) * fmax * teff * math.sqrt(z / math.pi) * \
        max(0.0, 1 - z) ** (0.5 * (N - 4))
    return (1 - max(0.0, 1 - z) ** (0.5 * (N - 3))) * math.exp(-tau)


def exact(case, seed):
    kind, H = case["kind"], case["harmonics"]
    data, freqs = _inputs(case, seed)
    dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")

    def up(x):
        return torch.as_tensor(np.asarray(x, np.float64), device=dev)

    out = []
    for (t, y, dy), f in zip(data, freqs):
        if kind == "nfft":
            df = 1.0 / (np.max(t) - np.min(t))
            z = _linear_sums(up(t), [up(y - np.mean(y))], 0.0, df, case["nf"], 1.0)[0]
            out.append(z.cpu().numpy())
            continue
        w = dy ** -2.0 / np.sum(dy ** -2.0)
        y = y - np.mean(y)
        ybar = float(np.dot(w, y))
        yw, yy = w * (y - ybar), float(np.dot(w, (y - ybar) ** 2))
        tt, W, YW = up(t - np.min(t)), up(w), up(yw)
        if kind == "custom":
            a = _listed_sums(tt, [YW, W], up(f), 1.0)
            out.append(_gls(a[0], a[1], _listed_sums(tt, [W], up(f), 2.0)[0], yy, ybar,
                            case["mode"]))
            continue
        grid = (float(f[0]), float(f[1] - f[0]), len(f))
        first = _linear_sums(tt, [YW, W], *grid, 1.0)
        ws = {1: first[1]}
        for h in range(2, 2 * H + 1):
            ws[h] = _linear_sums(tt, [W], *grid, float(h))[0]
        if H > 1:
            yws = {1: first[0]}
            for h in range(2, H + 1):
                yws[h] = _linear_sums(tt, [YW], *grid, float(h))[0]
            sums = {"yw": yws, "sum_w": float(w.sum()), "ybar": float(yw.sum())}
            out.append(_harmonic_gls(sums, ws, H, yy).numpy())
            continue
        P = _gls(first[0], ws[1], ws[2], yy, ybar, case["mode"])
        if kind == "best":
            k = int(torch.argmax(P))
            out.append((f[k], _significance(t - np.mean(t), dy, float(P[k]), float(np.max(f)))))
        else:
            out.append(P)
    if kind == "best":
        return {"freq": np.array([o[0] for o in out]),
                "significance": np.array([o[1] for o in out])}
    if kind in ("batch", "direct", "custom"):
        return torch.cat(out)
    return [o.cpu().numpy() if isinstance(o, torch.Tensor) else o for o in out]
