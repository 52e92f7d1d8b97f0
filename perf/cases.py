"""What a user of the framework has it do, as cases that can be timed and compared.

listed() gives the cases, draw(rng) more of the same ranges.  prepare(case, seed) makes what a
user's program holds before the call (detectors with their data, parameter rows, time series),
run(state) is one pass through the public entry points, work(case) what that pass cannot do
without, exact(case, seed) its result in 64 bits from plain torch where the inputs are plain
arrays.  The likelihoods have no value there: their waveform model (calibrated coefficients, Kerr
ringdown table) exists in the package alone.  They are timed in FP64, the precision every entry
point takes by default.

Kinds of case ("do"):
  lnl        batched log-likelihood, with or without the gradient over the 11 parameters
             (WhittleLikelihoodHip); one row goes through the scalar log_likelihood(dict) of the
             bilby-style interface
  response   links and TDI channels of one source from the device waveform model
             (InterferometerAntenna.update_detector_response, what inject_signal calls)
  container  the same from a waveform container that the program supplies
  td         time-domain links and TDI of a sampled waveform
  whittle    the standalone Whittle sum of data, response and PSD arrays
"""

import math

import numpy as np
import torch

YEAR = 31557600.0
SHORT = 655360.0  # 2^17 samples at 5 s: the short data set of the tests and the examples
C_SI, AU_SI, DAY = 299792458.0, 149597870700.0, 86400.0
HM = "22,21,33,32,44,43"
# name: (PSD model, minimum and maximum frequency, arm length, orbit kind, initial revolution)
DETECTORS = {"LISA": ("LISA_SciRDv1", 1e-4, 0.05, 2.5e9, 0, -math.pi / 9),
             "Taiji": ("Taiji_TDC", 1e-4, 0.06, 3.0e9, 0, math.pi / 9),
             "TianQin": ("Tianqin_GWSpace", 1e-3, 0.039, 1.7e8, 1, 0.0)}
ORBITS = {"LISA": "LISA_analytic", "Taiji": "Taiji_analytic", "TianQin": "Tianqin_analytic"}
NETWORK = "LISA,Taiji,TianQin"
# the canonical massive binary of the tests and the benchmark; t_c at 0.8 of the data's length
SOURCE = {"chirp_mass": 1.2e6, "mass_ratio": 0.6, "chi_1": 0.75, "chi_2": 0.62, "luminosity_distance": 56000.0,
          "reference_phase": 1.3, "inclination": 0.4, "ecliptic_longitude": 1.375, "ecliptic_latitude": -1.2108,
          "polarization": 2.659}
SKY = (1.375, -1.2108, 2.659)


def _lnl(name, detectors, modes, duration, rows, grad, cloud="local", tdi="1.5", channels="AET", duty=False,
         grid="rfft"):
    return {"name": name, "do": "lnl", "detectors": detectors, "modes": modes, "duration": duration, "rows": rows,
            "grad": grad, "cloud": cloud, "tdi": tdi, "channels": channels, "duty": duty, "grid": grid}


def listed():
    return [
        # a sampler that asks for one point at a time (bilby): the smallest call, all latency
        _lnl("one_point", "LISA", "22", SHORT, 1, False),
        # a handful of gradient chains (HMC) with the higher modes on the short data
        _lnl("chains_grad", "LISA", HM, SHORT, 16, True),
        # one round of a particle sampler on the short data, the reference's own configuration
        _lnl("particles_short", "LISA", "22", SHORT, 4096, False),
        # the quadrupole on a year of LISA data, a batch of particles
        _lnl("lisa_year", "LISA", "22", YEAR, 512, False),
        # the benchmark network (ragged grids, TianQin on duty three months in six), gradient
        _lnl("network_grad", NETWORK, HM, YEAR, 1024, True, duty=True),
        # the same without the gradient: a mutation round of the SMC sampler
        _lnl("network_lnl", NETWORK, HM, YEAR, 2048, False, duty=True),
        # rows anywhere in the prior (total mass 1e5 - 1e7, t_c in the year), an uneven batch
        _lnl("prior_grad", NETWORK, HM, YEAR, 257, True, cloud="prior", duty=True),
        # PhenomD evaluated at every one of 2^14 log-spaced bins (no interpolation), gradient
        _lnl("log_grid_grad", "LISA", "22", SHORT, 2048, True, grid="log"),
        # one source injected into a year of data: links and channels with the higher modes
        {"name": "response_year", "do": "response", "detector": "LISA", "modes": HM, "duration": YEAR, "tdi": "1.5",
         "orthogonal": True},
        # a waveform made elsewhere, six modes, through the response of a rotating geocentric orbit
        {"name": "container", "do": "container", "detector": "TianQin", "modes": 6, "duration": 0.25 * YEAR,
         "tdi": "2.0", "orthogonal": False},
        # a year of time-domain links and TDI at 5 s
        {"name": "td_year", "do": "td", "detector": "LISA", "duration": YEAR, "dt": 5.0, "tdi": "1.5",
         "orthogonal": True},
        # the Whittle sum of arrays that the program holds, a year of three channels
        {"name": "whittle_year", "do": "whittle", "channels": 3, "bins": 1574725},
    ]


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _bins(case):
    """Bins of each detector of a frequency-domain case (rfft grid of the duration at 5 s)."""
    names = case["detectors"].split(",") if "detectors" in case else [case["detector"]]
    if case.get("grid") == "log":
        return [2 ** 14 for _ in names]
    return [int((DETECTORS[n][2] - DETECTORS[n][1]) * case["duration"]) for n in names]


def draw(rng):
    do = rng.choice(["lnl"] * 6 + ["response", "container", "td", "whittle"])
    tdi, orth = rng.choice(["1.5", "2.0"]), rng.random() < 0.7
    if do == "lnl":
        grid = rng.choice(["rfft"] * 4 + ["log"])
        case = _lnl("", rng.choice(["LISA", "Taiji", "TianQin", "LISA,TianQin", NETWORK]) if grid == "rfft" else "LISA",
                    rng.choice(["22", "22,33,44", HM] if grid == "rfft" else ["22", "22,33,44"]),
                    round(_log_uniform(rng, SHORT, YEAR)), 1, rng.random() < 0.5,
                    rng.choice(["local", "local", "prior"]), tdi, rng.choice(["AET", "AE"]), rng.random() < 0.5, grid)
        del case["name"]
        # (bin, mode, row) triples at most a third of the largest listed case's, rows over 1 - 4096
        per_row = sum(_bins(case)) * len(case["modes"].split(",")) * (3 if case["grad"] else 1)
        case["rows"] = round(_log_uniform(rng, 1, min(4096.0 if grid == "rfft" else 2048.0, 2e10 / per_row)))
        return case
    if do == "response":
        return {"do": do, "detector": rng.choice(list(DETECTORS)), "modes": rng.choice(["22", "22,33,44", HM]),
                "duration": round(_log_uniform(rng, SHORT, YEAR)), "tdi": tdi, "orthogonal": orth}
    if do == "container":
        return {"do": do, "detector": rng.choice(list(DETECTORS)), "modes": rng.choice([1, 2, 3, 6]),
                "duration": round(_log_uniform(rng, SHORT, 0.5 * YEAR)), "tdi": tdi, "orthogonal": orth}
    if do == "td":
        dt = rng.choice([5.0, 5.0, 2.0, 10.0])
        return {"do": do, "detector": rng.choice(list(DETECTORS)), "tdi": tdi, "orthogonal": orth, "dt": dt,
                "duration": round(_log_uniform(rng, 1e5, YEAR * min(1.0, dt / 5.0)))}
    return {"do": do, "channels": rng.choice([1, 2, 3]), "bins": round(_log_uniform(rng, 1e3, 1.9e6))}


# ---- inputs -----------------------------------------------------------------------------------
def _antenna(name, case, labels, response=None, combination=None, duty=None, td=False):
    from pespace_amd.detector.antenna import FDResponseModelMarset2018, InterferometerAntenna
    from pespace_amd.detector.tdi import FDMichelsonConstantEqualArm, TDIChannelData
    _, lo, hi, *_ = DETECTORS[name]
    data = TDIChannelData(backend="hip")
    if td:
        data.set_td_data_from_zero(labels, case["duration"], case["dt"])
    elif case.get("grid") == "log":
        f = np.geomspace(lo, hi, 2 ** 14)
        data.set_fd_data_on_grid(labels, f, np.gradient(f))
    else:
        data.set_fd_data_from_zero(labels, case["duration"], 5.0, 0.0, lo, hi)
    return InterferometerAntenna(name, data, ORBITS[name], response or FDResponseModelMarset2018(),
                                 combination or FDMichelsonConstantEqualArm(case["tdi"], labels[0] == "A"),
                                 duty_cycle=duty)


def _rows(case, seed):
    """Parameter rows: a Gaussian of relative width 1e-3 around the source, or the wide prior."""
    rng = np.random.default_rng([seed, 1])
    n, span = case["rows"], case["duration"]
    if case["cloud"] == "prior":
        q = rng.uniform(1.0, 8.0, n)
        mass = 10.0 ** rng.uniform(5.0, 7.0, n)
        cols = [mass * (q / (1.0 + q) ** 2) ** 0.6, 1.0 / q, rng.uniform(-0.9, 0.9, n), rng.uniform(-0.9, 0.9, n),
                rng.uniform(5000.0, 50000.0, n), rng.uniform(0.0, 2 * np.pi, n), np.arccos(rng.uniform(-1, 1, n)),
                rng.uniform(0.0, 2 * np.pi, n), np.arcsin(rng.uniform(-1, 1, n)), rng.uniform(0.0, np.pi, n),
                rng.uniform(0.0, span, n)]
        return np.column_stack(cols)
    center = np.array([*SOURCE.values(), 0.8 * span])
    return center * (1.0 + 1e-3 * np.clip(rng.standard_normal((n, center.size)), -4.0, 4.0))


def _prepare_lnl(case, seed):
    from pespace_amd.inference.likelihood import LikelihoodBilbyInterfaceHip, WhittleLikelihoodHip
    from pespace_amd.waveform.phenom import IMRPhenomHM
    names, modes = case["detectors"].split(","), tuple(case["modes"].split(","))
    span, log = case["duration"], case["grid"] == "log"
    lo, hi = min(DETECTORS[n][1] for n in names), max(DETECTORS[n][2] for n in names)
    gen = torch.Generator(device="cuda").manual_seed(seed)
    source = dict(SOURCE, coalescence_time=0.8 * span)
    detectors, waveform = [], None
    for name in names:
        duty = (YEAR / 2, YEAR / 4, YEAR / 8, 86400.0) if case["duty"] and name == "TianQin" else None
        det = _antenna(name, case, ("A", "E", "T"), duty=duty)
        td = det.tdi_data
        td.set_fd_noise_power_density_from_model(DETECTORS[name][0], tdi_generation=case["tdi"])
        if waveform is None:
            waveform = IMRPhenomHM(td.frequency_samples, 0.0, modes=modes, n_nodes=0 if log else 1024, f_node_min=lo,
                                   f_node_max=hi)
            waveform.update_waveform(source)
        # the data: the source's response plus noise of the model's PSD
        det.update_detector_response(waveform.waveform_container, *SKY, source["coalescence_time"])
        noise = torch.randn(3, td.frequency_samples.size, dtype=torch.complex128, device="cuda", generator=gen)
        width = torch.as_tensor(np.sqrt(0.5 / np.asarray(td.frequency_weights())), device="cuda")
        psd = torch.as_tensor(np.stack(td.fd_noise_power_density), device="cuda")
        noise *= width * psd.sqrt()
        channels = torch.stack(list(det.tdi_response)) + noise
        td.fd_data = type(td.fd_data)(*channels.cpu().numpy())
        detectors.append(det)
    rows = _rows(case, seed)
    if case["rows"] == 1:
        like = LikelihoodBilbyInterfaceHip(waveform, tuple(detectors), tuple(case["channels"]))
        core = like._lk.core
        point = {k: float(v) for k, v in zip([*SOURCE, "coalescence_time"], rows[0])}
    else:
        like = WhittleLikelihoodHip(waveform, tuple(detectors), tuple(case["channels"]))
        core = like.core
        point = None
    core.n_bins  # uploads the detectors' data
    for det in detectors:  # the injection's own contexts are done with
        det._core = None
    return {"like": like, "rows": torch.as_tensor(rows, device="cuda"), "point": point}


def _prepare_response(case, seed):
    from pespace_amd.waveform.phenom import IMRPhenomHM
    det = _antenna(case["detector"], case, ("A", "E", "T") if case["orthogonal"] else ("X", "Y", "Z"))
    rng = np.random.default_rng(seed)
    _, lo, hi, *_ = DETECTORS[case["detector"]]
    waveform = IMRPhenomHM(det.tdi_data.frequency_samples, 0.0, modes=tuple(case["modes"].split(",")), n_nodes=1024,
                           f_node_min=lo, f_node_max=hi)
    waveform.update_waveform(dict(SOURCE, chirp_mass=1.2e6 * rng.uniform(0.8, 1.25), mass_ratio=rng.uniform(0.3, 1.0)))
    return {"det": det, "waveform": waveform.waveform_container,
            "where": (rng.uniform(0, 2 * np.pi), rng.uniform(-1.2, 1.2), rng.uniform(0, np.pi), 0.8 * case["duration"])}


def _container_inputs(case, seed, f):
    """Six modes of an inspiral-like signal: power-law amplitude, chirp phase and its t(f)."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    out = {}
    for m in range(case["modes"]):
        r = torch.rand(5, dtype=torch.float64, device="cuda", generator=gen)
        amp = 1e-19 * (0.1 + r[0]) * f ** (-7.0 / 6.0)
        scale = 2e-3 * (1.0 + 2.0 * r[1])
        h = torch.polar(amp, -(scale * f ** (-5.0 / 3.0) + 6.0 * r[2]))
        tf = -(5.0 / 3.0) * scale * f ** (-8.0 / 3.0) / (2.0 * math.pi)
        out[str(m)] = {"plus": h, "cross": h * torch.complex(0.2 * r[3], r[4] - 0.5), "tf": tf}
    return out


def _container_grid(case):
    _, lo, hi, *_ = DETECTORS[case["detector"]]
    n = int(case["duration"] // 5.0 + 1)
    f = np.fft.rfftfreq(n, 5.0)
    return torch.as_tensor(f[(f >= lo) & (f <= hi)], device="cuda")


def _prepare_container(case, seed):
    det = _antenna(case["detector"], case, ("A", "E", "T") if case["orthogonal"] else ("X", "Y", "Z"))
    f = torch.as_tensor(det.tdi_data.frequency_samples, device="cuda")
    return {"det": det, "waveform": _container_inputs(case, seed, f), "where": (*SKY, 0.8 * case["duration"])}


def _td_inputs(case, seed):
    """A tapered chirp that covers most of the data, (n, 2) samples of h+, hx, and its first time."""
    r = np.random.default_rng(seed).uniform(0.0, 1.0, 4)
    n = int(0.9 * case["duration"] / case["dt"])
    t = case["dt"] * torch.arange(n, dtype=torch.float64, device="cuda")
    f0 = 5e-4 * (1.0 + r[0])
    phase = 2 * math.pi * (f0 * t + 0.5 * (0.5 * f0 / (n * case["dt"])) * t * t)
    amp = 1e-21 * torch.sin(math.pi * t / t[-1]) ** 2
    data = torch.stack([amp * torch.cos(phase), (0.2 + r[1]) * amp * torch.sin(phase + r[2])], dim=1)
    return data.contiguous(), case["duration"] * 0.08 * r[3]


def _prepare_td(case, seed):
    from pespace_amd.detector.antenna import TDResponseModelCornish2003
    from pespace_amd.detector.tdi import TDMichelsonConstantEqualArm
    comb = TDMichelsonConstantEqualArm(case["tdi"], case["orthogonal"])
    det = _antenna(case["detector"], case, comb.labels, TDResponseModelCornish2003(), comb, td=True)
    data, start = _td_inputs(case, seed)
    return {"det": det, "waveform": {"t0": start, "data": data}, "where": (*SKY, 0.0)}


def _prepare_whittle(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    shape = (case["channels"], case["bins"])
    f = torch.linspace(1e-4, 0.05, case["bins"], dtype=torch.float64, device="cuda")
    psd = 1e-40 * (1.0 + (1e-3 / f) ** 2 + (f / 1e-2) ** 2).expand(shape).contiguous()
    noise = torch.randn(*shape, dtype=torch.complex128, device="cuda", generator=gen) * (psd / YEAR * 1e15).sqrt()
    signal = noise[:, :1].abs() * (1e-3 / f) ** 1.2 * torch.polar(torch.ones_like(f), -2e-3 * f ** (-5.0 / 3.0))
    return {"data": signal + noise, "response": signal.contiguous(), "psd": psd, "df": 1.0 / YEAR}


def prepare(case, seed):
    return dict({"lnl": _prepare_lnl, "response": _prepare_response, "container": _prepare_container,
                 "td": _prepare_td, "whittle": _prepare_whittle}[case["do"]](case, seed), case=case)


# ---- one pass ---------------------------------------------------------------------------------
def run(state):
    case = state["case"]
    if case["do"] == "lnl":
        like = state["like"]
        if case["rows"] == 1 and not case["grad"]:
            return like.log_likelihood(state["point"])
        like = like._lk if case["rows"] == 1 else like
        if case["grad"]:
            return like.log_likelihood_and_grad(state["rows"])
        return like.log_likelihood_batch(state["rows"])
    if case["do"] == "whittle":
        from pespace_amd.inference.likelihood import noise_weighted_inner_product
        return noise_weighted_inner_product(state["data"], state["response"], state["psd"], state["df"])
    det = state["det"]
    det.update_detector_response(state["waveform"], *state["where"])
    return {"links": det.single_link_response, "tdi": tuple(det.tdi_response)}


# ---- what a pass cannot do without ------------------------------------------------------------
def work(case):
    """Bytes: inputs read once, outputs written once.  Flops: the per-(bin, mode, row) arithmetic
    of the stationary-phase response (a phase, three transfer functions and their products: about
    150, twice that again for the adjoint) over the band that a source of 1e6 solar masses
    reaches; a few per sample for the streaming kinds."""
    do = case["do"]
    if do == "whittle":
        n = case["channels"] * case["bins"]
        return {"bytes": 40.0 * n + 8, "flops": 8.0 * n}
    if do == "td":
        n = case["duration"] / case["dt"]
        return {"bytes": n * (16 * 0.9 + 2 * 48 + 24), "flops": n * 250.0}
    n = float(sum(_bins(case)))
    if do == "response":
        return {"bytes": n * (20 + 2 * 96 + 48), "flops": n * len(case["modes"].split(",")) * 150.0}
    if do == "container":
        return {"bytes": n * (8 + 40 * case["modes"] + 2 * 96 + 48), "flops": n * case["modes"] * 150.0}
    rows, modes = case["rows"], len(case["modes"].split(","))
    per_bin = 100.0 if case["grid"] == "rfft" else 108.0
    band = 0.4 if case["grid"] == "rfft" else 0.9
    return {"bytes": n * per_bin + rows * 8 * (12 + (11 if case["grad"] else 0)),
            "flops": n * band * modes * rows * (450.0 if case["grad"] else 150.0)}


# ---- 64-bit results from plain torch ----------------------------------------------------------
def _basis(lam, beta, psi):
    sl, cl, sb, cb, sp, cp = (f(x) for x in (lam, beta, psi) for f in (math.sin, math.cos))
    p = (sl * cp - cl * sb * sp, -cl * cp - sl * sb * sp, cb * sp)
    q = (-sl * sp - cl * sb * cp, cl * sp - sl * sb * cp, cb * cp)
    return p, q, (-cb * cl, -cb * sl, -sb)


def _nodes(name, t):
    """The three nodes' positions (seconds, barycentric), each a list of x, y, z."""
    _, _, _, arm, kind, rev0 = DETECTORS[name]
    L = arm / C_SI
    alpha = 2 * math.pi / YEAR * t + rev0
    sa, ca = torch.sin(alpha), torch.cos(alpha)
    au = AU_SI / C_SI
    out = []
    for i in range(3):
        k = 2 * math.pi * i / 3
        if kind == 0:
            r, sk, ck = L / (2 * math.sqrt(3.0)), math.sin(k), math.cos(k)
            d = [r * (sa * ca * sk - (1 + sa * sa) * ck), r * (sa * ca * ck - (1 + ca * ca) * sk),
                 -math.sqrt(3.0) * r * (ca * ck + sa * sk)]
        else:
            rot = 2 * math.pi / (3.65 * DAY) * t + k
            sk, ck, r = torch.sin(rot), torch.cos(rot), L / math.sqrt(3.0)
            lr, br = 120.5 / 180 * math.pi, -4.7 / 180 * math.pi
            d = [r * (math.sin(br) * math.cos(lr) * sk + math.sin(lr) * ck),
                 r * (math.sin(br) * math.sin(lr) * sk - math.cos(lr) * ck), -r * math.cos(br) * sk]
        out.append([d[0] + au * ca, d[1] + au * sa, d[2]])
    return out


def _dot(a, b):
    return a[0] * b[0] + a[1] * b[1] + a[2] * b[2]


# links in the order 12, 21, 23, 32, 31, 13: (receiver, sender)
_LINKS = ((0, 1), (1, 0), (1, 2), (2, 1), (2, 0), (0, 2))


def _orthogonal(x, y, z):
    return [(z - x) / math.sqrt(2.0), (x - 2 * y + z) / math.sqrt(6.0), (x + y + z) / math.sqrt(3.0)]


def _exact_container(case, seed):
    f = _container_grid(case)
    arm = DETECTORS[case["detector"]][3]
    L = arm / C_SI
    p, q, k = _basis(*SKY)
    tc = 0.8 * case["duration"]
    shift = torch.polar(torch.ones_like(f), -2 * math.pi * f * tc)
    links = [0.0] * 6
    for w in _container_inputs(case, seed, f).values():
        x = _nodes(case["detector"], w["tf"] + tc)
        hp, hc = w["plus"] * shift, w["cross"] * shift
        for i, (r, s) in enumerate(_LINKS):
            n = [(x[r][a] - x[s][a]) / L for a in range(3)]  # along the light's path, s to r
            np_, nq, kn = _dot(n, p), _dot(n, q), _dot(n, k)
            h = (np_ ** 2 - nq ** 2) * hp + 2 * np_ * nq * hc
            xl = math.pi * f * L
            sinc = torch.sinc(xl * (1 - kn) / math.pi)
            phase = -math.pi * f * (L + _dot(k, x[r]) + _dot(k, x[s]))
            links[i] = links[i] - 1j * xl * sinc * h * torch.polar(torch.ones_like(f), phase)
    D = torch.polar(torch.ones_like(f), -2 * math.pi * f * L)
    pf = 1 - D ** 2 if case["tdi"] == "1.5" else (1 - D ** 2) * (1 - D ** 4)
    l12, l21, l23, l32, l31, l13 = links
    x = pf * (l13 - l12 + D * (l31 - l21))
    y = pf * (l21 - l23 + D * (l12 - l32))
    z = pf * (l32 - l31 + D * (l23 - l13))
    return {"links": torch.stack(links), "tdi": tuple(_orthogonal(x, y, z) if case["orthogonal"] else (x, y, z))}


def _exact_td(case, seed):
    dt, L = case["dt"], DETECTORS[case["detector"]][3] / C_SI
    data, start = _td_inputs(case, seed)
    n_out = int(case["duration"] // dt + 1)
    delays = 3 if case["tdi"] == "1.5" else 7
    added = int(delays * L // dt + 1)
    t = dt * (torch.arange(n_out + added, dtype=torch.float64, device="cuda") - added)
    p, q, k = _basis(*SKY)
    x = _nodes(case["detector"], t)
    last = data.shape[0] - 1

    def h(when):
        pos = (when - start) / dt
        i = pos.floor().clamp(0, last - 1).long()
        v = data[i] + (data[i + 1] - data[i]) * (pos - i)[:, None]
        return torch.where(((pos >= 0) & (pos <= last))[:, None], v, 0.0)

    links = []
    for r, s in _LINKS:
        n = [(x[r][a] - x[s][a]) / L for a in range(3)]
        np_, nq, kn = _dot(n, p), _dot(n, q), _dot(n, k)
        v = h(t - L - _dot(k, x[s])) - h(t - _dot(k, x[r]))
        links.append(((np_ ** 2 - nq ** 2) * v[:, 0] + 2 * np_ * nq * v[:, 1]) / (2 * (1 - kn)))

    def delayed(y, m):
        c = added - m * (L / dt)
        j = min(max(math.floor(c), 0), added - 1) if m else added
        if not m:
            return y[j:j + n_out]
        return y[j:j + n_out] + (y[j + 1:j + 1 + n_out] - y[j:j + n_out]) * (c - j)

    def channel(a, b, c, e):
        out = 0.0
        for m, sign in ((0, 1), (2, -1)) if case["tdi"] == "1.5" else ((0, 1), (2, -1), (4, -1), (6, 1)):
            out = out + sign * (delayed(links[a], m) - delayed(links[b], m)
                                + delayed(links[c], m + 1) - delayed(links[e], m + 1))
        return out

    xyz = channel(5, 0, 4, 1), channel(1, 2, 0, 3), channel(3, 4, 2, 5)
    return {"links": torch.stack(links), "tdi": tuple(_orthogonal(*xyz) if case["orthogonal"] else xyz)}


def exact(case, seed):
    if case["do"] == "whittle":
        s = _prepare_whittle(case, seed)
        r = s["data"] - s["response"]
        return -2.0 * s["df"] * ((r.real ** 2 + r.imag ** 2) / s["psd"]).sum()
    if case["do"] == "container":
        return _exact_container(case, seed)
    if case["do"] == "td":
        return _exact_td(case, seed)
    return None
