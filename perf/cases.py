"""The calls that a user of this engine times: likelihoods, models and gradients
of emission, transmission and secondary-eclipse retrievals, one live point or a
batch of them per call, over the sizes of the repository's configurations and
tests.

A case is a retrieval (forward model, atmosphere, opacity tables, observations)
and the call made on it.  A retrieval program builds one Retrieval, whose
tables stay on the GPU, and then calls it with new live points for hours; so
prepare() draws the live points of its seed from the priors and hands them over
with the case's Retrieval, which is kept for as long as the same case is asked
for.  Tables and observations depend on the case alone.

exact() evaluates the same model in 64 bits with torch operations, gradients by
torch.autograd.
"""

import json
import math
import os
import tempfile

import numpy as np
import torch

# cgs constants of the model
H, C, KB = 6.62606896e-27, 2.99792458e10, 1.3806504e-16
GAS, AVOGADRO = 8.314472e7, 6.022140857e23
R_JUP, R_SUN, PARSEC = 7.1492e9, 6.96342e10, 3.08567758135e18
MU = (0.211324865405187, 0.788675134594813)
WEIGHT = {"H2": 2.01588, "He": 4.002602, "H2O": 18.01528, "CH4": 16.04246, "CO": 28.0101, "CO2": 44.01,
          "NH3": 17.03052, "H2S": 34.09099, "HCN": 27.0253, "K": 39.0983, "Na": 22.98977, "TiO": 63.8664,
          "VO": 66.9409, "FeH": 56.853, "SO2": 64.066}
ABSORBERS = ["H2O", "CH4", "CO", "CO2", "NH3", "H2S", "HCN", "K", "TiO", "VO", "FeH", "SO2"]
P_BOTTOM, P_TOP = 100.0, 1e-6
TEMPERATURES = np.arange(100.0, 3001.0, 100.0)           # of the line and CIA tables

DEFAULTS = {"model": "emission", "call": "likelihood", "points": 1, "levels": 100, "absorbers": 6, "cia": True,
            "first": 1000.0, "step": 0.025, "wavenumbers": 100_000, "table_pressures": 9, "observation": "photometry",
            "bins": 100, "resolution": 0.0, "precision": "fp64", "cloud": False, "variable_gravity": False}


def _case(name, **kw):
    return dict(DEFAULTS, name=name, **kw)


def listed():
    return [
        # the plain single-evaluation retrieval of one R = 100 spectrum: the smallest call a sampler makes
        _case("point_small", levels=60, absorbers=2, cia=False, step=0.45, wavenumbers=20_001, observation="spectrum",
              bins=100, resolution=100.0),
        # one live point of the full-resolution photometric retrieval (the headline configuration)
        _case("point_emission", levels=100, wavenumbers=400_000, bins=300),
        # one transit model with its high-resolution spectrum, as it is plotted
        _case("model_transmission", model="transmission", call="model", levels=120, absorbers=5, first=2000.0,
              step=0.1, wavenumbers=60_013, observation="bands", bins=147, resolution=130.0),
        # a small nested-sampling batch, where launches and host work count
        _case("batch_small", call="likelihood_batch", points=16, levels=40, absorbers=3, first=2500.0, step=0.5,
              wavenumbers=9_001, observation="bands", bins=60, resolution=150.0),
        # a batch of live points in 64 bits, cloud-free emission
        _case("batch_emission", call="likelihood_batch", points=64, wavenumbers=99_777, bins=300),
        # the same with a grey cloud deck, whose parameters are fitted
        _case("batch_cloudy", call="likelihood_batch", points=24, levels=80, absorbers=4, step=0.05,
              wavenumbers=60_000, bins=80, cloud=True),
        # a large eclipse batch on 16-bit tables (12 absorbers, a blackbody star)
        _case("batch_eclipse_fp16", model="secondary_eclipse", call="likelihood_batch", points=192, absorbers=12,
              wavenumbers=300_000, table_pressures=12, bins=9, precision="fp16"),
        # the spectra of posterior samples: an eclipse model per point, on 32-bit tables
        _case("spectra_eclipse_fp32", model="secondary_eclipse", call="model_batch", points=13, levels=70, absorbers=5,
              first=2500.0, step=0.1, wavenumbers=45_000, observation="bands", bins=20, resolution=200.0,
              precision="fp32"),
        # a batch of transits in 64 bits: 200 tangent paths, eight absorbers
        _case("batch_transmission", model="transmission", call="likelihood_batch", points=48, levels=200, absorbers=8,
              first=2000.0, step=0.1, wavenumbers=60_000, observation="bands", bins=400, resolution=1000.0),
        # the same model on scaled 16-bit integers, gravity falling off with altitude
        _case("batch_transmission_int16", model="transmission", call="likelihood_batch", points=100, levels=100,
              absorbers=8, first=2000.0, step=0.1, wavenumbers=60_000, observation="bands", bins=147, resolution=300.0,
              precision="int16", variable_gravity=True),
        # value and gradient for a gradient-based sampler's chains
        _case("gradient_emission", call="gradient", points=32, wavenumbers=50_000, step=0.1, bins=300),
        _case("gradient_transmission", model="transmission", call="gradient", points=12, levels=100, absorbers=6,
              first=2000.0, step=0.2, wavenumbers=30_011, observation="bands", bins=147, resolution=130.0),
    ]


def draw(rng):
    """One more case: any call on any model, sizes over the listed ones' range, odd and ragged ones among them."""
    model = rng.choice(["emission", "secondary_eclipse", "transmission"])
    call = rng.choice(["likelihood", "model", "likelihood_batch", "likelihood_batch", "model_batch", "gradient"])
    batched = call in ("likelihood_batch", "model_batch")
    levels = rng.randint(30, 200 if model == "transmission" else 130)
    absorbers = rng.randint(1, 8 if model == "transmission" else 12)
    cia = rng.random() < 0.85
    most = 60_000 if call == "gradient" else 150_000
    n = int(math.exp(rng.uniform(math.log(4_000), math.log(most))))
    # no dearer than the listed batches: (point, level, species, wavenumber) terms within 6e9, gradients within 1.2e9
    room = (1.2e9 if call == "gradient" else 6e9) / (levels * (absorbers + 2) * n)
    if model == "transmission":
        room /= 1.0 + levels / 60.0
    top = max(1, min(128 if batched else 32, int(room)))
    points = 1 if call in ("likelihood", "model") else int(round(math.exp(rng.uniform(0.0, math.log(top)))))
    lsf = rng.random() < 0.5 or model == "transmission"
    first = rng.choice([1000.0, 1500.0, 2000.0, 2500.0])
    step = rng.uniform(5500.0, 8500.0) / n                # a few micron, whatever the resolution
    precision = rng.choice(["fp64", "fp64", "fp32", "fp16", "bf16", "int16"]) if batched else "fp64"
    cloud = model == "emission" and precision == "fp64" and rng.random() < 0.2
    return dict(DEFAULTS, model=model, call=call, points=points, levels=levels, absorbers=absorbers, cia=cia,
                first=first, step=step, wavenumbers=n, table_pressures=rng.randint(5, 12),
                observation="bands" if lsf else "photometry", bins=rng.randint(5, 200 if lsf else 50),
                resolution=rng.uniform(150.0, 600.0) if lsf else 0.0, precision=precision, cloud=cloud,
                variable_gravity=model == "transmission" and rng.random() < 0.4)


# ---------------------------------------------------------------- inputs
def _key(case):
    return json.dumps({k: v for k, v in case.items() if k != "name"}, sort_keys=True)


def _rng(case, salt):
    return np.random.default_rng([len(_key(case)), case["wavenumbers"], case["levels"], case["absorbers"], salt])


def _wavenumbers(case):
    return case["first"] + case["step"] * np.arange(case["wavenumbers"], dtype=np.float64)


def _table_pressures(case):
    return 10.0 ** np.linspace(-6.0, 2.0, case["table_pressures"])


def _species(case):
    """(symbol, folder, CIA partner or None) of every tabulated species."""
    out = [(s, s, None) for s in ABSORBERS[:case["absorbers"]]]
    if case["cia"]:
        out += [("CIA-H2-H2", "CIA/H2-H2", "H2"), ("CIA-H2-He", "CIA/H2-He", "He")]
    return out


def _table(case, k, device):
    """Table k as float32 [rows, wavenumbers] in (T, p) order, with its pressures: cross-sections, log10 of them for CIA.

    Line absorbers: lines every 3 cm^-1 on average, strengths over six decades,
    pressure-broadened Lorentzians of the five nearest cells, over a floor.
    CIA: smooth in wavenumber and temperature, one pressure."""
    rng = _rng(case, 100 + k)
    nu = torch.as_tensor(_wavenumbers(case), device=device)
    if _species(case)[k][2]:
        a, phase, centre = rng.uniform(0.5, 1.5), rng.uniform(0, 2 * math.pi), rng.uniform(float(nu[0]), float(nu[-1]))
        x = (nu - centre) / (nu[-1] - nu[0])
        t = torch.as_tensor(np.log10(TEMPERATURES / 1000.0), device=device)[:, None]
        lg = -45.5 + 0.6 * a * torch.sin(2 * math.pi * nu / 3000.0 + phase) - 3.0 * x * x + (0.9 - 0.2 * x) * t
        return lg.float(), np.array([1.0])
    p = _table_pressures(case)
    spacing = 3.0
    cells = int((float(nu[-1]) - float(nu[0])) / spacing) + 7
    lo = float(nu[0]) - 3 * spacing
    centre = torch.as_tensor(lo + spacing * (np.arange(cells) + rng.uniform(0, 1, cells)), device=device)
    strength = torch.as_tensor(10.0 ** rng.uniform(-24.0, -18.0, cells), device=device)
    energy = torch.as_tensor(rng.uniform(0.0, 4000.0, cells), device=device)
    at = ((nu - lo) / spacing).long()
    near = [(at + d).clamp(0, cells - 1) for d in (-2, -1, 0, 1, 2)]
    off2 = [(nu - centre[c]) ** 2 for c in near]
    out = torch.empty((TEMPERATURES.size, p.size, nu.numel()), dtype=torch.float32, device=device)
    for i, t in enumerate(TEMPERATURES):
        s = strength * (1000.0 / t) ** 1.5 * torch.exp(-H * C / KB * energy * (1.0 / t - 1e-3))
        gamma = torch.as_tensor(0.01 * math.sqrt(t / 1000.0) + 0.07 * p * (296.0 / t) ** 0.7, device=device)[:, None]
        sigma = torch.zeros((p.size, nu.numel()), dtype=torch.float64, device=device)
        for c, o in zip(near, off2):
            sigma += s[c] * (gamma / math.pi) / (o + gamma * gamma)
        out[i] = (1e-30 + sigma).float()
    return out.reshape(-1, nu.numel()), p


def _observation(case):
    """Bin edges (micron, descending), centres, data, errors, FWHMs, and per bin a bandpass or None."""
    rng = _rng(case, 7)
    nu = _wavenumbers(case)
    lo, hi = 1e4 / nu[-1], 1e4 / nu[0]
    n, r = case["bins"], case["resolution"]
    # with a line-spread function the bins leave its 5 sigma at the outermost centres inside the list
    m = 5.0 / (2.355 * r) if r else 0.0
    top = hi * (1 - 1e-4) / (1 + m) if r else hi * (1 - 1e-6)
    bottom = (lo * (1 + 1e-4) + m * (top - lo) / (2 * n)) / (1 - m) if r else lo * (1 + 1e-6)
    edges = np.linspace(top, bottom, n + 1)
    pairs = np.stack([edges[:-1], edges[1:]], axis=1)
    centres = pairs[:, 0] - (pairs[:, 0] - pairs[:, 1]) * 0.5
    if case["model"] == "emission":
        b = math.pi * 2 * H * C * C * (1e4 / centres) ** 3 / np.expm1(H * C * 1e4 / centres / KB / 1100.0) * 1e-3
        model = b * (R_JUP / (10 * PARSEC)) ** 2 / centres ** 2 * 1e4
        error = 0.02 * model
    else:
        model = np.full(n, 1.2e4 if case["model"] == "transmission" else 1500.0)
        error = np.full(n, 50.0 if case["model"] == "transmission" else 80.0)
    data = model + error * rng.standard_normal(n)
    filters = [None] * n
    if case["observation"] == "photometry":
        for b in range(n):
            x = np.linspace(0.0, 1.0, 50)
            f = np.sin(math.pi * x) ** rng.uniform(0.5, 2.0) * (1.0 + 0.2 * np.sin(2 * math.pi * rng.uniform(1, 3) * x))
            f[0] = f[-1] = 0.0
            filters[b] = ("photon" if b % 2 else "energy", pairs[b, 1] + (pairs[b, 0] - pairs[b, 1]) * x, np.abs(f))
    return {"edges": pairs, "centres": centres, "data": data, "error": error,
            "fwhm": centres / r if r else None, "filters": filters}


def _points(case, seed):
    """Live points drawn from the priors of their seed: [points, parameters]."""
    rng = np.random.default_rng([seed, 17])
    out = []
    for _ in range(case["points"]):
        if case["model"] == "emission":
            head = [rng.uniform(4.0, 5.5), rng.uniform(0.8, 1.2), 10 * PARSEC * rng.uniform(0.98, 1.02)]
        elif case["model"] == "secondary_eclipse":
            head = [rng.uniform(3.0, 4.0), rng.uniform(0.08, 0.15), rng.uniform(4500.0, 6500.0)]
        else:
            head = [rng.uniform(2.8, 3.8), R_JUP * rng.uniform(0.9, 1.1), R_SUN * rng.uniform(0.95, 1.05)]
        mixing = list(10.0 ** rng.uniform(-8.0, -3.0, case["absorbers"]))
        if case["model"] == "transmission":
            temperature = [rng.uniform(500.0, 2500.0)]
        else:
            t = np.sort(rng.uniform(500.0, 2500.0, 7))[::-1]
            temperature = [t[0]] + list(t[1:] / t[:-1])
        cloud = [10.0 ** rng.uniform(-1.0, 1.0), 10.0 ** rng.uniform(-3.0, 0.0), rng.uniform(3.0, 100.0)]
        out.append(head + mixing + temperature + (cloud if case["cloud"] else []))
    return np.array(out)


# ---------------------------------------------------------------- the calls
_kept = {}        # the last case's retrieval


def _retrieval(case):
    from bear_amd import api
    key = _key(case)
    if key in _kept:
        return _kept[key]
    for r in _kept.values():
        r.close()
    _kept.clear()
    api.clear_opacity_data()
    species = _species(case)
    for k, (_, folder, partner) in enumerate(species):
        rows, p = _table(case, k, "cuda")
        api.register_opacity_data(folder, np.repeat(TEMPERATURES, p.size), np.tile(p, TEMPERATURES.size),
                                  rows.cpu().numpy(), log_storage=partner is not None)
    o = _observation(case)
    if case["observation"] == "photometry":
        obs = [api.ObservationInput(f"band{b}", "photometry", o["data"][b:b + 1], o["error"][b:b + 1],
                                    bin_wavelength_edges=o["edges"][b:b + 1],
                                    filter_response=o["filters"][b][1:], filter_detector_type=o["filters"][b][0])
               for b in range(case["bins"])]
    elif case["observation"] == "bands":
        obs = [api.ObservationInput("bands", "band-spectroscopy", o["data"], o["error"],
                                    bin_wavelength_edges=o["edges"], instrument_profile_fwhm=o["fwhm"])]
    else:
        obs = [api.ObservationInput("spectrum", "spectroscopy", o["data"], o["error"], wavelengths=o["centres"],
                                    instrument_profile_fwhm=o["fwhm"])]
    names = ABSORBERS[:case["absorbers"]]
    opacity = [(s, f) for s, f, _ in species]
    if case["model"] == "transmission":
        opacity.append(("H2", "Rayleigh"))
    model = api.ModelConfig(case["levels"], P_BOTTOM, P_TOP, "const" if case["model"] == "transmission" else "poly 6 1",
                            ["iso " + " ".join(names), "bg H2He"], opacity,
                            use_variable_gravity=case["variable_gravity"],
                            cloud_model=["grey"] if case["cloud"] else [])
    with tempfile.TemporaryDirectory() as folder:
        path = os.path.join(folder, "wavenumbers.dat")
        with open(path, "w") as f:
            nu = _wavenumbers(case)
            f.write(f"{nu.size}\n" + "\n".join(map(repr, nu.tolist())) + "\n")
        config = api.GlobalConfig(wavenumber_file_path=path, spectral_resolution=case["step"])
        r = api.Retrieval(config, model, obs, forward_model_type=case["model"])
    api.clear_opacity_data()
    r.set_table_precision(case["precision"])
    _kept[key] = r
    return r


def prepare(case, seed):
    return {"call": case["call"], "retrieval": _retrieval(case), "points": _points(case, seed)}


def run(state):
    r, points = state["retrieval"], state["points"]
    if state["call"] == "likelihood":
        return {"log_likelihood": r.computeLikelihood(points[0])}
    if state["call"] == "model":
        m = r.computeModel(points[0], True)
        return {"spectrum": m.spectrum, "bins": m.spectrum_obs}
    if state["call"] == "likelihood_batch":
        return {"log_likelihood": r.computeLikelihoodBatch(points)}
    if state["call"] == "model_batch":
        spectra, bins, neglected = r.computeModelBatch(points, True)
        return {"spectrum": spectra, "bins": bins, "neglected": neglected}
    value, gradient = r.gradientBatch(points)
    return {"log_likelihood": value, "gradient": gradient}


def work(case):
    """Bytes: the table rows the points' levels fall between, each once, and the outputs.  Operations: per
    (point, level, species, wavenumber) the interpolation of four values and a power of ten (30), per (point,
    level, wavenumber) the layer's transfer (100; transmission: two per segment a path crosses, about a third of
    them before the path is opaque), and per gradient twice that again."""
    n, levels, points = case["wavenumbers"], case["levels"], case["points"]
    species = case["absorbers"] + 2 * case["cia"]
    if points >= 8:
        temperatures = 21                                        # the priors' whole range
    else:
        temperatures = 2 if case["model"] == "transmission" else 5
    rows = case["absorbers"] * temperatures * case["table_pressures"] + 2 * case["cia"] * temperatures
    width = {"fp64": 8, "fp32": 4}.get(case["precision"], 2)
    # a fixed pair of temperature rows at a time crosses each pressure row once
    if points < 8 and case["model"] != "transmission":
        rows = case["absorbers"] * 4 * case["table_pressures"] + 2 * case["cia"] * 20
    out = points * n * 8 if case["call"] in ("model", "model_batch") else points * 8
    layer = levels / 3.0 if case["model"] == "transmission" else 100.0
    flops = points * levels * n * (30.0 * species + layer) * (3.0 if case["call"] == "gradient" else 1.0)
    return {"bytes": float(rows * n * width + 2 * n * 8 + out), "flops": flops}


# ---------------------------------------------------------------- the same model in 64 bits
def _nearest(x, grid):
    """Index of the ascending grid's point nearest each x, the upper one on a tie."""
    k = np.searchsorted(grid, x)
    k = np.clip(k, 1, grid.size - 1)
    return np.where(np.abs(x - grid[k - 1]) < np.abs(x - grid[k]), k - 1, k)


def _operator(case, o, device):
    """The sampled wavenumbers, and the bins as a sparse matrix over them (bandpass, line-spread
    function and trapezoid per bin)."""
    full = _wavenumbers(case)
    edges = o["edges"]
    if case["observation"] == "spectrum":                         # bins half-way between the centres
        w = o["centres"]
        mid = 0.5 * (w[:-1] + w[1:])
        edges = np.stack([np.concatenate([[w[0] + (w[0] - w[1]) * 0.5], mid]),
                          np.concatenate([mid, [w[-1] - (w[-2] - w[-1]) * 0.5]])], axis=1)
    hi_w, lo_w = edges[0, 0], edges[-1, 1]
    if o["fwhm"] is not None:
        hi_w, lo_w = hi_w + 5.0 * o["fwhm"][0] / 2.355, lo_w - 5.0 * o["fwhm"][-1] / 2.355
    lo = int(np.searchsorted(full, 1.0 / hi_w * 1e4))
    lo -= full[lo] > 1.0 / hi_w * 1e4
    hi = int(np.searchsorted(full, 1.0 / lo_w * 1e4))
    nu = full[lo:hi + 1]
    lam = 1.0 / nu * 1e4
    flux = case["model"] != "transmission"
    sigma = np.zeros(nu.size)
    if o["fwhm"] is not None:
        c = o["centres"][::-1]
        inside = (lam >= c[0]) & (lam <= c[-1])
        sigma[inside] = np.interp(lam[inside], c, o["fwhm"][::-1]) / 2.355
        a = nu.size - 1 - _nearest_from_above(lam + 5 * sigma, lam)
        b = nu.size - 1 - _nearest_from_above(lam - 5 * sigma, lam)
        first, last = _nearest(1.0 / hi_w * 1e4, nu), _nearest(1.0 / lo_w * 1e4, nu)
    i0, i1 = _nearest(1.0 / edges[:, 0] * 1e4, nu), _nearest(1.0 / edges[:, 1] * 1e4, nu)
    lam_t = torch.as_tensor(lam, device=device)
    bins, at, weight = [], [], []
    for j in range(edges.shape[0]):
        i = np.arange(i0[j], i1[j] + 1)
        x = nu if flux else lam
        t = np.zeros(i.size)
        t[1:] += 0.5 * np.diff(x[i])
        t[:-1] += 0.5 * np.diff(x[i])
        width = abs(lam[i0[j]] - lam[i1[j]]) if flux or o["filters"][j] is None else 1.0
        t = np.abs(t) / width
        if o["fwhm"] is None:
            w, k = t, i
        else:
            i, t = i[(i >= first) & (i <= last)], t[(i >= first) & (i <= last)]
            plain = (sigma[i] == 0) | (a[i] == b[i])
            k0, k1 = min(int(a[i].min()), int(i[0])), max(int(b[i].max()), int(i[-1]))
            w = np.zeros(k1 - k0 + 1)
            np.add.at(w, i[plain] - k0, t[plain])
            rows, ts = i[~plain], t[~plain]
            k = np.arange(k0, k1 + 1)
            lk = lam_t[k0:k1 + 1]
            kk = torch.as_tensor(k, device=device)
            for s in range(0, rows.size, 256):
                r = rows[s:s + 256]
                ra, rb = (torch.as_tensor(v[r], device=device)[:, None] for v in (a, b))
                half = torch.zeros((r.size, k.size), dtype=torch.float64, device=device)
                d = 0.5 * (lk[:-1] - lk[1:])
                inside = (kk[:-1] >= ra) & (kk[1:] < rb)
                half[:, :-1] += torch.where(inside, d, 0.0)
                half[:, 1:] += torch.where(inside, d, 0.0)
                sg = torch.as_tensor(sigma[r], device=device)[:, None]
                g = math.sqrt(1.0 / (2.0 * math.pi)) / sg * torch.exp(-((lam_t[torch.as_tensor(r, device=device)]
                                                                         [:, None] - lk) / sg) ** 2 / 2)
                w += (torch.as_tensor(ts[s:s + 256], device=device)[:, None] * half * g).sum(0).cpu().numpy()
        if o["filters"][j] is not None:
            kind, fl, fr = o["filters"][j]
            y = fr * fl if kind == "photon" else fr
            norm = abs(float(np.sum(np.diff(fl) * (y[1:] + y[:-1]))) * 0.5)
            f = np.where((lam[k] >= fl[0]) & (lam[k] <= fl[-1]), np.interp(lam[k], fl, fr), 0.0)
            w = w * f * (lam[k] if kind == "photon" else 1.0) / norm
        bins.append(np.full(k.size, j))
        at.append(k)
        weight.append(w)
    m = torch.sparse_coo_tensor(torch.as_tensor(np.stack([np.concatenate(bins), np.concatenate(at)])),
                                torch.as_tensor(np.concatenate(weight)), (edges.shape[0], nu.size)).to(device)
    return lo, hi, torch.as_tensor(nu, device=device), m.coalesce()


def _nearest_from_above(x, descending):
    """_nearest on a descending list, the one further on in that list on a tie, as its index in the reversed list."""
    up = descending[::-1]
    k = np.clip(np.searchsorted(up, x, side="right") - 1, 0, up.size - 1)
    nxt = np.minimum(k + 1, up.size - 1)
    return np.where(np.abs(x - up[nxt]) < np.abs(x - up[k]), nxt, k)


def _planck(nu, t):
    return 2.0 * H * C * C * nu ** 3 / torch.expm1(H * C * nu / (KB * t))


class _Model:
    """One retrieval's forward model on torch tensors."""

    def __init__(self, case, device):
        self.case, self.device = case, device
        self.o = _observation(case)
        lo, hi, self.nu, self.bins = _operator(case, self.o, device)
        self.tables = []
        for k, (_, _, partner) in enumerate(_species(case)):
            rows, p = _table(case, k, device)
            t = rows[:, lo:hi + 1].double()
            t = t if partner else torch.log10(t)
            self.tables.append((t.reshape(TEMPERATURES.size, p.size, -1), p))
        levels = case["levels"]
        step = (math.log10(P_BOTTOM) - math.log10(P_TOP)) / (levels - 1.0)
        self.log_p = math.log10(P_BOTTOM) - step * np.arange(levels)
        self.p = torch.as_tensor(10.0 ** self.log_p, device=device)
        lam = 1e4 / self.nu
        n = 13.58e-5 * (1.0 + 7.52e-3 / (lam * lam)) + 1.0
        self.rayleigh = 24.0 * math.pi ** 3 * self.nu ** 4 / 2.651629e19 ** 2 * ((n * n - 1) / (n * n + 2)) ** 2

    def atmosphere(self, p):
        """Temperatures, densities by species and altitudes of the levels."""
        c, na = self.case, self.case["absorbers"]
        mixing, t = p[3:3 + na], p[3 + na:]
        if c["model"] == "transmission":
            temperature = t[0].expand(c["levels"])
        else:
            nodes = torch.cumprod(t[:7], 0)
            x = np.clip((math.log10(P_BOTTOM) - self.log_p) / (math.log10(P_BOTTOM) - math.log10(P_TOP)) * 6, 0, 6)
            k = np.minimum(x.astype(int), 5)
            f = torch.as_tensor(x - k, device=self.device)
            temperature = nodes[torch.as_tensor(k, device=self.device)] * (1 - f) + \
                nodes[torch.as_tensor(k + 1, device=self.device)] * f
        total = self.p * 1e6 / KB / temperature
        names = ABSORBERS[:na]
        share = {s: mixing[i] for i, s in enumerate(names)}
        if "K" in share:
            share["Na"] = share["K"] * 16.2181
        rest = 1.0 - sum(share.values())
        share["H2"], share["He"] = rest * 0.5 / 0.585114, rest * 0.085114 / 0.585114
        mu = sum(share[s] * WEIGHT[s] for s in share)
        rho = mu * self.p * 1e6 / (GAS * temperature)
        g = 10.0 ** p[0]
        z = [torch.zeros((), dtype=torch.float64, device=self.device)]
        for l in range(1, c["levels"]):
            gl = g * (p[1] / (p[1] + z[-1])) ** 2 if c["variable_gravity"] else g
            z.append(z[-1] + (1 / (rho[l] * gl) + 1 / (rho[l - 1] * gl)) * 0.5 * (self.p[l - 1] - self.p[l]) * 1e6)
        return temperature, {s: total * v for s, v in share.items()}, torch.stack(z)

    def opacity(self, temperature, density, a, b):
        """Absorption per level over wavenumbers [a, b)."""
        k_t = torch.clamp((temperature.detach() / 100.0).floor().long() - 1, 0, TEMPERATURES.size - 2)
        tg = torch.as_tensor(TEMPERATURES, device=self.device)
        f = ((temperature - tg[k_t]) / 100.0)[:, None]
        kappa = 0.0
        for (symbol, _, partner), (table, p) in zip(_species(self.case), self.tables):
            n = density["H2" if partner else symbol] * (density[partner] if partner else 1.0)
            v = table[:, :, a:b]
            if p.size == 1:
                lo, hi = v[k_t, 0], v[k_t + 1, 0]
            else:
                x = np.clip((self.log_p + 6.0) / 8.0 * (p.size - 1), 0, p.size - 1)
                k = np.minimum(x.astype(int), p.size - 2)
                w = torch.as_tensor(x - k, device=self.device)[:, None]
                k = torch.as_tensor(k, device=self.device)
                lo = v[k_t, k] * (1 - w) + v[k_t, k + 1] * w
                hi = v[k_t + 1, k] * (1 - w) + v[k_t + 1, k + 1] * w
            kappa = kappa + n[:, None] * 10.0 ** (lo * (1 - f) + hi * f)
        return kappa

    def cloud(self, p):
        """The grey cloud's optical depth per layer: tau over the layers between its bottom and top levels."""
        top_p, ratio = (float(v) for v in p[-2:].detach())
        pr = self.p.cpu().numpy()

        def level(x):
            return int(np.nonzero(((pr[:-1] > x) & (pr[1:] < x)) | (pr[:-1] == x))[0][-1])
        top = level(top_p)
        bottom = 0 if top_p * ratio >= pr[0] else level(top_p * ratio)
        if top == bottom:
            bottom -= 2
        if top < 2:
            top, bottom = 2, 0
        inside = torch.zeros(self.case["levels"] - 1, dtype=torch.float64, device=self.device)
        inside[bottom + 1:top + 1] = 1.0 / (top - bottom)
        return p[-3] * inside

    def spectrum(self, p, structure, a, b):
        """Flux (emission, eclipse) or transit depth over wavenumbers [a, b)."""
        c = self.case
        temperature, density, z = structure
        kappa = self.opacity(temperature, density, a, b)
        nu = self.nu[a:b]
        if c["model"] == "transmission":
            kappa = kappa + density["H2"][:, None] * self.rayleigh[a:b]
            r = p[1]
            seg = kappa[1:] + kappa[:-1]
            rz = r + z
            total = 0.0
            for t in range(c["levels"] - 1):
                s2 = rz[t + 1:] ** 2 - rz[t] ** 2
                d = torch.cat([torch.zeros(1, dtype=torch.float64, device=self.device), torch.sqrt(s2)])
                part = (d[1:] - d[:-1])[:, None] * seg[t:]
                run_ = torch.cumsum(part.detach(), 0)
                before = torch.cat([torch.zeros_like(run_[:1]), run_[:-1]])
                tau = torch.where(before <= 10.0, part, 0.0).sum(0)        # up to the first sum above 10
                total = total + rz[t] * (z[t + 1] - z[max(t - 1, 0)]) * -torch.expm1(-tau)
            return (total + r * r) / p[2] ** 2 * 1e6
        tau = (z[1:] - z[:-1])[:, None] * (kappa[1:] + kappa[:-1]) * 0.5
        if c["cloud"]:
            tau = tau + self.cloud(p)[:, None]
        planck = _planck(nu, temperature[:, None])
        flux = 0.0
        for m in MU:
            d = tau / m
            e = torch.exp(-d)
            q = torch.expm1(-d) / d
            i = planck[0]
            for l in range(c["levels"] - 1):
                i = i * e[l] + (1 + q[l]) * planck[l + 1] - (e[l] + q[l]) * planck[l]
            flux = flux + m * 0.5 * i
        scale = (R_JUP / p[2]) ** 2 * p[1] if c["model"] == "emission" else 1.0
        return 2 * math.pi * flux * 1e-3 * scale

    def observed(self, p, spectrum):
        """Bins and log-likelihood."""
        bins = torch.mv(self.bins, spectrum)
        if self.case["model"] == "secondary_eclipse":
            star = math.pi * 1e-3 * _planck(self.nu, p[2])
            bins = bins / torch.mv(self.bins, star) * p[1] ** 2 * 1e6
        d = torch.as_tensor(self.o["data"], device=self.device)
        e2 = torch.as_tensor(self.o["error"], device=self.device) ** 2
        return bins, (-0.5 * torch.log(2 * math.pi * e2) - 0.5 * (d - bins) ** 2 / e2).sum()

    def high_res(self, p, spectrum):
        if self.case["model"] == "emission":
            return spectrum * self.nu ** 2 / 1e4
        if self.case["model"] == "secondary_eclipse":
            return spectrum / (math.pi * 1e-3 * _planck(self.nu, p[2])) * p[1] ** 2 * 1e6
        return spectrum

    def chunks(self):
        """Pieces of the grid whose level arrays take at most about 2^24 values."""
        n = self.nu.numel()
        step = max(64, (1 << 24) // self.case["levels"])
        return [(a, min(n, a + step)) for a in range(0, n, step)]


def exact(case, seed):
    n = case["points"] * case["levels"] * case["wavenumbers"] * (case["absorbers"] + 2)
    if case["model"] == "transmission":
        n *= 1 + case["levels"] / 20
    if n > (4e9 if case["call"] == "gradient" else 1e11):
        return None                                               # over about 20 seconds
    device = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    m = _Model(case, device)
    lls, grads, spectra, binned = [], [], [], []
    for v in _points(case, seed):
        p = torch.tensor(v, dtype=torch.float64, device=device)
        with torch.no_grad():
            structure = m.atmosphere(p)
            spectrum = torch.cat([m.spectrum(p, structure, a, b) for a, b in m.chunks()])
            bins, ll = m.observed(p, spectrum)
        lls.append(float(ll))
        spectra.append(m.high_res(p, spectrum).cpu())
        binned.append(bins.cpu())
        if case["call"] == "gradient":
            p.requires_grad_(True)
            spectrum.requires_grad_(True)
            m.observed(p, spectrum)[1].backward()
            for a, b in m.chunks():
                m.spectrum(p, m.atmosphere(p), a, b).backward(spectrum.grad[a:b])
            grads.append(p.grad.cpu())
    if case["call"] == "likelihood":
        return {"log_likelihood": lls[0]}
    if case["call"] == "likelihood_batch":
        return {"log_likelihood": np.array(lls)}
    if case["call"] == "gradient":
        return {"log_likelihood": np.array(lls), "gradient": torch.stack(grads)}
    # one array of bins per observation: every band is its own photometric observation
    split = range(case["bins"]) if case["observation"] == "photometry" else None
    if case["call"] == "model":
        b = [binned[0][k:k + 1] for k in split] if split else [binned[0]]
        return {"spectrum": spectra[0], "bins": b}
    b = torch.stack(binned)
    return {"spectrum": torch.stack(spectra), "bins": [b[:, k:k + 1] for k in split] if split else [b],
            "neglected": None}
