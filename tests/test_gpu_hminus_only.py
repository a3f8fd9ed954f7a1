"""Layers whose only absorber is the H- continuum: H- listed alone, H- without
H and electrons (bound-free only, so nothing absorbs above 1.64 micron), and
the tabulated species at zero mixing ratio, in every emission and eclipse call
and in the direct model, where H- may also end at a level.  Against the oracle at
the bars of the parity tests (spectra 1e-5; log-likelihoods 1e-6, relative
where they are far from the data), gradients at the gradient tests' bar (1e-4
beside the central differences' own error, which counts here: free-free layers
are so thin that e^-tau - 1 moves in steps of rounding)."""

import os

import numpy as np
import pytest

from bear_amd import api, synth
from oracle import api as oracle_api
from test_gpu_gradient import central, check, steps

pytestmark = pytest.mark.gpu


def _case(model, kind):
    case = synth.hminus_case()
    if kind == "alone":
        case.species = []
        case.chemistry = [("iso", ["H-", "H", "e-"]), ("bg", ["H2He"])]
        case.parameters = np.delete(case.parameters, 3)
    else:
        case.species = case.species[:1]                       # H2O at zero mixing, no collision-induced absorption
        case.parameters[3] = 0.0
    if kind == "bound-free":
        case.chemistry = [("iso", ["H2O", "H-"]), ("bg", ["H2He"])]
        case.parameters = np.delete(case.parameters, [5, 6])
    if model == "eclipse":
        case.model = "secondary_eclipse"
        case.parameters[1:3] = [0.11, 5500.0]
        for o in case.observations:
            o.data = np.full_like(o.data, 2000.0)
            o.error = np.full_like(o.error, 200.0)
    return case


@pytest.mark.parametrize("model", ["emission", "eclipse"])
@pytest.mark.parametrize("kind", ["alone", "zero mixing", "bound-free"])
def test_hminus_as_the_only_absorber(model, kind, tmp_path):
    case = _case(model, kind)
    folder = os.path.join(str(tmp_path), "case", "")
    synth.write_case(case, folder)
    r, o = synth.open_retrieval(folder), oracle_api.EmissionOracle(folder)
    p = case.parameters
    print(f"[gpu] {model}, H- {kind}", flush=True)
    ref = o.evaluate(p)
    out = r.computeModel(p, True)
    np.testing.assert_allclose(out.spectrum, ref["spectrum"], rtol=1e-5)
    np.testing.assert_allclose(r.computeLikelihood(p), ref["loglike"], rtol=1e-6)
    spectra, _, _ = r.computeModelBatch(np.tile(p, (3, 1)), True)
    np.testing.assert_allclose(spectra, np.tile(ref["spectrum"], (3, 1)), rtol=1e-5)
    ll, grad = r.gradientBatch(p[None, :])
    np.testing.assert_allclose(ll[0], ref["loglike"], rtol=1e-6)
    h = steps(p)
    fd, fd2 = central(r.computeLikelihood, p, h), central(r.computeLikelihood, p, h / 2)
    check(grad[0], fd2, f"{model}, H- {kind}", np.abs(fd - fd2))
    r.close()


def test_direct_model_with_hminus_only(tmp_path):
    case = synth.hminus_case()
    case.species = case.species[:1]
    levels = 24
    case.nb_levels = levels
    span = (0.55, 4.5)
    folder = synth.write_direct_case(case, os.path.join(str(tmp_path), "case", ""), span)
    cfg = api.GlobalConfig(retrieval_folder_path=folder, cross_section_file_path=folder + "opacity/",
                           wavenumber_file_path=folder + "wavenumber_full.dat",
                           spectral_resolution=case.spectral_resolution)
    m = api.EmissionModel(cfg, api.SpectralGrid(cfg, *span), levels, "scm", [], [s for s, _ in case.opacity_entries],
                          [f for _, f in case.opacity_entries])
    o = oracle_api.EmissionOracle(folder)
    names = ["H-", "H", "e-", "H2"]
    p = np.logspace(2.0, -5.0, levels)
    t = np.linspace(3000.0, 2200.0, levels)
    x = np.tile([1e-9, 5e-3, 2e-6, 0.9], (levels, 1))
    for top in (levels, levels // 2):                         # H- at every level, and none from half way up
        x[top:, 0] = 0.0
        print(f"[gpu] direct emission, H- on {top} of {levels} levels", flush=True)
        spec = m.calcSpectrum(1500.0, synth.RADIUS_JUPITER, 10 * synth.PARSEC, p, t, names, x)
        ref = o.direct_spectrum(1500.0, synth.RADIUS_JUPITER, 10 * synth.PARSEC, p, t, names, x, False)
        np.testing.assert_allclose(spec, ref, rtol=1e-5)
    m.close()
