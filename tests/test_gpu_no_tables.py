"""Retrievals that list no tabulated species: their padding slot still reads a
table row, which the store has to hold.  Rayleigh scattering alone (transits)
and no opacity at all (emission: the flux of the lowest level), against the
oracle at the parity tests' bar of 1e-5 of a spectrum (reduced-precision
tables too: they hold nothing here); the log-likelihoods are far from the data,
-1e3 to -1e7, so their bar of 1e-6 is taken relative."""

import os

import numpy as np
import pytest

from bear_amd import synth
from oracle import api as oracle_api

pytestmark = pytest.mark.gpu


def _case(model, profile):
    case = synth.transmission_small() if model == "transmission" else synth.eclipse_small() if model == "eclipse" \
        else synth.tiny_case()
    case.species = []
    if model == "transmission":
        case.temperature_model = profile
        if len(profile) > 1:
            k = case.parameters.size - 1                       # before the shift: the temperature's
            case.parameters = np.concatenate([case.parameters[:k], [0.95] * 6, case.parameters[k:]])
    return case


def _open(case, folder, storage="fp64"):
    synth.write_case(case, folder)
    r = synth.open_retrieval(folder, table_storage=storage)
    element = {"fp64": 8, "fp32": 4, "int16": 2}[storage]
    assert r.stats()["table_device_bytes"] >= element * r.nb_spectral_points      # before any kernel reads the row
    return r


@pytest.mark.parametrize("model,profile", [("transmission", ("const",)), ("transmission", ("poly", 6, 1)),
                                           ("emission", None), ("eclipse", None)])
def test_without_tabulated_species(model, profile, tmp_path):
    case = _case(model, profile)
    folder = os.path.join(str(tmp_path), "case", "")
    r = _open(case, folder)
    o = oracle_api.EmissionOracle(folder)
    p = case.parameters
    print(f"[gpu] {model} without tables", flush=True)
    ref = o.evaluate(p)
    out = r.computeModel(p, True)
    np.testing.assert_allclose(out.spectrum, ref["spectrum"], rtol=1e-5)
    np.testing.assert_allclose(r.computeLikelihood(p), ref["loglike"], rtol=1e-6)
    for staging in (True, False):
        r.set_device_staging(staging)
        spectra, _, _ = r.computeModelBatch(np.tile(p, (3, 1)), True)
        np.testing.assert_allclose(spectra, np.tile(ref["spectrum"], (3, 1)), rtol=1e-5)
    ll, grad = r.gradientBatch(p[None, :])
    np.testing.assert_allclose(ll[0], ref["loglike"], rtol=1e-6)
    assert np.all(np.isfinite(grad))
    r.close()
    for storage in ("fp32", "int16"):
        r = _open(case, folder, storage)
        spectra, _, _ = r.computeModelBatch(np.tile(p, (2, 1)), True)
        np.testing.assert_allclose(spectra, np.tile(ref["spectrum"], (2, 1)), rtol=1e-5)
        r.close()
    r = _open(case, folder)
    for precision in ("fp16", "bf16", "fp64"):
        r.set_table_precision(precision)
        spectra, _, _ = r.computeModelBatch(np.tile(p, (2, 1)), True)
        np.testing.assert_allclose(spectra, np.tile(ref["spectrum"], (2, 1)), rtol=1e-5)
    r.close()
