"""Layers without any absorber pass the intensity on unchanged, whatever their
temperatures: above a cold absorbing atmosphere, hot transparent layers (at
visible wavelengths their Planck function is larger by up to 1e30) must not
enter the sums; nor must a hot transparent region between absorbing layers.
Against the oracle at the parity tests' bar of 1e-5 of a spectrum, gradients at
the gradient tests' bar."""

import os

import numpy as np
import pytest

from bear_amd import api, synth
from oracle import api as oracle_api
from test_gpu_gradient import central, check, steps

pytestmark = pytest.mark.gpu

NU = 2000.0 + 8.0 * np.arange(3501)                     # 0.33 to 5 micron


def _tables():
    rng = np.random.default_rng(8)
    temps, press = np.array([400.0, 900.0, 1700.0, 2600.0]), np.array([1e-5, 1e-2, 10.0])
    return [synth.line_table(rng, "H2O", "H2O", NU, temps, press, n_lines=400)]


def _case():
    case = synth.hminus_case()
    case.continuum = []
    case.wavenumber_full = NU
    case.spectral_resolution = 8.0
    case.species = _tables()
    case.chemistry = [("iso", ["H2O"]), ("bg", ["H2He"])]
    case.parameters = np.delete(case.parameters, [4, 5, 6])
    return case


LEVELS = 41


def _direct(folder, model):
    case = _case()
    case.model = model
    case.nb_levels = LEVELS
    span = (0.4, 4.5)
    lam = np.linspace(0.3, 5.2, 4001)
    stellar = (lam, synth.blackbody_flux_lambda(lam, 5200.0, 1.0)) if model == "secondary_eclipse" else None
    folder = synth.write_direct_case(case, folder, span, stellar)
    cfg = api.GlobalConfig(retrieval_folder_path=folder, cross_section_file_path=folder + "opacity/",
                           wavenumber_file_path=folder + "wavenumber_full.dat",
                           spectral_resolution=case.spectral_resolution)
    grid = api.SpectralGrid(cfg, *span)
    if model == "emission":
        return api.EmissionModel(cfg, grid, LEVELS, "scm", [], ["H2O"], ["H2O"]), oracle_api.EmissionOracle(folder)
    return (api.OccultationModel(cfg, grid, LEVELS, stellar[0], stellar[1], ["H2O"], ["H2O"]),
            oracle_api.EmissionOracle(folder))


# where H2O is (level ranges), over 500 K with 2600 K in the given levels
STRUCTURES = {"transparent top": ([(0, 20)], (24, 41)), "a single hot level at the top": ([(0, 20)], (40, 41)),
              "transparent middle": ([(0, 12), (30, 41)], (16, 26)), "transparent bottom": ([(20, 41)], (4, 15)),
              "no absorber": ([], (10, 41))}


@pytest.mark.parametrize("model", ["emission", "secondary_eclipse"])
@pytest.mark.parametrize("structure", list(STRUCTURES))
def test_direct_models_with_hot_transparent_layers(model, structure, tmp_path):
    m, o = _direct(os.path.join(str(tmp_path), "case", ""), model)
    where, hot = STRUCTURES[structure]
    p = np.logspace(2.0, -5.0, LEVELS)
    t = 500.0 + 100.0 * np.linspace(1.0, 0.0, LEVELS)
    t[hot[0]:hot[1]] = 2600.0
    x = np.tile([0.0, 1.0], (LEVELS, 1))
    for a, b in where:
        x[a:b] = [2e-4, 1.0 - 2e-4]
    print(f"[gpu] {model}: {structure}", flush=True)
    radius, distance = synth.RADIUS_JUPITER, 10 * synth.PARSEC
    if model == "emission":
        spec = m.calcSpectrum(1500.0, radius, distance, p, t, ["H2O", "N2"], x)
        ref = o.direct_spectrum(1500.0, radius, distance, p, t, ["H2O", "N2"], x, False)
    else:
        spec = m.calcSpectrum(1500.0, 0.11, p, t, ["H2O", "N2"], x)
        ref = o.direct_spectrum(1500.0, 0.11, 0.0, p, t, ["H2O", "N2"], x, False)
    m.close()
    np.testing.assert_allclose(spec, ref, rtol=1e-5)


def test_direct_model_with_a_cloud_in_transparent_layers(tmp_path):
    """The cloud's layers absorb where no gas does."""
    m, o = _direct(os.path.join(str(tmp_path), "case", ""), "emission")
    p = np.logspace(2.0, -5.0, LEVELS)
    t = 500.0 + 100.0 * np.linspace(1.0, 0.0, LEVELS)
    t[26:] = 2600.0
    x = np.tile([0.0, 1.0], (LEVELS, 1))
    x[:20] = [2e-4, 1.0 - 2e-4]
    cloud = np.zeros((LEVELS - 1, m.nb_spectral_points))
    cloud[30:33] = 0.3
    args = (1500.0, synth.RADIUS_JUPITER, 10 * synth.PARSEC, p, t, ["H2O", "N2"], x)
    spec = m.calcSpectrum(*args, cloud)
    ref = o.direct_spectrum(*args, False, cloud)
    m.close()
    np.testing.assert_allclose(spec, ref, rtol=1e-5)


def test_retrieval_without_absorption_under_an_inversion(tmp_path):
    """H2O at zero mixing ratio and a temperature that rises by a factor of
    five with altitude: the flux of the lowest level in every call."""
    case = _case()
    case.parameters[3] = 0.0
    case.parameters[4:11] = [500.0] + [1.31] * 6
    folder = os.path.join(str(tmp_path), "case", "")
    synth.write_case(case, folder)
    r, o = synth.open_retrieval(folder), oracle_api.EmissionOracle(folder)
    p = case.parameters
    ref = o.evaluate(p)
    np.testing.assert_allclose(r.computeModel(p, True).spectrum, ref["spectrum"], rtol=1e-5)
    for staging in (True, False):
        r.set_device_staging(staging)
        spectra, _, _ = r.computeModelBatch(np.tile(p, (2, 1)), True)
        np.testing.assert_allclose(spectra, np.tile(ref["spectrum"], (2, 1)), rtol=1e-5)
        ll, grad = r.gradientBatch(p[None, :])
        np.testing.assert_allclose(ll[0], ref["loglike"], rtol=1e-6)
        h = steps(p)
        f = lambda q: r.computeLikelihood(np.where(np.arange(p.size) == 3, 0.0, q))
        fd, fd2 = central(f, p, h), central(f, p, h / 2)
        fd[3] = fd2[3] = grad[0, 3] = 0.0                     # no derivative by a density of zero
        check(grad[0], fd2, "inversion without absorption", np.abs(fd - fd2))
    for precision in ("fp32", "fp16", "bf16", "int16"):
        r.set_table_precision(precision)
        spectra, _, _ = r.computeModelBatch(np.tile(p, (2, 1)), True)
        np.testing.assert_allclose(spectra, np.tile(ref["spectrum"], (2, 1)), rtol=1e-5)
    r.close()
