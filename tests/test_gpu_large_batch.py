"""Batches of more threads than one launch takes (2^32): emission in several
launches, transits on reduced-precision tables with workgroups that walk on.
The live points repeat with a period of 16, so every point's log-likelihood has
to repeat to the last bit, whichever launch or round computed it, and to agree
with a batch of the 16 alone; there the launch shape may be another, which
regroups sums of some 100 terms: 1e-9 of the log-likelihood in FP64, 1e-4 where
the optical depths are FP32."""

import numpy as np
import pytest

from bear_amd import synth

pytestmark = pytest.mark.gpu

POINTS, PERIOD = 65_535, 16


def _case(model, levels, wavenumbers):
    case = synth.tiny_case() if model == "emission" else synth.transmission_small()
    nu = np.linspace(case.wavenumber_full[0], case.wavenumber_full[-1], wavenumbers)
    rng = np.random.default_rng(3)
    temps, press = np.array([500.0, 1500.0, 2500.0]), np.array([1e-4, 1.0])
    case.species = [synth.line_table(rng, s, s, nu, temps, press, n_lines=20) for s in ("H2O", "CH4")]
    case.rayleigh = []
    case.wavenumber_full = nu
    case.spectral_resolution = float(nu[1] - nu[0])
    case.nb_levels = levels
    case.observations = [o for o in case.observations if o.type == "band-spectroscopy"][:1]
    for o in case.observations:
        o.modifier, o.fwhm = "none", None
    # three general parameters, two mixing ratios, the temperature's
    case.parameters = case.parameters[:6 if model == "transmission" else 12]
    return case


@pytest.mark.parametrize("model,levels,wavenumbers,precision",
                         [("transmission", 8, 60_000, "int16"), ("emission", 4, 100_000, "fp64")])
def test_more_points_than_a_launch_takes(model, levels, wavenumbers, precision, tmp_path):
    case = _case(model, levels, wavenumbers)
    r = synth.open_retrieval_in_memory(case, str(tmp_path))
    # threads: emission one per wavenumber, transits 512 per 64 or 128
    assert r.nb_spectral_points * POINTS * (4 if model == "transmission" else 1) > 2 ** 32
    r.set_table_precision(precision)
    few = np.tile(case.parameters, (PERIOD, 1))
    few[:, 0] += 0.02 * np.arange(PERIOD)
    p = np.tile(few, (POINTS // PERIOD + 1, 1))[:POINTS]
    print(f"[gpu] {model}: {POINTS} points of {r.nb_spectral_points} wavenumbers", flush=True)
    ll = r.computeLikelihoodBatch(p)
    small = r.computeLikelihoodBatch(few)
    r.close()
    assert np.all(np.isfinite(ll)) and np.unique(small).size == PERIOD
    whole = ll[:POINTS // PERIOD * PERIOD].reshape(-1, PERIOD)
    assert np.array_equal(whole, np.tile(whole[0], (whole.shape[0], 1)))
    assert np.array_equal(ll[whole.size:], ll[:POINTS - whole.size])
    np.testing.assert_allclose(whole[0], small, rtol=1e-9 if precision == "fp64" else 1e-4)
