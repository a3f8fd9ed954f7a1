"""Parameters that are not numbers give likelihoods that are not: a NaN
temperature or gravity reaches every level's density and thickness, and neither
the count of a level's absorbers (a NaN density is no zero) nor the zero
thickness of layers that absorb nothing (0 times NaN) may lose it."""

import numpy as np
import pytest

from bear_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mixing", [1e-4, 0.0])
@pytest.mark.parametrize("parameter", [0, 4])                 # log g, the lowest temperature
def test_nan_parameters_stay_nan(parameter, mixing, tmp_path):
    case = synth.tiny_case()
    case.species = case.species[:1]                           # H2O, no collision-induced absorption
    case.chemistry = [("iso", ["H2O"]), ("bg", ["H2He"])]
    case.parameters = np.delete(case.parameters, 4)
    case.parameters[3] = mixing
    r = synth.open_retrieval_in_memory(case, str(tmp_path))
    p = np.tile(case.parameters, (3, 1))
    p[1, parameter] = np.nan
    for staging in (True, False):
        r.set_device_staging(staging)
        ll = r.computeLikelihoodBatch(p)
        up, _ = r.gradientBatch(p)
        for values in (ll, up):
            assert np.isnan(values[1]) and np.all(np.isfinite(values[[0, 2]])), (staging, values)
    assert np.isnan(r.computeLikelihood(p[1])) and np.isfinite(r.computeLikelihood(p[0]))
    assert np.all(np.isnan(r.computeModel(p[1], True).spectrum))
    r.set_table_precision("fp32")
    assert np.isnan(r.computeLikelihoodBatch(p)[1])
    r.close()
