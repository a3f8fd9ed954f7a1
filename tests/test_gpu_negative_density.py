"""A density that is not positive counts as zero, so a layer between levels of
such densities alone is transparent and passes the intensity on unchanged: a
mixing ratio of -1e-30, which leaves the mean molecular weight as it is, gives
the bits of a mixing ratio of 0."""

import numpy as np
import pytest

from bear_amd import synth

pytestmark = pytest.mark.gpu


def test_negative_mixing_ratio_counts_as_zero(tmp_path):
    case = synth.tiny_case()
    case.species = case.species[:1]                           # H2O, no collision-induced absorption
    r = synth.open_retrieval_in_memory(case, str(tmp_path))
    zero = np.tile(case.parameters, (3, 1))
    zero[:, 3] = 0.0
    negative = zero.copy()
    negative[:, 3] = -1e-30
    out = []
    for p in (zero, negative):
        spectra = [r.computeModel(p[0], True).spectrum]
        for staging in (True, False):
            r.set_device_staging(staging)
            spectra += list(r.computeModelBatch(p, True)[0])
        out.append(np.array(spectra))
    r.close()
    assert np.array_equal(out[0], out[1])
