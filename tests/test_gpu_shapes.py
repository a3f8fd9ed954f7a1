"""Sizes at which the split of the work over threads and wavefronts can go
wrong: levels fewer than, equal to and just above the emission sweep's 16
runs and beyond the staging kernel's 512 threads, wavenumbers around the tile
sizes, tables on more grids than share stencils, outputs longer than the
pinned ring they leave through.

The gradient's forward sweep runs from the bottom up over every level, the
other calls from the top down over runs of levels until the column is opaque
(2^-60 left): their likelihoods and the single-point and batched spectra agree
to the rounding of some 100 FP64 operations per level, 1e-11 of the flux; the
likelihood's differences of data and model raise that by less than 100."""

import numpy as np
import pytest

from bear_amd import synth

pytestmark = pytest.mark.gpu


def _case(levels, extra, absorbers=3, grids=1):
    case = synth.many_species_case()
    donor = synth.many_species_case()
    step = donor.wavenumber_full[1] - donor.wavenumber_full[0]
    case.wavenumber_full = donor.wavenumber_full[0] + step * np.arange(donor.wavenumber_full.size + extra)
    case.nb_levels = levels
    names = [s for s in synth.MANY_ABSORBERS if s != "Na"][:absorbers]
    rng = np.random.default_rng(levels + extra)
    t = donor.species[0].temperatures
    case.species = [synth.line_table(rng, s, s, case.wavenumber_full, t[k % grids:] if k % grids else t,
                                     donor.species[0].pressures, n_lines=60) for k, s in enumerate(names)]
    case.chemistry = [("iso", list(names)), ("bg", ["H2He"])]
    mixing = 10.0 ** rng.uniform(-6.0, -3.0, absorbers)
    case.parameters = np.concatenate([[4.6, 1.0, 10 * synth.PARSEC], mixing,
                                      [2000.0, 0.9, 0.9, 0.9, 0.9, 0.9, 0.95]])
    return case


def _points(case, count):
    p = np.tile(case.parameters, (count, 1))
    p[:, 0] += 0.01 * np.arange(count)
    return p


@pytest.mark.parametrize("levels,extra", [(7, 0), (15, 1), (16, 63), (17, 64), (31, 65), (33, 127), (65, 129), (600, 2)])
def test_sweeps_agree(levels, extra, tmp_path):
    r = synth.open_retrieval_in_memory(_case(levels, extra), str(tmp_path))
    p = _points(_case(levels, extra), 3)
    single = np.array([r.computeModel(q, True).spectrum for q in p])
    spectra, _, _ = r.computeModelBatch(p, True)
    ll = r.computeLikelihoodBatch(p)
    ll_up, _ = r.gradientBatch(p)
    r.close()
    assert np.all(np.isfinite(spectra))
    np.testing.assert_allclose(spectra, single, rtol=1e-11)
    np.testing.assert_allclose(ll, ll_up, rtol=1e-9)


@pytest.mark.parametrize("levels", [7, 600])
@pytest.mark.parametrize("grids", [1, 2, 3])
def test_staging_of_many_levels_and_grids(levels, grids, tmp_path):
    case = _case(levels, 0, absorbers=6, grids=grids)
    r = synth.open_retrieval_in_memory(case, str(tmp_path))
    p = _points(case, 3)
    p[2, 3] = 0.0                                              # a level without one of its absorbers
    out = []
    for on in (False, True):
        r.set_device_staging(on)
        out.append(r.computeModelBatch(p, True)[0])
    r.close()
    np.testing.assert_allclose(out[1], out[0], rtol=1e-10)


def test_output_longer_than_the_ring(tmp_path):
    case = _case(16, 65)
    r = synth.open_retrieval_in_memory(case, str(tmp_path))
    count = 4 * (1 << 17) // case.wavenumber_full.size + 40
    p = _points(case, count)
    spectra, _, _ = r.computeModelBatch(p, True)
    for k in (0, count // 2, count - 1):
        one, _, _ = r.computeModelBatch(p[k:k + 1], True)
        assert np.array_equal(spectra[k], one[0]), k
    r.close()
