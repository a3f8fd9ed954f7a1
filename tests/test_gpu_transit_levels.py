"""Isothermal transits at level counts on both sides of each limit that the
workgroup's 160 KiB of LDS sets: a tile of 128 wavenumbers with the exponential
table and without it, a tile of 64 with the table and without it, for 16
wavefronts per tile (up to 12 slots) and for 8.  Against the same atmosphere
as a polynomial profile of ratio 1, which takes the general stencils.

The opacity terms of the two forms differ by at most their exponentials'
relative errors, 6e-13 and 1.1e-12; the transit depth follows the opacity's
logarithm times the scale height over the radius, so 1e-11 leaves a factor of
several."""

import numpy as np
import pytest

from bear_amd import synth

pytestmark = pytest.mark.gpu


def _case(levels, absorbers, profile):
    donor = synth.many_species_case()
    case = synth.transmission_small()
    case.nb_levels = levels
    case.wavenumber_full = 2500.0 + 4.0 * np.arange(1501)
    names = [s for s in synth.MANY_ABSORBERS if s != "Na"][:absorbers]
    rng = np.random.default_rng(levels + absorbers)
    case.species = [synth.line_table(rng, s, s, case.wavenumber_full, donor.species[0].temperatures,
                                     donor.species[0].pressures, n_lines=40) for s in names]
    case.chemistry = [("iso", list(names)), ("bg", ["H2He"])]
    case.temperature_model = profile
    mixing = 10.0 ** rng.uniform(-6.0, -3.0, absorbers)
    tail = [1340.0] + ([1.0] * 6 if len(profile) > 1 else [])
    case.parameters = np.concatenate([[3.2, synth.RADIUS_JUPITER, synth.RADIUS_SUN], mixing, tail, [0.0]])
    return case


@pytest.mark.parametrize("levels,absorbers",
                         [(n, 3) for n in (137, 138, 150, 153, 154, 273, 274)] + [(n, 12) for n in (137, 138, 153, 154)] +
                         [(n, 13) for n in (141, 142, 157, 158, 281, 282)])
def test_isothermal_transits_at_the_lds_limits(levels, absorbers, tmp_path):
    results = []
    for profile in (("const",), ("poly", 6, 1)):
        case = _case(levels, absorbers, profile)
        print(f"[gpu] transit of {levels} levels, {absorbers} slots, {profile[0]}", flush=True)
        r = synth.open_retrieval_in_memory(case, str(tmp_path / profile[0]))
        single = r.computeModel(case.parameters, True).spectrum
        ll = r.computeLikelihood(case.parameters)
        batch, _, _ = r.computeModelBatch(case.parameters[None, :], True)
        r.close()
        results.append((single, batch[0], ll))
    for k in range(2):
        assert np.all(np.isfinite(results[0][k]))
        np.testing.assert_allclose(results[0][k], results[1][k], rtol=1e-11)
    # the depths' differences of 1e-11 over errors of some 1e-2 of the depth
    np.testing.assert_allclose(results[0][2], results[1][2], rtol=1e-8)
