"""Every stencil-slot count of the register-cached kernels (1 to 16 tabulated
species, one instantiation each): a retrieval of S species against the same
retrieval with one more species of zero mixing ratio, which runs the next
instantiation and contributes exact zeros.  The sums then differ only in the
rounding of adding zero and of regrouped reductions (1e-12 covers both)."""

import numpy as np
import pytest

from bear_amd import synth

pytestmark = pytest.mark.gpu


def _case(model, absorbers, zero):
    case = synth.many_species_case() if model == "emission" else synth.transmission_small()
    donor = synth.many_species_case()
    step = donor.wavenumber_full[1] - donor.wavenumber_full[0]
    # without Na: listing it, even at zero, frees it from its ratio to K
    names = [s for s in synth.MANY_ABSORBERS if s != "Na"][:absorbers + 1]
    rng = np.random.default_rng(absorbers)
    if model == "transmission":
        case.wavenumber_full = donor.wavenumber_full[0] + step * np.arange(donor.wavenumber_full.size + 1000)
        case.nb_levels = 18
    case.species = [synth.line_table(rng, s, s, case.wavenumber_full, donor.species[0].temperatures,
                                     donor.species[0].pressures, n_lines=60) for s in names]
    mixing = 10.0 ** rng.uniform(-6.0, -3.0, absorbers + 1)
    if zero:
        mixing[-1] = 0.0
    else:
        case.species, names, mixing = case.species[:-1], names[:-1], mixing[:-1]
    case.chemistry = [("iso", list(names)), ("bg", ["H2He"])]
    if model == "transmission":
        head, tail = [3.2, synth.RADIUS_JUPITER, synth.RADIUS_SUN], [1300.0, 0.0]
    else:
        head, tail = [4.6, 1.0, 10 * synth.PARSEC], [2000.0, 0.9, 0.9, 0.9, 0.9, 0.9, 0.95]
    case.parameters = np.concatenate([head, mixing, tail])
    return case


@pytest.mark.parametrize("model", ["emission", "transmission"])
@pytest.mark.parametrize("absorbers", [1, 2, 3, 5, 6, 7, 9, 11, 13, 14, 15])
def test_slot_counts_agree(model, absorbers, tmp_path):
    results = []
    for zero in (False, True):
        case = _case(model, absorbers, zero)
        r = synth.open_retrieval_in_memory(case, str(tmp_path / str(zero)))
        p = np.array([case.parameters, case.parameters.copy()])
        p[1, 0] += 0.1
        out = {"single": r.computeModel(p[0], True).spectrum}
        out["fp64"], _, _ = r.computeModelBatch(p, True)
        ll, grad = r.gradientBatch(p)
        out["ll"] = ll
        out["grad"] = np.delete(grad, 3 + absorbers, axis=1) if zero else grad
        for precision in ("fp32", "fp16", "bf16", "int16"):
            r.set_table_precision(precision)
            out[precision], _, _ = r.computeModelBatch(p, True)
        r.close()
        results.append(out)
    for k in results[0]:
        a, b = results[0][k], results[1][k]
        assert np.all(np.isfinite(a)), k
        scale = np.abs(a).max(axis=0) if k == "grad" else np.abs(a)
        assert np.max(np.abs(a - b) / scale) < 1e-12, k
