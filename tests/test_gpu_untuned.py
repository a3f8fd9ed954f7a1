"""Batches without the autotuner: the launch shape comes from the tiles of the
batch alone (one, four or eight wavefronts per tile) and, as a tuned shape,
leaves the bits as they are."""

import numpy as np
import pytest

from bear_amd import synth

pytestmark = pytest.mark.gpu


def test_untuned_shapes_leave_the_bits(tmp_path):
    case = synth.tiny_case()
    out, blocks = [], []
    for autotune in (True, False):
        r = synth.open_retrieval_in_memory(case, str(tmp_path))
        r.set_batch_options(True, autotune)
        tiles = -(-r.nb_spectral_points // 64)
        batches = [1, 8 * 256 // tiles, 8 * 256 // tiles + 1, 16 * 256 // tiles, 16 * 256 // tiles + 1, 200]
        p = np.tile(case.parameters, (max(batches), 1))
        p[:, 0] += 0.001 * np.arange(len(p))
        for batch in batches:
            out.append(r.computeLikelihoodBatch(p[:batch]))
            blocks.append(r.batch_stats()["block"])
        r.close()
    k = len(batches)
    for batch, tuned, untuned in zip(batches, out[:k], out[k:]):
        assert np.array_equal(tuned, untuned), batch
    assert blocks[k:] == [512, 512, 256, 256, 256, 256]       # 8 wavefronts per tile; 4; whole columns in 256
