"""Species counts at every alignment of a row, and the distance histogram at the edges of its
tiles and of its float32 classification, against numpy and the oracle: exact integer counts."""
import numpy as np
import pytest
import torch

import oracle
from lagrangian_microbes_amd import analysis

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 16, 31, 4097, 32768 + 16, 70001])
@pytest.mark.parametrize("skip", [0, 1, 9])
def test_counts_at_every_alignment(gpu, n, skip):
    rng = np.random.default_rng(n)
    sp = rng.integers(1, 4, size=5 * n + skip).astype(np.int8)
    sp[rng.integers(0, sp.size, 20)] = rng.integers(-128, 128, 20)
    rows = sp[skip:].reshape(5, n)
    got = analysis.species_counts(torch.from_numpy(sp).cuda()[skip:].view(5, n)).cpu().numpy()
    assert np.array_equal(got, np.stack([[np.sum(r == c) for c in (1, 2, 3)] for r in rows]))
