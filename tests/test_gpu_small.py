"""The one-workgroup kernels of small populations at the sizes where they begin, change and end,
and the general kernels on inputs as small as those that only they take otherwise: bit-exact
against the oracle."""
import numpy as np
import pytest
import torch

import oracle
from test_gpu_kernels import R, T, gpu_pairs, gpu_rps, random_pairs
from lagrangian_microbes_amd import device as dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [3, 1024, 1025, 4096, 4097, 12287, 12288, 12289])
@pytest.mark.parametrize("width,p", [(0.9, 2.0), (9.0, np.inf)])  # a patch within the table, and wrapping it
def test_pairs_at_the_sizes_where_kernels_change(gpu, n, width, p):
    rng = np.random.default_rng(n)
    x = (210.0 + width * rng.random(n)).astype(np.float32)
    y = (30.0 + rng.uniform(-0.05, 0.05, n) * 12000 / max(n, 1000)).astype(np.float32)
    x[-3:] = [209.0, 300.0, x[0]]  # outside the box, far away
    gi, gj = gpu_pairs(x, y, R, p, bbox=(209.9, 210.0 + width, 29.9, 30.1))
    bi, bj = oracle.pairs_bruteforce(x, y, R, p)
    assert np.array_equal(gi, bi) and np.array_equal(gj, bj)


@pytest.mark.parametrize("n", [5000, 12000])
def test_pairs_of_a_crowd(gpu, n):
    # most particles within one radius of each other beside a sparse rest: rows of a few to
    # thousands of partners, emitted by selection and by index order
    rng = np.random.default_rng(n)
    m = n // 8
    x = np.concatenate([210.0 + rng.uniform(0, R, m), 210.5 + rng.random(n - m)])
    y = np.concatenate([30.0 + rng.uniform(0, R, m), 30.0 + 0.2 * rng.random(n - m)])
    o = rng.permutation(n)
    x, y = x[o].astype(np.float32), y[o].astype(np.float32)
    gi, gj = gpu_pairs(x, y, R)
    bi, bj = oracle.pairs_bruteforce(x, y, R)
    assert np.array_equal(gi, bi) and np.array_equal(gj, bj)
