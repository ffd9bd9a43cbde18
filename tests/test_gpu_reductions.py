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


def spread(kind, n, rng):
    if kind == "lattice":  # equal distances again and again, duplicates
        k = np.arange(n)
        return 205.0 + 0.0143 * (k // 40), 25.0 + 0.0143 * (k % 40) * (k % 7 > 0)
    if kind == "ocean":  # up to 150 degrees apart
        return rng.uniform(100.0, 250.0, n), rng.uniform(-70.0, 70.0, n)
    if kind == "globe":  # more than 180 degrees apart, the poles among them
        return rng.uniform(0.0, 360.0, n), np.where(rng.random(n) < 0.05, 90.0, rng.uniform(-90.0, 90.0, n))
    lon, lat = rng.uniform(200.0, 201.0, n), rng.uniform(-0.5, 0.5, n)  # a position that is not a number
    lon[n // 3] = np.nan
    return lon, lat


@pytest.mark.parametrize("kind", ["lattice", "ocean", "globe", "nan"])
@pytest.mark.parametrize("n,bins", [(2, 70), (511, 70), (513, 1), (1281, 72), (1300, 128), (769, 129)])
def test_histogram_at_the_edges(gpu, kind, n, bins):
    lon, lat = (a.astype(np.float32) for a in spread(kind, n, np.random.default_rng(n)))
    radius = analysis.EARTH_RADIUS_M if bins < 100 else 10.0 ** (0.1 * bins)  # thresholds that increase
    got = analysis.distance_histogram(torch.from_numpy(lon).cuda(), torch.from_numpy(lat).cuda(), bins, radius)
    assert np.array_equal(got, oracle.distance_histogram(lon, lat, analysis.haversine_thresholds(bins, radius)))


def histogram_us(lon, lat):
    """The kernel alone, from events around the call's launches."""
    lon, lat, best = torch.from_numpy(lon).cuda(), torch.from_numpy(lat).cuda(), np.inf
    for _ in range(4):
        a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        a.record()
        analysis.distance_histogram(lon, lat)
        b.record()
        torch.cuda.synchronize()
        best = min(best, 1e3 * a.elapsed_time(b))
    return best


def test_points_all_over_the_globe_cost_little_more(gpu):
    # bound between 1.2 (what it takes) and 2.5 times the basin's (with cosines and a search per pair)
    rng = np.random.default_rng(3)
    n = 40_000
    near = histogram_us(rng.uniform(120.0, 280.0, n).astype(np.float32), rng.uniform(-60.0, 60.0, n).astype(np.float32))
    far = histogram_us(rng.uniform(0.0, 360.0, n).astype(np.float32), rng.uniform(-90.0, 90.0, n).astype(np.float32))
    assert far < 1.8 * near


def haversine_term(lon, lat, i, j):
    """The term of one pair as the oracle computes it."""
    xi, yi, xj, yj = (float(v) for v in (lon[i], lat[i], lon[j], lat[j]))
    s1, s2 = oracle.sin_deg(0.5 * (yj - yi)), oracle.sin_deg(0.5 * (xj - xi))
    return s1 * s1 + (oracle.cos_deg(yi) * oracle.cos_deg(yj)) * (s2 * s2)


@pytest.mark.parametrize("n", [2, 513, 1300])
def test_thresholds_that_terms_meet(gpu, n):
    # the thresholds are terms of the points' own pairs, and their neighbours, so that every
    # one of them has a term on it or one step away; near and far apart, and increasing as they have to
    from lagrangian_microbes_amd import _lib
    rng = np.random.default_rng(n)
    for spread_deg in (8.0, 300.0):
        lon = (20.0 + spread_deg * rng.random(n)).astype(np.float32)
        lat = (-0.2 * spread_deg + 0.4 * spread_deg * rng.random(n)).clip(-90, 90).astype(np.float32)
        i, j = rng.integers(0, n - 1, 36), rng.integers(0, n, 36)
        j = np.where(j > i, j, i + 1)
        term = np.array([haversine_term(lon, lat, a, b) for a, b in zip(i, j)])
        near = [term, np.nextafter(term, 0), np.nextafter(term, 1)]
        edges = np.unique(np.concatenate(near + [term * (1 + 1e-6 * f) for f in (-5, -3, 3, 5)])[:255])
        hist = torch.zeros(len(edges) + 1, dtype=torch.int64, device="cuda")
        dev = [torch.from_numpy(a).cuda() for a in (lon, lat, edges)]
        _lib.check(_lib.load().lm_distance_histogram(n, _lib.ptr(dev[0]), _lib.ptr(dev[1]), len(edges) + 1, _lib.ptr(dev[2]),
                                                     _lib.ptr(hist), _lib.stream_ptr()))
        assert np.array_equal(hist.cpu().numpy().astype(np.uint64), oracle.distance_histogram(lon, lat, edges))
