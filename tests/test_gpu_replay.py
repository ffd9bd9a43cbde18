"""The replay's component classes on both sides of their limits, for populations on both sides of
the sizes where the small class and the grouping change, against the sequential oracle."""
import numpy as np
import pytest

import oracle
from test_gpu_kernels import gpu_rps

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [12_289, 131_072, 131_073, 1 << 20, (1 << 20) + 1, 1 << 21, (1 << 21) + 1])
def test_component_classes(gpu, n):
    rng = np.random.default_rng(n)
    # particles and pairs beyond a spanning tree, per component: 16, 17, 32, 33 pairs, one window and
    # two, the links pass's classes, more slots than the LDS holds
    sizes = [(s, e) for s in (2, 3, 9, 16, 17, 18, 32, 33, 34) for e in (0, 1, 2)] * 8
    sizes += [(12, 20), (12, 21), (20, 46), (40, 26), (250, 7), (250, 8), (300, 200), (2049, 100), (4200, 300)]
    perm, pairs, at, npairs = rng.permutation(n), set(), 0, []
    for size, extra in sizes:
        ids = perm[at:at + size]
        at += size
        mine = set()
        for a in range(1, size):
            b = int(rng.integers(max(0, a - 3), a))
            mine.add((min(ids[a], ids[b]), max(ids[a], ids[b])))
        want = min(len(mine) + extra, size * (size - 1) // 2)
        while len(mine) < want:
            a, b = rng.choice(ids, 2, replace=False)
            mine.add((min(a, b), max(a, b)))
        npairs.append(len(mine))
        pairs |= mine
    assert at <= n
    arr = np.array(sorted(pairs), dtype=np.int32)
    species = rng.integers(0, 5, n).astype(np.int8)  # 0 and 4 never interact
    args = (0.5, 0.6, 0.4, (n, 9), 3)
    got, up = gpu_rps(species, arr[:, 0], arr[:, 1], *args)
    assert np.array_equal(got, oracle.rps_sequential(species, arr[:, 0], arr[:, 1], *args))
    st, wide = up.component_stats(), [p for p in npairs if p > 32]
    assert st.components == len(sizes) and st.pairs == len(arr) and st.max_pairs == max(npairs)
    assert st.wide_components == len(wide) and st.wide_pairs == sum(wide)


def components(n, sizes, rng):
    """Sorted pairs of components of (particles, pairs) each on shuffled indices."""
    perm, pairs, at = rng.permutation(n), set(), 0
    for size, count in sizes:
        ids = np.sort(perm[at:at + size])
        at += size
        mine = {(int(ids[int(rng.integers(max(0, a - 3), a))]), int(ids[a])) for a in range(1, size)}  # a spanning tree
        while len(mine) < count:
            a, b = np.sort(rng.choice(ids, 2, replace=False))
            mine.add((int(a), int(b)))
        assert len(mine) == count
        pairs |= mine
    assert at <= n
    return np.array(sorted(pairs), dtype=np.int32)


# on both sides of the number of steps from which the links of smaller and larger components take a
# launch each, and of the population from which components of 17 to 32 pairs are small
@pytest.mark.parametrize("n,steps", [(12_289, 23), (12_289, 24), (140_000, 25)])
def test_component_classes_of_a_batch(gpu, n, steps):
    import torch
    from lagrangian_microbes_amd import device as dev
    rng = np.random.default_rng(n + steps)
    # pairs on both sides of the launches' limit (256) with few particles and with as many as pairs allow, on both
    # sides of the tables' slots (264, 2,048), and more particles than the replay holds in LDS (4,112)
    sizes = [(16, 16), (17, 17), (32, 32), (30, 33), (65, 64), (66, 65), (200, 255), (257, 256), (60, 256), (258, 257),
             (60, 257), (264, 300), (265, 300), (266, 300), (500, 2000), (2048, 2100), (2049, 2100)]
    lists = [components(n, sizes, rng), components(n, sizes[:10] + [(4112, 4200)], rng),
             components(n, sizes[8:] + [(4113, 4500)], rng), components(n, sizes[:4], rng)]
    cap = max(len(a) for a in lists)
    pi, pj = np.zeros((steps, cap), np.int32), np.zeros((steps, cap), np.int32)
    count = np.zeros(steps, np.int64)
    for s in range(steps):
        a = lists[s % 4]
        pi[s, :len(a)], pj[s, :len(a)], count[s] = a[:, 0], a[:, 1], len(a)
    sp = rng.integers(0, 5, n).astype(np.int8)
    up = dev.RPSUpdater(n, steps_max=steps)
    up.prepare(n, *(torch.from_numpy(a).cuda() for a in (pi, pj, count)), 0.55, 0.5, 0.45, (3, 4), 17)
    rec = torch.zeros((steps, n), dtype=torch.int8, device="cuda")
    up.play_steps(steps, torch.from_numpy(sp).cuda(), rec)
    rec = rec.cpu().numpy()
    for s in range(steps):
        sp = oracle.rps_sequential(sp, pi[s, :count[s]], pj[s, :count[s]], 0.55, 0.5, 0.45, (3, 4), 17 + s)
        assert np.array_equal(rec[s], sp), s


@pytest.mark.parametrize("form", ["plain", "read-only", "strided", "reversed"])
def test_reset_takes_any_array(gpu, form):
    from lagrangian_microbes_amd import FusedRunner, VelocityField
    rng = np.random.default_rng(4)
    lon, lat = 200.0 + rng.random(300), 20.0 + rng.random(300)
    species = rng.integers(1, 4, 300).astype(np.int8)
    host = [lon, lat, species]
    if form == "strided":
        host = [np.repeat(a, 2)[::2] for a in host]
    elif form == "reversed":
        host = [a[::-1].copy()[::-1] for a in host]
    elif form == "read-only":
        for a in host:
            a.flags.writeable = False
    f = VelocityField(np.array([199.0, 202.0]), np.array([19.0, 22.0]), np.zeros((1, 2, 2)), np.zeros((1, 2, 2)), None)
    r = FusedRunner(*host, f, 0.01, {"pRS": 0.5, "pPR": 0.5, "pSP": 0.5}, (1, 0), 3600.0, chunk=2)
    for got, want in zip((r.lon, r.lat, r.species), (lon, lat, species)):
        assert np.array_equal(got.cpu().numpy(), want)
    if form == "plain":  # what the arrays hold at the reset counts, and only then
        before = lon.copy()
        lon += 0.25
        assert np.array_equal(r.lon.cpu().numpy(), before)
        r.reset()
        assert np.array_equal(r.lon.cpu().numpy(), lon)
    r.run(2)
    assert r.step == 2
