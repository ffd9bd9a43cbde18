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


def clumps(n, sizes, width, rng):
    """Clumps of the given sizes, each within a tenth of a radius, spread over a patch of the given
    width, and particles far from each other: the k-th of a clump of m has m - 1 - k partners above."""
    m = sum(sizes)
    x, y = 210.0 + width * rng.random(n), 30.0 + 0.2 * rng.random(n)
    centre = np.repeat(np.arange(len(sizes)), sizes)
    x[:m] = 210.0 + width * (centre + 0.5) / len(sizes) + 0.1 * R * rng.random(m)
    y[:m] = 30.1 + 0.1 * R * rng.random(m)
    o = rng.permutation(n)
    return x[o].astype(np.float32), y[o].astype(np.float32)


# clumps on both sides of the rows that are kept, gathered and found in index order, a chunk of 64
# candidates and a wavefront's share of rows
@pytest.mark.parametrize("n,sizes", [(700, [513, 18]), (4096, [17, 18, 64, 66, 513, 514]), (4097, [600, 65, 17, 130] + [19] * 90),
                                     (12288, [700, 514] + [18] * 300)])
@pytest.mark.parametrize("width,p", [(0.9, 2.0), (9.0, 1.0), (9.0, 3.0), (2.0, np.inf)])
def test_pairs_of_crowded_rows(gpu, n, sizes, width, p):
    x, y = clumps(n, sizes, width, np.random.default_rng(n))
    gi, gj = gpu_pairs(x, y, R, p)
    bi, bj = oracle.pairs_bruteforce(x, y, R, p)
    assert np.array_equal(gi, bi) and np.array_equal(gj, bj)


@pytest.mark.parametrize("n,steps", [(3000, 30), (12000, 25)])
def test_pairs_of_crowded_rows_in_a_batch(gpu, n, steps):
    # more steps than the workgroups of four lanes per particle and 256 rows are for
    rng = np.random.default_rng(n)
    at = [clumps(n, [[600, 30], [17], [], [40] * 20][s % 4], 0.9, rng) for s in range(steps)]
    x, y = (np.stack([a[k] for a in at]) for k in (0, 1))
    cap = 300 * n
    ps = dev.PairSearch(n, (210.0, 210.9, 30.0, 30.2), R, steps_max=steps)
    pi, pj = (torch.zeros((steps, cap), dtype=torch.int32, device="cuda") for _ in range(2))
    count = torch.zeros(steps, dtype=torch.int64, device="cuda")
    ps.query_batch(T(x), T(y), R, 2.0, pi, pj, count)
    for s in [0, 1, 2, 3, steps - 1]:
        bi, bj = oracle.pairs_bruteforce(x[s], y[s], R)
        assert int(count[s]) == len(bi) <= cap
        assert np.array_equal(pi[s, :len(bi)].cpu().numpy(), bi) and np.array_equal(pj[s, :len(bi)].cpu().numpy(), bj)


@pytest.mark.parametrize("n,steps", [(4200, 52), (4200, 300), (5000, 130), (8193, 100), (8200, 257)])
def test_pairs_of_many_steps(gpu, n, steps):
    # a step's workgroups in several turns, and batches of more steps than workgroups run at once
    rng = np.random.default_rng(steps)
    few = 12  # distinct steps
    x, y = (210.0 + 0.6 * rng.random((few, n))).astype(np.float32), (30.0 + 0.6 * rng.random((few, n))).astype(np.float32)
    of = np.arange(steps) % few
    cap = 4 * n
    ps = dev.PairSearch(n, (210.0, 210.6, 30.0, 30.6), R, steps_max=steps)
    pi, pj = (torch.zeros((steps, cap), dtype=torch.int32, device="cuda") for _ in range(2))
    count = torch.zeros(steps, dtype=torch.int64, device="cuda")
    ps.query_batch(T(x[of]), T(y[of]), R, 2.0, pi, pj, count)
    count, pi, pj = count.cpu().numpy(), pi.cpu().numpy(), pj.cpu().numpy()
    for k in range(few):
        bi, bj = oracle.pairs_bruteforce(x[k], y[k], R)
        assert 0 < len(bi) <= cap
        for s in np.flatnonzero(of == k):
            assert count[s] == len(bi) and np.array_equal(pi[s, :len(bi)], bi) and np.array_equal(pj[s, :len(bi)], bj), s


def search_us(n, n_max, x, y):
    ps, best = dev.PairSearch(n_max, (210.0, 212.0, 30.0, 32.0), R), np.inf
    pi, pj = (torch.zeros(40 * n, dtype=torch.int32, device="cuda") for _ in range(2))
    for _ in range(4):
        a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        a.record()
        ps.query(x, y, R, 2.0, pi, pj, ps.npairs)
        b.record()
        torch.cuda.synchronize()
        best = min(best, 1e3 * a.elapsed_time(b))
    return best


def test_search_of_a_dense_population(gpu):
    # wide bound: finding every crowded row among all particles took 15 times the general kernels
    rng = np.random.default_rng(0)
    n, side = 12289, R * np.sqrt(12289 * np.pi / 24.0)  # twelve partners above each
    x, y = (T((a + side * rng.random(n)).astype(np.float32)) for a in (210.0, 30.0))
    assert search_us(n - 1, n, x[:-1].contiguous(), y[:-1].contiguous()) < 4 * search_us(n, n, x, y)


def star_and_chain(n):
    pairs = {(0, k) for k in range(1, n)} | {(k, k + 1) for k in range(n - 1)}
    return np.array(sorted(pairs), dtype=np.int32)


@pytest.mark.parametrize("n", [2, 1025, 12288, 12289])
def test_rps_star_and_chain(gpu, n):
    # every pair waits for another: one play after the other, several windows of pairs
    arr = star_and_chain(n)
    sp = np.random.default_rng(n).integers(0, 5, n).astype(np.int8)
    args = (0.5, 0.6, 0.4, (n, 1), 3)
    g, up = gpu_rps(sp, arr[:, 0], arr[:, 1], *args)
    assert np.array_equal(g, oracle.rps_sequential(sp, arr[:, 0], arr[:, 1], *args))
    st = up.component_stats()
    assert st.components == 1 and st.pairs == st.max_pairs == len(arr) and st.touched == st.max_particles == n


@pytest.mark.parametrize("n", [900, 20000])
def test_rps_pairs_in_any_direction(gpu, n):
    # sorted by (i, j), with j below i, on itself and out of range as well
    rng = np.random.default_rng(n)
    a, b = rng.integers(0, n, (2, 2 * n))
    b[::50] = n + 3
    b[25::50] = -1
    b[10::50] = a[10::50]
    arr = np.unique(np.stack([a, b], 1), axis=0).astype(np.int32)
    sp = rng.integers(1, 4, n).astype(np.int8)
    args = (0.5, 0.6, 0.4, (5, 1), 3)
    g, _ = gpu_rps(sp, arr[:, 0], arr[:, 1], *args)
    ref = sp.copy()
    u = oracle.philox_uniforms(len(arr), 0, 3, 0, 0, 5, 1)
    p = {(1, 3): 0.5, (2, 1): 0.6, (3, 2): 0.4}  # (winner, loser) of a forward outcome
    for k, (i, j) in enumerate(arr.tolist()):
        if 0 <= j < n and ref[i] != ref[j]:
            si, sj = int(ref[i]), int(ref[j])
            win, lose = (si, sj) if (si, sj) in p else (sj, si)
            w = win if u[k] < p[win, lose] else lose
            ref[i] = ref[j] = w
    assert np.array_equal(g, ref)


def batch_us(n, pi, pj, counts):
    """Prepare and replay of a batch."""
    up, best = dev.RPSUpdater(n, steps_max=len(counts)), np.inf
    species = torch.ones(n, dtype=torch.int8, device="cuda")
    species[::3], species[1::3] = 2, 3
    rec = torch.zeros((len(counts), n), dtype=torch.int8, device="cuda")
    for _ in range(5):
        a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        a.record()
        up.prepare(n, pi, pj, counts, 0.5, 0.5, 0.5, (1, 2), 0)
        up.play_steps(len(counts), species, rec)
        b.record()
        torch.cuda.synchronize()
        best = min(best, 1e3 * a.elapsed_time(b))
    return best


def test_a_batch_is_not_slower_below_the_line(gpu):
    # 12,288 particles with 1.5 partners above each, 24 steps: the general kernels, which 12,289
    # take, need 315 us, one workgroup 915; the bound lies between
    rng = np.random.default_rng(5)
    n, S = 12288, 24
    side = R * np.sqrt(n * np.pi / 3.0)
    x, y = (T((a + side * rng.random((S, n))).astype(np.float32)) for a in (210.0, 30.0))
    ps = dev.PairSearch(n, (210.0, 210.0 + side, 30.0, 30.0 + side), R, steps_max=S)
    pi, pj = (torch.zeros((S, 2 * n), dtype=torch.int32, device="cuda") for _ in range(2))
    counts = torch.zeros(S, dtype=torch.int64, device="cuda")
    ps.query_batch(x, y, R, 2.0, pi, pj, counts)
    assert int(counts.max()) <= 2 * n
    assert batch_us(n, pi, pj, counts) < 1.7 * batch_us(n + 1, pi, pj, counts)


def crowded(kind, n, rng):
    """Sorted pair lists with many pairs of one j."""
    ids = np.arange(n)
    if kind == "hub last":
        pairs = [(k, n - 1) for k in range(n - 1)]
    elif kind == "hub between":  # its pairs have it as i, as j, and as j below i
        h = n // 2
        pairs = [(k, h) for k in range(n) if k != h] + [(h, k) for k in range(0, n, 3) if k != h]
    elif kind == "crowd":
        m = np.sort(rng.permutation(n)[:n // 8])
        pairs = np.stack([m[a] for a in np.triu_indices(len(m), 1)], 1)
    elif kind == "lists of 16":
        pairs = [(k, j) for j in range(16, n, 16) for k in range(j - 16, j)]
    else:
        assert kind == "one list of 17"
        pairs = [(k, j) for j in range(16, n, 16) for k in range(j - 16, j)] + [(0, 32)]
    return np.unique(np.array(pairs, dtype=np.int32), axis=0)


def buffers(arr, cap):
    """The pairs in buffers of a larger capacity."""
    out = np.zeros((2, max(cap, len(arr))), np.int32)
    out[:, :len(arr)] = arr.T
    return T(out[0]), T(out[1])


@pytest.mark.parametrize("n", [66, 2500, 12288])
@pytest.mark.parametrize("kind", ["hub last", "hub between", "crowd", "lists of 16", "one list of 17"])
def test_rps_many_pairs_of_one_j(gpu, kind, n):
    rng = np.random.default_rng(n)
    arr = crowded(kind, n, rng)
    sp = rng.integers(0, 5, n).astype(np.int8)
    args = (0.5, 0.6, 0.4, (n, 2), 5)
    got = T(sp)
    dev.RPSUpdater(n).update(got, *buffers(arr, 3 * n), T(np.array([len(arr)])), *args)
    assert np.array_equal(got.cpu().numpy(), oracle.rps_sequential(sp, arr[:, 0], arr[:, 1], *args))


# on both sides of the populations and of the pair capacity that the small kernels are for
@pytest.mark.parametrize("n", [5120, 5121, 12288])
@pytest.mark.parametrize("over", [-1, 0])
def test_rps_at_the_lines_of_the_class(gpu, n, over):
    rng = np.random.default_rng(n + over)
    S, cap = 4, n * 5 // 2 + over
    lists = [np.stack(random_pairs(rng, n, m), 1) for m in (n // 2, n, 2 * n, n * 5 // 2 - 1)]
    lists[1] = star_and_chain(n)
    pi, pj = (torch.stack(b) for b in zip(*(buffers(a, cap) for a in lists)))
    counts = np.array([len(a) for a in lists])
    assert counts.max() <= cap
    sp = rng.integers(0, 5, n).astype(np.int8)
    up = dev.RPSUpdater(n, steps_max=S)
    up.prepare(n, pi, pj, T(counts), 0.55, 0.5, 0.45, (3, 4), 17)
    rec = torch.zeros((S, n), dtype=torch.int8, device="cuda")
    up.play_steps(S, T(sp), rec)
    for s, a in enumerate(lists):
        sp = oracle.rps_sequential(sp, a[:, 0], a[:, 1], 0.55, 0.5, 0.45, (3, 4), 17 + s)
        assert np.array_equal(rec[s].cpu().numpy(), sp), s
    st = up.component_stats(1)
    assert st.components == 1 and st.pairs == st.max_pairs == len(lists[1]) and st.touched == st.max_particles == n


def prepare_us(n, arr):
    pi, pj = (b[None] for b in buffers(arr, 3 * n))
    count, up, best = T(np.array([len(arr)])), dev.RPSUpdater(n), np.inf
    for _ in range(4):
        a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
        a.record()
        up.prepare(n, pi, pj, count, 0.5, 0.5, 0.5, (1, 2), 0)
        b.record()
        torch.cuda.synchronize()
        best = min(best, 1e3 * a.elapsed_time(b))
    return best


def test_prepare_is_linear_in_the_pairs(gpu):
    # wide bounds: quadratic lists took 360 times the hub with the lowest index, and 40 times the
    # general kernels on the crowd
    n, rng = 12288, np.random.default_rng(1)
    first = np.array([(0, k) for k in range(1, n)], dtype=np.int32)
    assert prepare_us(n, crowded("hub last", n, rng)) < 20 * prepare_us(n, first)
    crowd = crowded("crowd", 8 * 1000, rng)
    assert prepare_us(n, crowd) < 8 * prepare_us(n + 1, crowd)


@pytest.mark.parametrize("n,out", [(9001, 9001), (9000, 9016), (15000, 15000)])
def test_play_steps_matches_single_steps(gpu, n, out):
    rng = np.random.default_rng(n)
    S, cap = 5, 2 * n
    pi, pj = np.zeros((S, cap), np.int32), np.zeros((S, cap), np.int32)
    counts = np.zeros(S, np.int64)
    for s in range(S):
        m = [n, 0, 3, 2 * n, n // 2][s]
        a, b = random_pairs(rng, n, max(m, 1))
        pi[s, :m], pj[s, :m], counts[s] = a[:m], b[:m], m
    counts[4] = cap + 1  # too many for the buffers: the step changes nothing
    sp = rng.integers(1, 4, n).astype(np.int8)
    up = dev.RPSUpdater(n, steps_max=S)
    up.prepare(n, T(pi), T(pj), T(counts), 0.55, 0.5, 0.45, (3, 4), 17)
    rec = torch.zeros((S, out), dtype=torch.int8, device="cuda")[:, :n]
    up.play_steps(S, T(sp), rec)
    ref = sp
    for s in range(S):
        if s < 4:
            ref = oracle.rps_sequential(ref, pi[s, :counts[s]], pj[s, :counts[s]], 0.55, 0.5, 0.45, (3, 4), 17 + s)
        assert np.array_equal(rec[s].cpu().numpy(), ref), s
    one = rec[2].clone()
    up.play(3, one, one)  # a step by itself, in place
    assert torch.equal(one, rec[3])


@pytest.mark.parametrize("seed", [0, 1])
def test_general_replay_of_every_component_size(gpu, seed):
    # components of 2 to 3,000 particles among as many without pairs, above the small kernels' sizes
    rng = np.random.default_rng(seed)
    sizes = [2, 3, 5, 9] * 50 + [12, 40, 100] * 10 + [60] * 3 + [400, 1500] + [3000]
    n = 20000
    perm, pairs, at = rng.permutation(n), set(), 0
    for s in sizes:
        ids = perm[at:at + s]
        at += s
        for a in range(1, s):
            b = int(rng.integers(0, a))
            pairs.add((int(min(ids[a], ids[b])), int(max(ids[a], ids[b]))))
        for _ in range(12 * s if s == 60 else s):
            a, b = (int(v) for v in rng.choice(ids, 2, replace=False))
            pairs.add((min(a, b), max(a, b)))
    arr = np.array(sorted(pairs), dtype=np.int32)
    sp = rng.integers(1, 4, n).astype(np.int8)
    args = (0.5, 0.6, 0.4, (seed, 9), 21)
    g, up = gpu_rps(sp, arr[:, 0], arr[:, 1], *args)
    assert np.array_equal(g, oracle.rps_sequential(sp, arr[:, 0], arr[:, 1], *args))
    st = up.component_stats()
    assert st.components == len(sizes) and st.pairs == len(arr) and st.touched == at
