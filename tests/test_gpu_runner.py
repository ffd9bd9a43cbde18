"""FusedRunner.run's streams: a population whose chunks replay on a stream of their own and one whose
replay is the caller's, against runs of one chunk at a time; with callbacks that read, change and
fail, and without."""
import numpy as np
import pytest
import torch

from lagrangian_microbes_amd import FusedRunner, VelocityField
from lagrangian_microbes_amd.simulator import SMALL_POPULATION, chunk_schedule

pytestmark = pytest.mark.gpu

STEPS, CHUNK = 22, 5
SIZES = [3000, 13000]


def runner(n):
    assert (n > SMALL_POPULATION) == (n == SIZES[1])
    rng = np.random.default_rng(n)
    axis = np.linspace(0.0, 4.0, 17)
    f = VelocityField(208.0 + axis, 28.0 + axis, 0.3 * rng.standard_normal((1, 17, 17)),
                      0.3 * rng.standard_normal((1, 17, 17)), None)
    side = np.sqrt(n * np.pi * 0.01 ** 2 / 2.0)  # a partner above each
    return FusedRunner(210.0 + side * rng.random(n), 30.0 + side * rng.random(n), rng.integers(1, 4, n).astype(np.int8), f,
                       0.01, {"pRS": 0.5, "pPR": 0.6, "pSP": 0.4}, (n, 1), 600.0, chunk=CHUNK)


def one_by_one(n, change=None):
    """Species after every chunk of the same schedule, each advanced by itself."""
    r, out = runner(n), []
    for k in chunk_schedule(STEPS, CHUNK):
        r.advance(k)
        out.append(r.species.cpu().numpy())
        if change is not None:
            change(r)
    return r, out


def busy(t):
    """Some milliseconds of work on the current stream, whose result is t."""
    a = torch.ones((4096, 4096), device=t.device)
    for _ in range(4):
        a = a @ a * 0.0 + 1.0
    return t + (a[0, 0] * 0.0).to(t.dtype)


@pytest.mark.parametrize("n", SIZES)
def test_without_a_callback(gpu, n):
    ref, after = one_by_one(n)
    r = runner(n)
    rec = [torch.zeros((STEPS, n), dtype=t, device="cuda") for t in (torch.float32, torch.float32, torch.int8)]
    assert r.run(STEPS, records=rec) == STEPS
    got = r.species.clone()  # at once, on the caller's stream
    assert np.array_equal(got.cpu().numpy(), after[-1]) and torch.equal(rec[2][-1], got)
    assert torch.equal(r.lon, ref.lon) and torch.equal(r.lat, ref.lat)
    ends = np.cumsum(chunk_schedule(STEPS, CHUNK)) - 1
    for e, want in zip(ends, after):
        assert np.array_equal(rec[2][e].cpu().numpy(), want)


@pytest.mark.parametrize("n", SIZES)
def test_a_callback_that_reads_late(gpu, n):
    # its reads are queued behind other work, while the host goes on to the next chunks
    _, after = one_by_one(n)
    r, seen = runner(n), []

    def look(k, rx, ry, rs, npairs):
        seen.append((busy(r.species), busy(rs[k - 1])))

    r.run(STEPS, on_chunk=look)
    assert len(seen) == len(after)
    for (species, last), want in zip(seen, after):
        assert np.array_equal(species.cpu().numpy(), want) and np.array_equal(last.cpu().numpy(), want)


@pytest.mark.parametrize("n", SIZES)
def test_a_callback_that_changes_the_species(gpu, n):
    def change(r):
        r.species.copy_(busy(r.species.roll(7)))

    ref, after = one_by_one(n, change)
    r, seen = runner(n), []

    def look(k, rx, ry, rs, npairs):
        seen.append(rs[k - 1].clone())
        change(r)

    r.run(STEPS, on_chunk=look)
    for got, want in zip(seen, after):
        assert np.array_equal(got.cpu().numpy(), want)
    assert torch.equal(r.species, ref.species)


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("at", [0, 2])
def test_a_callback_that_fails(gpu, n, at):
    _, after = one_by_one(n)
    r, calls = runner(n), []

    def fail(k, rx, ry, rs, npairs):
        calls.append(k)
        if len(calls) == at + 1:
            raise KeyError("callback")

    with pytest.raises(KeyError):
        r.run(STEPS, on_chunk=fail)
    assert len(calls) == at + 1
    # the caller's stream waits for the others: what they used may be written now
    r.lon.fill_(0.0)
    r.species.fill_(0)
    r.rec_s.fill_(9)
    r.reset()
    r.run(STEPS)
    assert np.array_equal(r.species.cpu().numpy(), after[-1])


@pytest.mark.parametrize("n", SIZES)
def test_pair_buffers_that_grow_under_way(gpu, n):
    _, after = one_by_one(n)
    r, seen = runner(n), []
    r.engine.capacity = 0
    r.engine._grow(64)  # every chunk's first preparation overflows
    r.run(STEPS, on_chunk=lambda k, rx, ry, rs, npairs: seen.append(rs[k - 1].clone()))
    for got, want in zip(seen, after):
        assert np.array_equal(got.cpu().numpy(), want)


@pytest.mark.parametrize("n", SIZES)
def test_on_another_stream(gpu, n):
    _, after = one_by_one(n)
    r, st = runner(n), torch.cuda.Stream()
    st.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(st):
        r.run(CHUNK)
        r.run(STEPS - CHUNK)
        got = r.species.clone()
    st.synchronize()
    whole = runner(n)
    whole.run(CHUNK)
    whole.run(STEPS - CHUNK)
    assert torch.equal(got, whole.species) and np.array_equal(got.cpu().numpy(), after[-1])
