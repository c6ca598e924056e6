"""Batches whose tiles fall on the edges of their paths, each stream against its plain call:
MRG32k3a engines that wrap at, before and after a tile's end, misaligned outputs, one launch
for a batch of several groups and little work and one per group for any other, streams
without values."""
import ctypes

import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from rocrand_amd import rocrand as R  # noqa: E402

S = 131072
DT = {R.BATCH_UINT: torch.int32, R.BATCH_UNIFORM_FLOAT: torch.float32, R.BATCH_UNIFORM_DOUBLE: torch.float64,
      R.BATCH_NORMAL_FLOAT: torch.float32, R.BATCH_NORMAL_DOUBLE: torch.float64,
      R.BATCH_LOG_NORMAL_FLOAT: torch.float32, R.BATCH_LOG_NORMAL_DOUBLE: torch.float64, R.BATCH_POISSON: torch.int32}


def _plain(rng, kind, seed, offset, view, a, b):
    g = R.PRNG(rng, seed=seed, offset=offset)
    if kind == R.BATCH_UINT:
        g.generate(view)
    elif kind in (R.BATCH_UNIFORM_FLOAT, R.BATCH_UNIFORM_DOUBLE):
        g.uniform(view)
    elif kind in (R.BATCH_NORMAL_FLOAT, R.BATCH_NORMAL_DOUBLE):
        g.normal(view, a, b)
    elif kind in (R.BATCH_LOG_NORMAL_FLOAT, R.BATCH_LOG_NORMAL_DOUBLE):
        g.lognormal(view, a, b)
    else:
        g.poisson(view, a)


def _check(streams):
    """streams: (rng, kind, seed, offset, n, shift); the one-shot call, the no-allocation call and a plan."""
    want, got = [], []
    for rng, kind, seed, offset, n, shift in streams:
        for out in (want, got):
            buf = torch.zeros(n + 16, dtype=DT[kind], device="cuda")
            out.append(buf[shift:shift + n])
    par = [(4.0, 0.0) if k == R.BATCH_POISSON else (0.5, 2.0) for _, k, *_ in streams]
    for (rng, kind, seed, offset, n, _), v, (a, b) in zip(streams, want, par):
        if n:
            _plain(rng, kind, seed, offset, v, a, b)
    arr = (R.BatchStream * len(streams))(*[
        R.BatchStream(rng, kind, seed, offset, n, a, b, v.data_ptr())
        for (rng, kind, seed, offset, n, _), v, (a, b) in zip(streams, got, par)])
    L = R.load()
    calls = [lambda: R.check_rocrand(L.rocrand_generate_batched(arr, len(arr), None)),
             lambda: R.check_rocrand(L.rocrand_generate_batched_noalloc(arr, len(arr), None))]
    plan = ctypes.c_void_p()
    R.check_rocrand(L.rocrand_batch_plan_create(ctypes.byref(plan), arr, len(arr), None))
    calls += [lambda: R.check_rocrand(L.rocrand_batch_plan_launch(plan))] * 3
    for call in calls:
        for v in got:
            v.zero_()
        call()
        torch.cuda.synchronize()
        for i, (g, w) in enumerate(zip(got, want)):
            assert torch.equal(g.view(torch.uint8), w.view(torch.uint8)), (i, streams[i])
    R.check_rocrand(L.rocrand_batch_plan_destroy(plan))


@pytest.mark.parametrize("kind", sorted(DT))
def test_mrg32k3a_wraps_at_tile_edges(kind):
    streams = []
    for k, left in enumerate((1, 255, 256, 257, 511, 512)):  # engines before the wrap
        for shift in (0, 1, 3):
            start = S - left
            streams.append((R.MRG32K3A, kind, 100 + k, 5 * S + start, 2 * 777 + k, shift))
    streams.append((R.MRG32K3A, kind, 7, 0, 300, 0))
    streams.append((R.MRG32K3A, kind, 8, S - 1, 1, 1))
    _check(streams)


def test_small_and_large_batches():
    for count in (1, 3, 200):
        streams = []
        for i in range(count):
            rng = R.PHILOX4_32_10 if i % 2 else R.MRG32K3A
            n = (0, 1, 5, 1023, 1024, 1025, 40001)[i % 7]
            streams.append((rng, sorted(DT)[(i // 2) % 8], i, i * 7919, n, i % 3))
        _check(streams)
    # past one launch's tiles: every kind, engines that all wrap and take several steps
    streams = [(R.MRG32K3A if i % 2 else R.PHILOX4_32_10, sorted(DT)[(i // 2) % 8], i, (1 << 20) + 7 + i, 3 * S + 5 + i,
                i % 4) for i in range(40)]
    _check(streams)


@pytest.mark.parametrize("rng,kind", [(R.PHILOX4_32_10, R.BATCH_UNIFORM_FLOAT), (R.PHILOX4_32_10, R.BATCH_NORMAL_DOUBLE),
                                      (R.MRG32K3A, R.BATCH_NORMAL_FLOAT)])
def test_one_group(rng, kind):
    for n in (3, 4099, (1 << 17) + 1, (1 << 20) + 5):
        _check([(rng, kind, i, i * 7919, n + i, i) for i in range(4)])


def test_batches_next_to_the_limit_of_one_launch():
    """512 MiB of output: 12 streams of two kinds just within it and just past it."""
    n = (512 << 20) // 48
    for extra in (-6, 6):
        _check([(R.MRG32K3A if i % 2 else R.PHILOX4_32_10, (R.BATCH_UINT, R.BATCH_UNIFORM_FLOAT)[(i // 2) % 2], i, i, n + extra,
                 0) for i in range(12)])


def test_empty_batches():
    """No streams, or only streams without values: every call succeeds and writes nothing."""
    _check([])
    _check([(R.MRG32K3A, R.BATCH_UINT, 1, 5, 0, 0), (R.PHILOX4_32_10, R.BATCH_NORMAL_FLOAT, 1, 5, 0, 1)])


def _request(count, seed):
    """`count` mixed streams, their outputs, and the values that plain calls give."""
    specs = [(R.MRG32K3A if i % 2 else R.PHILOX4_32_10, R.BATCH_UNIFORM_FLOAT, seed + i, i * 7919, 257 + i % 3) for i in range(count)]
    got = [torch.zeros(s[4], dtype=torch.float32, device="cuda") for s in specs]
    want = [torch.zeros_like(v) for v in got]
    for (rng, kind, sd, off, _), w in zip(specs, want):
        _plain(rng, kind, sd, off, w, 0.0, 0.0)
    arr = (R.BatchStream * count)(*[R.BatchStream(*s, 0.0, 0.0, v.data_ptr()) for s, v in zip(specs, got)])
    torch.cuda.synchronize()
    return arr, got, want


def test_one_shot_calls_on_streams_that_are_destroyed():
    """A program that makes a stream, calls, waits and destroys the stream, again and again: right
    values, no status but success and no block more for each call."""
    from test_gpu_graphs import Hip

    hip, L = Hip(), R.load()
    arr, got, want = _request(3000, 1)  # a descriptor image of about 1 MiB
    free = None
    for turn in range(40):
        s = hip.stream()
        for v in got[:4]:
            v.zero_()
        torch.cuda.synchronize()
        assert L.rocrand_generate_batched(arr, len(arr), s) == 0
        hip.check(hip.lib.hipStreamSynchronize(s))
        hip.check(hip.lib.hipStreamDestroy(s))
        assert all(torch.equal(g, w) for g, w in zip(got[:4], want[:4])), turn
        if turn == 3:
            free = torch.cuda.mem_get_info()[0]
    assert all(torch.equal(g, w) for g, w in zip(got, want))
    assert free - torch.cuda.mem_get_info()[0] < 8 << 20


@pytest.mark.parametrize("name", ["rocrand_generate_batched", "rocrand_generate_batched_noalloc"])
def test_captured_one_shot_call(name):
    """Every replay of a captured call, with other calls (and other host allocations) between them."""
    from test_gpu_graphs import Hip

    hip, generate = Hip(), getattr(R.load(), name)
    arr, got, want = _request(8, 100)
    other, got2, want2 = _request(9, 200)
    s = hip.stream()
    for calls in (2, 1):  # the third finds both blocks done and leaves one to capture with
        for _ in range(calls):
            R.check_rocrand(generate(arr, len(arr), s))
        hip.check(hip.lib.hipStreamSynchronize(s))
    graph, exe = hip.capture(s, lambda: R.check_rocrand(generate(arr, len(arr), s)))
    for _ in range(4):
        for v in got + got2:
            v.zero_()
        torch.cuda.synchronize()
        R.check_rocrand(generate(other, len(other), s))
        hip.launch(s, exe)
        R.check_rocrand(generate(other, len(other), s))
        hip.check(hip.lib.hipStreamSynchronize(s))
        assert all(torch.equal(g, w) for g, w in zip(got + got2, want + want2))
    hip.destroy(graph, exe)
    hip.check(hip.lib.hipStreamDestroy(s))
