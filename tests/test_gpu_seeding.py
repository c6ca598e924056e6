"""GPU parity of engine states under new seeds: a generator seeded again and again (its
scratch and states are reused), and generators on different streams seeded at once, against
the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from oracle import oracle as O  # noqa: E402
from rocrand_amd import rocrand as R  # noqa: E402


def _words(g, n):
    buf = torch.zeros(n, dtype=torch.uint32, device="cuda")
    g.generate(buf)
    return buf


def _want(rng, n, **kw):
    st, w = O.OracleGen(rng, **kw).generate("u32", n)
    assert st == 0
    return w


def test_mt19937_states_under_new_seeds():
    """The first two words of every lane of all 8192 generators (both digits of the jump, their
    zero digits among them), under the seeds at the ends of the range."""
    g, n = R.PRNG(R.MT19937), 2 * 65536
    for seed in (0, 1, 0xFFFFFFFF, 0x8000000000000000, 0x0123456789ABCDEF):
        print(f"case mt19937 seed={seed:#x}", flush=True)
        g.seed = seed
        got = _words(g, n)
        torch.cuda.synchronize()
        assert np.array_equal(got.cpu().numpy(), _want(O.MT19937, n, seed=seed))


def test_mt19937_seeded_on_two_streams():
    n, seeds = 65536, (5, 6)
    streams = [torch.cuda.Stream() for _ in seeds]
    gens = [R.PRNG(R.MT19937, stream=s) for s in streams]
    for g in gens:
        g.initialize()
    bufs = [torch.zeros(n, dtype=torch.uint32, device="cuda") for _ in seeds]
    torch.cuda.synchronize()
    for g, b, seed in zip(gens, bufs, seeds):
        g.seed = seed
        g.generate(b)
    torch.cuda.synchronize()
    for b, seed in zip(bufs, seeds):
        assert np.array_equal(b.cpu().numpy(), _want(O.MT19937, n, seed=seed))


@pytest.mark.parametrize("rng", [R.XORWOW, R.LFSR113], ids=["xorwow", "lfsr113"])
def test_gf2_engine_states_under_new_seeds(rng):
    """Two words of every engine: no steps, one step more below `offset mod S`, every digit of
    the step count (past 2^32 steps LFSR113 counts modulo 2^32)."""
    S = 131072
    g, n = R.PRNG(rng), 2 * S + 3
    for seed, offset in ((0, 0), (1, S - 1), (0xFFFFFFFFFFFFFFFF, S), (5, 27 * S + 77), (6, (1 << 50) + 12345),
                         (7, 0xFFFFFFFFFFFFFFFF)):
        print(f"case {rng} seed={seed:#x} offset={offset:#x}", flush=True)
        g.seed = seed
        g.offset = offset
        got = _words(g, n)
        torch.cuda.synchronize()
        assert np.array_equal(got.cpu().numpy(), _want(rng, n, seed=seed, offset=offset))


@pytest.mark.parametrize("rng", [R.XORWOW, R.LFSR113], ids=["xorwow", "lfsr113"])
@pytest.mark.parametrize("blocks", [256, 1024, 2048])
def test_gf2_engine_states_on_other_grids(rng, blocks):
    """Engine counts below the DEFAULT grid's, at the end of the high jumps' table (2^18) and past it."""
    S = 256 * blocks
    R.set_dynamic_grid(rng, 256, blocks)
    try:
        g = R.PRNG(rng, seed=77, offset=5 * S + 3)
        g.set_ordering(R.ORDERING_PSEUDO_DYNAMIC)
        got = _words(g, S + 9)
        torch.cuda.synchronize()
    finally:
        R.set_dynamic_grid(rng, 0, 0)
    assert np.array_equal(got.cpu().numpy(), _want(rng, S + 9, seed=77, offset=5 * S + 3, grid=(256, blocks)))


def test_mtgp32_states_under_new_seeds():
    """Every generator's first words under the seeds at the ends of the range."""
    g, n = R.PRNG(R.MTGP32), 3 * 512 * 256
    for seed in (0, 1, 0xFFFFFFFF, 0x8000000000000000, 0xFFFFFFFFFFFFFFFF, 0x0123456789ABCDEF):
        print(f"case mtgp32 seed={seed:#x}", flush=True)
        g.seed = seed
        got = _words(g, n)
        torch.cuda.synchronize()
        assert np.array_equal(got.cpu().numpy(), _want(O.MTGP32, n, seed=seed))


@pytest.mark.parametrize("call", ["initialize", "generate_null"])
def test_mtgp32_set_up_returns_with_the_states_made(call):
    """Set up on a busy stream, then used on another one without a wait between them."""
    n, seed = 512 * 256 + 3, 42
    busy, other = torch.cuda.Stream(), torch.cuda.Stream()
    work = torch.empty(1 << 28, device="cuda")
    torch.cuda.synchronize()
    p = R.PRNG(R.PHILOX4_32_10, stream=busy)
    for _ in range(20):  # 3 ms of stores
        p.uniform(work)
    g = R.PRNG(R.MTGP32, seed=seed, stream=busy)
    if call == "initialize":
        g.initialize()
    else:
        assert R.load().rocrand_generate(g._gen, None, 0) == 0
    g.stream = other
    buf = torch.empty(n, dtype=torch.uint32, device="cuda")
    g.generate(buf)
    torch.cuda.synchronize()
    assert np.array_equal(buf.cpu().numpy(), _want(O.MTGP32, n, seed=seed))
