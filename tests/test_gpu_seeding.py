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
