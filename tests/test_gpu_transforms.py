"""The normal and log-normal transforms' paths on the GPU: calls that stage their tables in
LDS (from 2^20 vecs of four words) against the same words through calls that do not, and
parameters that are infinite or not a number."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from rocrand_amd import rocrand as R  # noqa: E402


@pytest.mark.parametrize("kind,dt,per_word", [("normal", torch.float32, 1), ("lognormal", torch.float32, 1),
                                              ("normal", torch.float16, 2), ("lognormal", torch.float16, 2)])
@pytest.mark.parametrize("offset", [0, 3])
def test_staged_call_equals_unstaged_calls(kind, dt, per_word, offset):
    piece = 1 << 19  # words
    for words in (1 << 22, (1 << 22) - 4, (1 << 22) + 4 * 257 + 2):  # at the threshold, below it, a ragged end
        n = words * per_word
        big = torch.empty(n, dtype=dt, device="cuda")
        g = R.PRNG(R.PHILOX4_32_10, seed=9, offset=offset)
        getattr(g, kind)(big, 0.5, 2.0)
        small = torch.empty(n, dtype=dt, device="cuda")
        for w in range(0, words, piece):
            g = R.PRNG(R.PHILOX4_32_10, seed=9, offset=offset + w)
            getattr(g, kind)(small[w * per_word:(w + piece) * per_word], 0.5, 2.0)
        torch.cuda.synchronize()
        print(f"case {kind} {dt} offset={offset} words={words}", flush=True)
        bits = torch.int16 if dt == torch.float16 else torch.int32
        assert torch.equal(big.view(bits), small.view(bits))


@pytest.mark.parametrize("rng", [R.PHILOX4_32_10, R.XORWOW, R.MTGP32, R.MT19937, R.SOBOL32])
@pytest.mark.parametrize("dt", [torch.float32, torch.float64])
def test_infinite_and_nan_parameters(rng, dt):
    g = R.QRNG(rng) if rng == R.SOBOL32 else R.PRNG(rng, seed=1)
    buf = torch.empty(4098, dtype=dt, device="cuda")
    for kind, mean, want in (("lognormal", np.inf, np.inf), ("lognormal", -np.inf, 0.0), ("lognormal", np.nan, np.nan),
                             ("lognormal", 800.0, np.inf), ("lognormal", -800.0, 0.0), ("normal", np.inf, np.inf),
                             ("normal", np.nan, np.nan)):
        getattr(g, kind)(buf, mean, 1.0)
        torch.cuda.synchronize()
        got = buf.cpu().numpy()
        assert np.array_equal(got, np.full_like(got, want), equal_nan=True), (kind, mean, got[:4])
